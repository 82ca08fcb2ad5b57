"""The seeded fill against the oracle's at the widths where a row's share of a wavefront
changes, with and without the rows of stone, and with more ids than travel by value."""
import numpy as np
import pytest

import sandengine_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 33, 64, 65, 127, 128, 129, 255, 256, 257, 600]
_ctx = []


def ruleset():
    if not _ctx:
        _ctx.append(S.Context(0))
        _ctx.append(S.RuleSet(_ctx[0], S.bundled_ruleset("twelve_materials")))
    return _ctx


@pytest.mark.parametrize("n", [1, 4, 16, 17], ids=["1id", "4ids", "16ids", "17ids"])
@pytest.mark.parametrize("w", WIDTHS)
def test_fill_matches_oracle(w, n):
    print(f"\n[gpu] fill {w} wide, {n} ids", flush=True)
    ctx, r = ruleset()
    ids = [(5 * i) % 15 for i in range(n)]  # repeats where there are more ids than materials
    pct = [100 // n] * (n - 1)
    pct.append(100 - sum(pct))
    for h, stone in ((1, 0), (67, 9), (300, 0)):
        a = S.World(ctx, r, w, h)
        a.fill_seeded(11, ids, pct, stone_rows=stone, stone_id=5)
        want = O.fill(11, w, h, ids, pct)
        if stone:
            want[h - stone:] = 5
        np.testing.assert_array_equal(a.download(), want)
        a.close()
