"""Modification lists of the plain kernel: up to 8 travel in its arguments, longer ones
in the world's buffer.  Both against the oracle, at the line between them and on
both sides of a strip's end (column 256); a list ends at its first size-0 entry.
"""
import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu
W, H = 261, 37


@pytest.mark.parametrize("n", [1, 7, 8, 9, 256])
def test_list_lengths(n):
    print(f"\n[gpu] plain kernel, {n} modifications", flush=True)
    text = S.bundled_ruleset("four_materials")
    blob = O.compile_ruleset(L.parse_string(text))
    ctx = S.Context(0)
    w = S.World(ctx, S.RuleSet(ctx, text), W, H)
    rng = np.random.RandomState(n)
    grid = O.fill(9, W, H, [0, 3, 4], [60, 25, 15])
    w.step(1)
    w.upload(grid)
    w.frame = 1
    for f in range(2, 7):
        mods = [(int(rng.choice([0, 254, 255, 256, 257, W - 1, rng.randint(W)])), int(rng.randint(-2, H + 2)),
                 int(rng.randint(2)), int(rng.randint(1, 12)), int(rng.choice([0, 1, 3, 4, 5]))) for _ in range(n)]
        if f == 5:
            mods[n // 2] = mods[n // 2][:3] + (0, 3)  # the list ends here
        for m in mods:
            w.push_modification(*m)
        w.step(1)
        grid = O.step(blob, grid, f, mods=mods)
        np.testing.assert_array_equal(w.download(), grid, err_msg=f"frame {f}")
    w.close()
