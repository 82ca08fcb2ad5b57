"""A run whose last chunk of hash planes takes another form than the first: its planes,
with the frames that the step kernel loads ahead, need more room than the first chunk's."""
import numpy as np
import pytest

import sandengine_amd as S

pytestmark = pytest.mark.gpu


def test_last_chunk_in_the_other_form():
    print("\n[gpu] features 131039x106, 45 steps, 16 a launch", flush=True)
    ctx = S.Context(0)
    r = S.RuleSet(ctx, S.bundled_ruleset("features"))
    a, b = S.World(ctx, r, 131039, 106), S.World(ctx, r, 131039, 106)
    for w in (a, b):
        w.frame = 1
        w.fill_seeded(7, [0, 3, 4, 5, 6, 7], [40, 20, 12, 12, 8, 8])
    a.step(45)
    b.step_blocked(45, 16)
    assert a.frame == b.frame == 46
    np.testing.assert_array_equal(a.download(), b.download())
    a.close()
    b.close()
