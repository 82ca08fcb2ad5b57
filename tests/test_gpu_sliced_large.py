"""The sliced kernels of large worlds -- tiles of one wavefront, from 2048 and from 8192
squares of 64 cells on -- with rules that change WALL cells, and batches that reach them."""
import numpy as np
import pytest

import sandengine_amd as S

pytestmark = pytest.mark.gpu

_ctx = None
_rs = {}
FILL = {"features": ([0, 3, 4, 5, 6, 7, 2], [36, 20, 12, 12, 8, 8, 4]),
        "four_materials": ([0, 3, 4, 5, 2], [48, 25, 13, 10, 4])}


def rs(name):
    global _ctx
    if _ctx is None:
        _ctx = S.Context(0)
    if name not in _rs:
        _rs[name] = S.RuleSet(_ctx, S.bundled_ruleset(name))
    return _rs[name]


def pair(name, w, h, seed, frame):
    r, out = rs(name), []
    for _ in range(2):
        v = S.World(_ctx, r, w, h)
        v.frame = frame
        v.fill_seeded(seed, *FILL[name])
        out.append(v)
    return out


@pytest.mark.parametrize("size,first", [((2999, 3001), 2), ((5903, 6101), 3)], ids=["2999x3001", "5903x6101"])
def test_rules_that_change_wall(size, first):
    print(f"\n[gpu] sliced features {size}", flush=True)
    a, b = pair("features", *size, 3, first)
    a.step(41)
    b.step_blocked(41)
    assert a.frame == b.frame
    np.testing.assert_array_equal(a.download(), b.download())
    a.close()
    b.close()


@pytest.mark.parametrize("sizes", [[(700, 3001), (64, 64), (2500, 1300)], [(5903, 3101), (3100, 2900)]],
                         ids=["2x2", "4x2"])
def test_batches_of_large_worlds(sizes):
    print(f"\n[gpu] sliced batch {sizes}", flush=True)
    rs("features")
    b, worlds = S.Batch(_ctx), []
    for i, (w, h) in enumerate(sizes):
        for name in ("features", "four_materials"):
            x, y = pair(name, w, h, 5 + i, 2 + i)
            b.add(x, 30 + 7 * i)
            worlds.append((x, y, 30 + 7 * i))
    b.run(mode=1)
    for x, y, steps in worlds:
        y.step(steps)
        assert x.frame == y.frame
        np.testing.assert_array_equal(x.download(), y.download(), err_msg=f"{x.W}x{x.H}")
        x.close()
        y.close()
    b.close()
