"""Grids inside one tile in the rounds of larger ones (se_grids_step_noalloc): grid,
frame and the buffer that holds the result, at numbers of steps where the rounds that a
small grid takes come out even, odd, one and as many as the large grids'.
"""
import ctypes

import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O
from tests.test_zz_no_alloc import DevGrid, hip, ok

pytestmark = pytest.mark.gpu
IDS = ([0, 3, 4], [60, 25, 15])


# steps of the small grids, steps of the large one (8 a round)
@pytest.mark.parametrize("small,large", [((1, 2, 3, 16), 17), ((40, 33, 9, 17), 40), ((50, 7, 100, 8), 16),
                                         ((23, 24, 25, 64), 8)])
def test_small_grids_in_rounds(small, large):
    print(f"\n[gpu] small grids {small} beside {large} steps", flush=True)
    text = S.bundled_ruleset("four_materials")
    blob = O.compile_ruleset(L.parse_string(text))
    ctx = S.Context(0)
    rs = S.RuleSet(ctx, text)
    H = hip()
    sizes = [(60, 50), (112, 112), (1, 9), (111, 3), (230, 120)]
    steps = list(small) + [large]
    bufs, grids, want, mods = [], [], [], [(30, 20, 0, 7, 3)]
    for j, ((w, h), n) in enumerate(zip(sizes, steps)):
        pitch = (w + 63) // 64 * 64
        g = O.fill(31 + j, w, h, *IDS)
        t = DevGrid(H, w, h, pitch)
        t.upload(j % 2, g)
        bufs.append(t)
        grids.append(dict(grid0=t.ptr(0), grid1=t.ptr(1), w=w, h=h, pitch=pitch, cur=j % 2, frame=4 + j, nsteps=n,
                          mod_first=0, mod_count=1 if j == 0 else 0))
        for s in range(n):
            g = O.step(blob, g, 5 + j + s, mods=mods if j == 0 and s == 0 else None)
        want.append(g)
    stream = ctypes.c_void_p()
    ok(H.hipStreamCreate(ctypes.byref(stream)))
    out = S.grids_step_noalloc(ctx, rs, grids, mods, stream.value)
    ok(H.hipStreamSynchronize(stream))
    for j, ((cur, frame), t, g) in enumerate(zip(out, bufs, want)):
        rounds = 1 if j < 4 else -(-large // 8)  # a small grid ends where one launch would leave it
        assert (cur, frame) == ((j + rounds) % 2, 4 + j + steps[j])
        np.testing.assert_array_equal(t.download(cur), g, err_msg=f"grid {j}")
        t.free()
    ok(H.hipStreamDestroy(stream))
    ctx.close()
