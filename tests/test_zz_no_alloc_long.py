"""One-tile grids of very many steps beside a larger grid of two rounds
(se_grids_step_noalloc): the call divides their steps over the rounds without counting
through them, and returns before the device is done."""
import ctypes
import time

import numpy as np
import pytest

import sandengine_amd as S
from tests.test_zz_no_alloc import DevGrid, hip, ok

pytestmark = pytest.mark.gpu


def test_long_runs_are_divided_at_once():
    print("\n[gpu] 600 grids of 2x1 cells, 400000 steps each", flush=True)
    ctx = S.Context(0)
    rs = S.RuleSet(ctx, S.bundled_ruleset("four_materials"))
    H = hip()
    n, steps = 600, 400000
    small = DevGrid(H, 64, 2 * n, 64)  # rows of 64 cells: grid j is row 2 j, its other buffer row 2 j + 1
    large = DevGrid(H, 300, 200, 320)
    grids = [dict(grid0=small.ptr(0) + 512 * j, grid1=small.ptr(0) + 512 * j + 256, w=2, h=1, pitch=64, cur=0, frame=1,
                  nsteps=steps) for j in range(n)]
    grids.append(dict(grid0=large.ptr(0), grid1=large.ptr(1), w=300, h=200, pitch=320, cur=0, frame=1, nsteps=16))
    stream = ctypes.c_void_p()
    ok(H.hipStreamCreate(ctypes.byref(stream)))
    t = time.perf_counter()
    out = S.grids_step_noalloc(ctx, rs, grids, [], stream.value)
    host = time.perf_counter() - t
    ok(H.hipStreamSynchronize(stream))
    assert out == [(1, 1 + steps)] * n + [(0, 17)]
    assert host < 0.1  # a count of 200000 steps a grid takes more than 0.3 s
    assert not np.any(small.download(1)) and not np.any(large.download(0))  # EMPTY stays
    small.free()
    large.free()
    ok(H.hipStreamDestroy(stream))
    ctx.close()
