"""Light and colour at the edges of the render kernels' strips and row groups.

The kernels take 1, 2 or 4 rows a wavefront by the world's size; each is run on worlds
whose height leaves a remainder and whose width leaves a partial strip.  Light is compared,
bit for bit, with the same float32 formula in numpy (every operation is one
IEEE operation in the shader's order, setCell's light loop, math.glsl:154-166); colour with that of
a short world of one row a wavefront whose first rows hold the same cells.
"""
import numpy as np
import pytest

import sandengine_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


def light_step(prev, light):
    """four_materials: no material emits, and only empty cells let light through."""
    h, w = prev.shape
    term = light.copy()
    term[..., :3] *= np.where(prev == 0, F(1), F(0))[..., None]
    term[..., :3] *= light[..., 3:]
    pad = np.zeros((h + 2, w + 2, 4), F)
    pad[1:-1, 1:-1] = term
    there = np.zeros((h + 2, w + 2), bool)
    there[1:-1, 1:-1] = True
    avg, top, n, most = np.zeros((h, w, 4), F), np.zeros((h, w, 4), F), np.zeros((h, w), F), np.zeros((h, w), F)
    for dx, dy in ((0, 1), (0, -1), (-1, 1), (-1, -1), (1, 1), (1, -1), (1, 0), (-1, 0)):
        here = np.s_[1 + dy:1 + dy + h, 1 + dx:1 + dx + w]
        t, ok = pad[here].copy(), there[here]
        t[..., 3] = np.where(t[..., 3] == 0, most, t[..., 3])
        avg = np.where(ok[..., None], avg + t, avg)
        top = np.where(ok[..., None], np.maximum(top, t), top)
        most = np.where(ok, np.maximum(t[..., 3], most), most)
        n += ok
    avg /= np.maximum(n, F(1))[..., None]
    out = avg * F(0.5) + top * F(0.5)
    out[..., 3] = avg[..., 3]
    out[0] = np.array([1, 1, 1, 0.999999], F)
    return out


# strips of 64 columns x rows: up to 2048 one row a wavefront, up to 32768 two, then four
@pytest.mark.parametrize("w,h", [(1, 1), (63, 2), (65, 1024), (64, 2049), (129, 683), (65, 16385), (1, 32771)])
def test_light_and_colour_over_row_groups(w, h):
    print(f"\n[gpu] render rows {w}x{h}", flush=True)
    ctx = S.Context(0)
    rules = S.RuleSet(ctx, S.bundled_ruleset("four_materials"))
    cells = O.fill(3, w, h, [0, 3, 4], [80, 12, 8])
    top = min(h, 24)

    def world(grid):
        a = S.World(ctx, rules, grid.shape[1], grid.shape[0])
        a.set_render(True)
        a.step(1)
        a.upload(grid)
        a.frame = 1
        return a

    big, small = world(cells), world(cells[:top])
    for _ in range(4):
        prev, light = big.download(), big.render_download()[1]
        big.step(1)
        small.step(1)
        col, new = big.render_download()
        np.testing.assert_array_equal(new, light_step(prev, light))
    same = h if top == h else top - 12  # a step reaches two rows, light one
    np.testing.assert_array_equal(col[:same], small.render_download()[0][:same])
    big.close()
    small.close()
