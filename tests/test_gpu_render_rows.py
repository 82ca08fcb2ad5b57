"""Grid, light and colour at the edges of the frame kernels' strips and row groups.

The kernels step one or two block rows a wavefront, by the world's size, and write their
colour and light in the same pass; each is run at all four offsets on worlds
whose height leaves a remainder and whose width leaves a partial strip.  The grid is compared with
a world stepped without outputs, with short and long modification lists; light, bit for bit, with the same float32 formula in numpy (every operation is one
IEEE operation in the shader's order, setCell's light loop, math.glsl:154-166); colour with that of
a short world whose first rows hold the same cells.
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


# strips of 64 columns x rows: up to 32768 one block row a wavefront, then two
@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (63, 2), (64, 3), (65, 1024), (129, 683), (257, 6), (65, 16385), (1, 32771)])
def test_frames_over_row_groups(w, h):
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

    big, small, plain = world(cells), world(cells[:top]), world(cells)
    plain.set_render(False)
    rng = np.random.RandomState(w + h)
    for f in range(5):
        prev, light = big.download(), big.render_download()[1]
        for _ in range((0, 2, 0, 9, 1)[f] if h > top else 0):  # below the rows that `small` holds
            m = (int(rng.randint(w)), int(rng.randint(top + 9, h + 9)), int(rng.randint(2)), int(rng.randint(1, 9)),
                 int(rng.choice([0, 3, 4])))
            big.push_modification(*m)
            plain.push_modification(*m)
        for a in (big, small, plain):
            a.step(1)
        np.testing.assert_array_equal(big.download(), plain.download())
        col, new = big.render_download()
        np.testing.assert_array_equal(new, light_step(prev, light))
    same = h if top == h else top - 12  # a step reaches at most two rows
    np.testing.assert_array_equal(col[:same], small.render_download()[0][:same])
    for a in (big, small, plain):
        a.close()
