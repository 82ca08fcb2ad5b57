"""The sliced kernels (bit planes, 32 blocks to a word) against the plain kernel
and the oracle: worlds at the edges of the one-tile forms and of the tiles'
columns and rows, every phase of the Margolus cycle as the first step, NULL, WALL
and unknown ids inside the world, queued brushes, and launch depths that divide
the run or do not.  Whole numbers, so equality."""
import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu

_ctx = None
_rs = {}
FILL = {"four_materials": ([0, 3, 4, 5], [50, 25, 15, 10]),
        "twelve_materials": ([0] + list(range(3, 15)), [40] + [5] * 12),
        "features": ([0, 3, 4, 5, 6, 7], [40, 20, 12, 12, 8, 8])}
# one tile of 128 x 128 or 256 x 128 cells holds 123 x 126 or 251 x 126; further
# on, multiples of a tile's 64 useful columns and of its rows, and one beside them
SIZES = [(1, 1), (2, 3), (64, 64), (123, 126), (124, 126), (123, 127), (251, 126), (252, 126), (251, 127), (1, 700),
         (700, 1), (256, 128), (257, 129), (530, 301), (640, 193), (1021, 67)]


def rs(name):
    global _ctx
    if _ctx is None:
        _ctx = S.Context(0)
    if name not in _rs:
        _rs[name] = S.RuleSet(_ctx, S.bundled_ruleset(name))
    return _rs[name]


def grid(name, w, h, seed):
    ids, pct = FILL[name]
    g = O.fill(seed, w, h, ids, pct)
    rng = np.random.RandomState(seed)
    for v in (1, 2, 200):  # NULL, WALL and an id no material has
        k = max(1, w * h // 200)
        g[rng.randint(0, h, k), rng.randint(0, w, k)] = v
    return g


@pytest.mark.parametrize("name", list(FILL))
@pytest.mark.parametrize("size", SIZES, ids=[f"{w}x{h}" for w, h in SIZES])
def test_sliced_equals_plain(name, size):
    print(f"\n[gpu] sliced {name} {size}", flush=True)
    r, (W, H) = rs(name), size
    a, b = S.World(_ctx, r, W, H), S.World(_ctx, r, W, H)
    g = grid(name, W, H, 5)
    for first, steps, sub in ((2, 12, 0), (3, 37, 8), (4, 70, 0), (1, 29, 13)):
        for w in (a, b):
            w.upload(g)
            w.frame = first
            w.push_modification(W // 2, H // 3, 0, 5, 3)
            w.push_modification(W - 2, H - 3, 1, 4, 2)
        a.step(steps)
        b.step_blocked(steps, sub)
        assert a.frame == b.frame == first + steps
        np.testing.assert_array_equal(a.download(), b.download(), err_msg=f"first {first} steps {steps} sub {sub}")
    a.close()
    b.close()


@pytest.mark.parametrize("name", ["four_materials", "twelve_materials"])
@pytest.mark.parametrize("size,first,steps", [((5003, 4999), 3, 45), ((9001, 2801), 2147483000, 38)],
                         ids=["5003x4999", "9001x2801_late"])
def test_sliced_shared_hash_planes(name, size, first, steps):
    """Worlds large enough to share hash planes between block rows and frames (rows
    past 461 wrap); a start near the last frame, where the hash inputs wrap."""
    print(f"\n[gpu] sliced {name} {size} from frame {first}", flush=True)
    r, (W, H) = rs(name), size
    a, b = S.World(_ctx, r, W, H), S.World(_ctx, r, W, H)
    for w in (a, b):
        w.fill_seeded(3, *FILL[name])
        w.frame = first
    a.step(steps)
    b.step_blocked(steps)
    assert a.frame == b.frame == first + steps
    np.testing.assert_array_equal(a.download(), b.download())
    a.close()
    b.close()


@pytest.mark.parametrize("name", list(FILL))
def test_sliced_equals_oracle(name):
    print(f"\n[gpu] sliced {name} against the oracle", flush=True)
    r, W, H, steps = rs(name), 389, 211, 45
    blob = O.compile_ruleset(L.parse_string(S.bundled_ruleset(name)))
    g = grid(name, W, H, 9)
    w = S.World(_ctx, r, W, H)
    w.upload(g)
    w.frame = 6
    w.step_blocked(steps)
    np.testing.assert_array_equal(w.download(), O.run(blob, g, 7, steps))
    w.close()


@pytest.mark.parametrize("graph", [False, True], ids=["streams", "graph"])
@pytest.mark.parametrize("k", [0, 5, 16])
def test_sliced_batch_equals_per_world_plain(graph, k):
    """A batch of both rule-set forms: worlds inside one tile and beyond it, with
    equal and with different first frames and step counts, one of them 0."""
    print(f"\n[gpu] sliced batch graph={graph} k={k}", flush=True)
    b, pairs = S.Batch(rs("four_materials").ctx), []
    for i, (W, H) in enumerate([(64, 64), (123, 126), (124, 126), (1, 300), (300, 1), (389, 211), (640, 193), (17, 90)]):
        for name, first, steps in (("four_materials", 2, 40 + 13 * i), ("twelve_materials", 2 + i % 3, 9 + 31 * (i % 4)),
                                   ("features", 2147483000 if i == 5 else 7, 60 if i else 0)):
            x, y = S.World(_ctx, rs(name), W, H), S.World(_ctx, rs(name), W, H)
            for w in (x, y):
                w.upload(grid(name, W, H, 20 + i))
                w.frame = first
            pairs.append((x, y, steps))
            b.add(x, steps)
    for _ in range(2):
        b.run(mode=1, k=k, graph=graph)
        for x, y, steps in pairs:
            y.step(steps)
            assert x.frame == y.frame
            np.testing.assert_array_equal(x.download(), y.download(), err_msg=f"{x.W}x{x.H} {x.rules.nmat} {steps}")
    b.close()
    for x, y, _ in pairs:
        x.close()
        y.close()


def test_sliced_long_run_of_a_small_world():
    """More steps in one call than one launch hashes ahead."""
    print("\n[gpu] sliced 40000 steps of a 20x14 world", flush=True)
    r = rs("four_materials")
    a, b = S.World(_ctx, r, 20, 14), S.World(_ctx, r, 20, 14)
    for w in (a, b):
        w.upload(grid("four_materials", 20, 14, 3))
        w.frame = 1
    a.step(40000)
    b.step_blocked(40000)
    assert a.frame == b.frame
    np.testing.assert_array_equal(a.download(), b.download())
    a.close()
    b.close()
