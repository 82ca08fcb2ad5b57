"""Sleeping of the sliced kernels (settled tiles skip their sub-steps, squares known to be
uniform are not packed or unpacked) and modifications of a run's first step leave every
result as it is: worlds with settled regions are advanced with sleeping on and off and
compared cell for cell with the plain kernel while everything that must wake a region or
end the record happens."""
import ctypes

import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O
from tests.test_zz_no_alloc import H2D, hip, ok

pytestmark = pytest.mark.gpu

_ctx = None
_rs = {}
FILL = {"four_materials": ([0, 3, 4], [85, 10, 5]), "twelve_materials": ([0, 3, 5], [90, 5, 5]),
        "features": ([0, 3, 4], [90, 5, 5])}


def rs(name):
    global _ctx
    if _ctx is None:
        _ctx = S.Context(0)
    if name not in _rs:
        _rs[name] = S.RuleSet(_ctx, S.bundled_ruleset(name))
    return _rs[name]


def sliced_index(w):
    i = 0
    while True:
        try:
            w.variant_info(1, i)
        except S.SandengineError:
            return i - 1
        i += 1


def world(name, W, H, sleep=True, sliced=True):
    w = S.World(_ctx, rs(name), W, H)
    w.frame = 1
    w.fill_seeded(5, *FILL[name], stone_rows=H // 2, stone_id=5)
    if sliced:
        w.set_variant(3, sliced_index(w))
        w.set_sleep(sleep)
    return w


def seeded_mods(W, H, seed, n):
    rng = np.random.RandomState(seed)
    return [(int(rng.randint(-40, W + 40)), int(rng.randint(-40, H + 40)), int(rng.randint(0, 3)), int(rng.randint(1, 60)),
             int(rng.randint(-1, 6))) for _ in range(n)]


# a record is kept from 1024 squares of 64 x 64 cells on; launches of 12, 16 and 32 steps
SIZES = {"four_materials": (2303, 2113), "twelve_materials": (2304, 2112), "features": (2500, 2001)}
SCRIPT = [("step", 20), ("step", 14), ("mods", 3), ("step", 25), ("step", 9), ("mods", 40), ("step", 2), ("step", 33),
          ("plain", 1), ("step", 12), ("step", 12), ("lds", 5), ("step", 13), ("upload", 0), ("step", 12), ("step", 12),
          ("unknown", 0), ("step", 11), ("step", 11), ("sub", 5), ("step", 12), ("clear", 0), ("step", 30), ("step", 10)]


@pytest.mark.parametrize("name", list(SIZES))
def test_sleeping_equals_plain_and_dense(name):
    W, H = SIZES[name]
    rs(name)
    worlds = {"plain": world(name, W, H, sliced=False), "sleep": world(name, W, H, True), "dense": world(name, W, H, False)}
    for at, (kind, arg) in enumerate(SCRIPT):
        print(f"[gpu] sliced sleep {name} {W}x{H} {at}: {kind} {arg}", flush=True)
        for label, w in worlds.items():
            if kind == "step":
                w.step(arg) if label == "plain" else w.step_blocked(arg)
            elif kind == "sub":
                w.step(21) if label == "plain" else w.step_blocked(21, arg)
            elif kind == "plain":
                w.step(arg)
            elif kind == "lds" and label != "plain":
                last = sliced_index(w)
                w.set_variant(3, w.variant_info(2, 0)[0] if w.variant_info(2, 0)[0] != last else 0)
                w.step_blocked(arg)
                w.set_variant(3, last)
            elif kind == "lds":
                w.step(arg)
            elif kind == "mods":
                for m in seeded_mods(W, H, at, arg):
                    w.push_modification(*m)
            elif kind == "upload":
                w.upload(w.download())
            elif kind == "unknown":  # squares of an id that no material has
                g = w.download()
                g[64:700, 64:900] = 200
                g[1200:1400, :] = 3
                w.upload(g)
            elif kind == "clear":
                w.frame = 0
        want = worlds["plain"].download()
        for label in ("sleep", "dense"):
            got = worlds[label].download()
            bad = np.argwhere(got != want)
            assert len(bad) == 0, f"{label}: {len(bad)} cells differ after {at} {kind} {arg}, first {bad[0]}"
    assert len({w.frame for w in worlds.values()}) == 1
    for w in worlds.values():
        w.close()


def test_a_caller_with_the_grids_address_writes_between_runs():
    """Once a grid's address was given out nothing is known of the grids: cells written
    through it between two runs are stepped."""
    print("\n[gpu] sliced sleep, a grid written through its address", flush=True)
    rs("four_materials")
    a = world("four_materials", 2304, 2112)
    b = world("four_materials", 2304, 2112, sliced=False)
    ptrs = []
    for w in (a, b):
        for _ in range(2):  # both grids of a world, by the step between
            p, pitch = ctypes.c_void_p(), ctypes.c_uint32()
            assert S.lib().se_world_device_ptr(w._p, ctypes.byref(p), ctypes.byref(pitch)) == 0
            ptrs.append(p.value)
            w.step(1)
    H = hip()
    rows = np.full((200, 2304), 4, np.uint32)
    for run in range(3):
        for w, (p0, p1) in ((a, ptrs[:2]), (b, ptrs[2:])):
            (w.step_blocked if w is a else w.step)(24)
            w.sync()
            # 24 steps: an even number of plain steps, one exchange of the grids in a sliced run
            cur = (p0 if run % 2 == 1 else p1) if w is a else p0
            ok(H.hipMemcpy(cur + 4 * 2304 * 1500, rows.ctypes.data, rows.nbytes, H2D))
        np.testing.assert_array_equal(a.download(), b.download())
    a.close()
    b.close()


@pytest.mark.parametrize("name", ["four_materials", "features"])
@pytest.mark.parametrize("size", [(1, 1), (124, 126), (700, 333), (70001, 3), (3, 70001), (2081, 2047)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_modifications_of_the_first_step(name, size):
    """Worlds whose first step is a plain one, and beyond 2048 squares worlds that take them into
    the packed grid, against the oracle: lists that travel by value and lists that do not, overlapping
    boxes, later entries over earlier ones, NULL materials that hide them, a list cut at
    size 0, boxes larger than the world, beside it and across its sides."""
    W, H = size
    print(f"\n[gpu] sliced modifications {name} {size}", flush=True)
    rs(name)
    blob = O.compile_ruleset(L.parse_string(S.bundled_ruleset(name)))
    g = O.fill(3, W, H, *FILL[name])
    for n, lst in enumerate([[(W // 2, H // 2, 0, 5, 3)], seeded_mods(W, H, 1, 8), seeded_mods(W, H, 2, 9),
                             seeded_mods(W, H, 3, 200),
                             [(0, 0, 1, 3, 4), (1, 1, 0, 4, 1), (2, 1, 1, 2, 3), (W, H, 0, 0, 3), (3, 3, 1, 9, 4)],
                             [(W // 2, H // 2, 1, 1 << 30, 3), (W // 3, 0, 0, 7, 0), (-5, H // 2, 0, 9, 4), (0, 0, 1, -3, 4)]]):
        w = world(name, W, H)
        w.upload(g)
        w.frame = 2 + n
        for m in lst:
            w.push_modification(*m)
        w.step_blocked(10 + n)
        cut = next((i for i, m in enumerate(lst) if m[3] == 0), len(lst))
        want = O.run(blob, g, 3 + n, 10 + n, [list(m) for m in lst[:cut]])
        np.testing.assert_array_equal(w.download(), want, err_msg=f"list {n}")
        w.close()
