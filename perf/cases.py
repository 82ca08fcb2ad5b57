"""The work that programs have this framework do, as cases to time.

Four kinds of call, over the sizes that the tests, the benchmark and the rule
sets of this repository use:

* ``frame``    one interactive frame: a brush is queued and the world advances one
  step with the plain kernel, with or without the colour and light images;
* ``episode``  a world is seeded on the device, optionally hit by brushes, and
  advanced many steps with the blocked path (a rollout, a benchmark run);
* ``batch``    worlds of uneven sizes and step counts advance together
  (``Batch.run``), both large rule sets mixed;
* ``grids``    the step over grids that the caller owns in torch memory
  (``grids_step_noalloc``), restored from a checkpoint before each run.

Grids come back as device views of the buffers that hold them; nothing is copied
to the host.  An episode starts from its own seeded fill each time, so a pass
finds the same contents however often it runs.
"""
import ctypes
import math

import numpy as np
import torch

import sandengine_amd as S

FILLS = {
    "four_materials": ([0, 3, 4], [60, 25, 15]),
    "twelve_materials": ([0] + list(range(3, 15)), [40] + [5] * 12),
    "features": ([0, 3, 4, 5, 6, 7], [40, 20, 12, 12, 8, 8]),
}
SOLID = {"four_materials": 5, "twelve_materials": 5, "features": 7}


def listed():
    return [
        # the smallest call: the interactive loop of a 256x256 world, one step and one brush
        dict(name="frame_256", kind="frame", rules="four_materials", w=256, h=256, render=False, brush=6, warm=0),
        # the interactive loop with what a renderer samples: grid, colour and light
        dict(name="frame_960x540_render", kind="frame", rules="four_materials", w=960, h=540, render=True, brush=9,
             warm=16),
        # single steps of a large world of odd size, as a viewer that shows every step takes them
        dict(name="frame_3001x2003", kind="frame", rules="twelve_materials", w=3001, h=2003, render=False, brush=40,
             warm=0),
        # a world as small as one tile, run for a long time: a serial chain of steps
        dict(name="episode_100x90", kind="episode", rules="four_materials", w=100, h=90, steps=500, brushes=0,
             stone=0.0),
        # an ordinary rollout with explosions and brushes at its start
        dict(name="episode_1000x700", kind="episode", rules="four_materials", w=1000, h=700, steps=200, brushes=4,
             stone=0.1),
        dict(name="episode_4096", kind="episode", rules="four_materials", w=4096, h=4096, steps=200, brushes=0,
             stone=0.0),
        # the benchmark's world: 16384x16384 with a stone floor
        dict(name="episode_16384", kind="episode", rules="four_materials", w=16384, h=16384, steps=100, brushes=0,
             stone=0.3),
        # many materials with SET and RAND: a ragged ordinary size, and the benchmark's
        dict(name="rich_1537x1111", kind="episode", rules="twelve_materials", w=1537, h=1111, steps=150, brushes=3,
             stone=0.0),
        dict(name="rich_8192", kind="episode", rules="twelve_materials", w=8192, h=8192, steps=64, brushes=0,
             stone=0.0),
        # a rule file with Right rules and raw rand lanes (neither table form fits it)
        dict(name="features_1280", kind="episode", rules="features", w=1280, h=1280, steps=100, brushes=0, stone=0.0),
        # the benchmark's batch at a size that a call of it usually has: uneven worlds, both rule sets
        dict(name="batch_48", kind="batch", rules="mixed", n=48, lo=64, hi=1024, steps_lo=100, steps_hi=1000,
             graph=True),
        # caller-owned grids between other work of a torch program
        dict(name="grids_40", kind="grids", rules="four_materials", n=40, lo=64, hi=512, steps_lo=20, steps_hi=200),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "episode", "episode", "episode", "batch", "grids"])
    rules = rng.choice(["four_materials", "four_materials", "twelve_materials", "twelve_materials", "features"])
    if kind == "frame":
        render = rng.random() < 0.4
        top = 1400 if render else 4096
        return dict(kind=kind, rules="four_materials" if render else rules, w=_log(rng, 64, top), h=_log(rng, 64, top),
                    render=render, brush=rng.randint(1, 60), warm=rng.randint(4, 16) if render else 0)
    if kind == "episode":
        w, h = _log(rng, 64, 8192), _log(rng, 64, 8192)
        # at most 16384^2 cells for 100 steps, and for the slower rule sets a fourth of that
        most = 16384 * 16384 * (100 if rules == "four_materials" else 16 if rules == "twelve_materials" else 8)
        steps = max(1, min(_log(rng, 8, 600), most // (w * h)))
        return dict(kind=kind, rules=rules, w=w, h=h, steps=steps, brushes=rng.choice([0, 0, 1, 4, 12]),
                    stone=rng.choice([0.0, 0.0, 0.1, 0.3]))
    if kind == "batch":
        return dict(kind=kind, rules=rng.choice(["mixed", "four_materials", "twelve_materials"]), n=rng.randint(4, 56),
                    lo=64, hi=rng.choice([128, 256, 512, 1024]), steps_lo=rng.choice([10, 50, 100]),
                    steps_hi=rng.choice([200, 500, 1000]), graph=rng.random() < 0.5)
    return dict(kind=kind, rules=rng.choice(["four_materials", "twelve_materials"]), n=rng.randint(1, 60),
                lo=rng.choice([33, 64, 100]), hi=rng.choice([128, 300, 512]), steps_lo=rng.choice([1, 8, 20]),
                steps_hi=rng.choice([20, 100, 200]))


# ------------------------------------------------------------------ what a program keeps
_CTX = None
_RULES = {}
_STREAM = None


def _context():
    global _CTX
    if _CTX is None:
        _CTX = S.Context(torch.cuda.current_device())
    return _CTX


def _stream():
    """The stream of every grids_step_noalloc call: calls on several streams would share its scratch array at once,
    which its contract rules out."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def _rules(name):
    if name not in _RULES:
        _RULES[name] = S.RuleSet(_context(), S.bundled_ruleset(name))
    return _RULES[name]


class _Memory:
    """A device buffer for torch, with the world that owns the memory: whoever holds the view holds the world."""

    def __init__(self, owner, ptr, shape, strides, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, strides=strides, typestr=typestr, version=2)


def _view(views, ptr, make):
    if ptr not in views:
        memory = make(ptr)
        views[ptr] = torch.as_tensor(memory, device=torch.device("cuda", torch.cuda.current_device()))
        views[ptr].owner = memory.owner
        assert views[ptr].data_ptr() == ptr  # in place, not a copy
    return views[ptr]


def _grid(world, views):
    """The world's current grid in place (a world has two buffers, each seen once)."""
    ptr, pitch = ctypes.c_void_p(), ctypes.c_uint32()
    S._check(S.lib().se_world_device_ptr(world._p, ctypes.byref(ptr), ctypes.byref(pitch)))
    return _view(views, ptr.value, lambda p: _Memory(world, p, (world.H, world.W), (pitch.value * 4, 4), "<i4"))


def _images(world, views):
    col, light, pitch = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_uint32()
    S._check(S.lib().se_world_render_ptrs(world._p, ctypes.byref(col), ctypes.byref(light), ctypes.byref(pitch)))
    return [_view(views, q.value, lambda p: _Memory(world, p, (world.H, world.W, 4), (pitch.value * 16, 16, 4), "<f4"))
            for q in (col, light)]


def _specs(case, seed):
    """Sides, rule sets, step counts and seeds of the worlds of a batch."""
    rng = np.random.RandomState(seed % (1 << 31))
    out = []
    for i in range(case["n"]):
        side = [max(1, int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))))) for _ in range(2)]
        rules = case["rules"] if case["rules"] != "mixed" else ("four_materials", "twelve_materials")[rng.randint(2)]
        out.append((side[0], side[1], rules, int(rng.randint(case["steps_lo"], case["steps_hi"] + 1)),
                    int(rng.randint(1 << 20))))
    return out


def _sizes(case):
    """The sizes of a batch do not depend on the inputs' seed: what is timed is one shape."""
    return _specs(case, 4242)


def _host_fill(case, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    ids, pct = FILLS[case["rules"]]
    g = rng.choice(np.array(ids, np.uint32), size=(case["h"], case["w"]), p=np.array(pct) / 100.0)
    return np.ascontiguousarray(g, dtype=np.uint32)


def _brush(case, k):
    """The brush of frame k: sand, water or a hole, moving over the world."""
    return ((37 + 61 * k) % case["w"], (11 + 23 * k) % case["h"], k % 2, case["brush"], (3, 4, 0)[k % 3])


def _frame(state):
    world, case = state["world"], state["case"]
    world.push_modification(*_brush(case, state["k"]))
    state["k"] += 1
    world.step(1)


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    if kind == "frame":
        world = S.World(ctx, _rules(case["rules"]), case["w"], case["h"])
        if case["render"]:
            world.set_render(True)
        world.frame = 1
        world.upload(_host_fill(case, seed))
        state = dict(case=case, world=world, views={}, k=0)
        for _ in range(case["warm"]):
            _frame(state)
        return state
    if kind == "episode":
        world = S.World(ctx, _rules(case["rules"]), case["w"], case["h"])
        rng = np.random.RandomState(seed % (1 << 31))
        mods = [(int(rng.randint(case["w"])), int(rng.randint(case["h"])), int(rng.randint(2)),
                 int(rng.randint(2, 65)), (0, 3, 4)[rng.randint(3)]) for _ in range(case["brushes"])]
        return dict(case=case, world=world, views={}, seed=seed % (1 << 24), mods=mods)
    if kind == "batch":
        batch, worlds = S.Batch(ctx), []
        for i, (w, h, rules, steps, _) in enumerate(_sizes(case)):
            world = S.World(ctx, _rules(rules), w, h)
            world.frame = 1
            ids, pct = FILLS[rules]
            world.fill_seeded((seed * 64 + i) % (1 << 24), ids, pct)
            batch.add(world, steps)
            worlds.append(world)
        return dict(case=case, batch=batch, worlds=worlds, views={})
    grids, at = [], 0
    for w, h, _, steps, _ in _sizes(case):
        pitch = (w + 63) // 64 * 64
        grids.append(dict(w=w, h=h, pitch=pitch, at=at, steps=steps))
        at += pitch * h
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    ids, pct = FILLS[case["rules"]]
    edges = torch.tensor(np.cumsum(pct)[:-1] / 100.0, dtype=torch.float32, device="cuda")
    draws = torch.bucketize(torch.rand(at, generator=gen, device="cuda"), edges, right=True)
    init = torch.tensor(ids, dtype=torch.int32, device="cuda")[draws].contiguous()
    arena = torch.zeros((2, at), dtype=torch.int32, device="cuda")
    return dict(case=case, grids=grids, init=init, arena=arena, stream=_stream(), rules=_rules(case["rules"]))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        _frame(state)
        out = [_grid(state["world"], state["views"])]
        return out + _images(state["world"], state["views"]) if case["render"] else out
    if kind == "episode":
        world = state["world"]
        ids, pct = FILLS[case["rules"]]
        world.frame = 1
        world.fill_seeded(state["seed"], ids, pct, stone_rows=int(case["stone"] * case["h"]),
                          stone_id=SOLID[case["rules"]])
        for m in state["mods"]:
            world.push_modification(*m)
        world.step_blocked(case["steps"])
        return [_grid(world, state["views"])]
    if kind == "batch":
        state["batch"].run(graph=case["graph"])
        return [_grid(w, state["views"]) for w in state["worlds"]]
    arena, stream = state["arena"], state["stream"]
    with torch.cuda.stream(stream):
        arena[0].copy_(state["init"], non_blocking=True)
        base = [arena[0].data_ptr(), arena[1].data_ptr()]
        done = S.grids_step_noalloc(
            _context(), state["rules"],
            [dict(grid0=base[0] + 4 * g["at"], grid1=base[1] + 4 * g["at"], w=g["w"], h=g["h"], pitch=g["pitch"],
                  cur=0, frame=1, nsteps=g["steps"]) for g in state["grids"]], stream=stream.cuda_stream)
    return [arena[cur][g["at"]:g["at"] + g["pitch"] * g["h"]].view(g["h"], g["pitch"])[:, :g["w"]]
            for g, (cur, _) in zip(state["grids"], done)]


def work(case):
    """Bytes: each cell read once and written once, and the images of a frame.  flops: one operation per cell and
    step, as integer work (a cell is decided once in each step)."""
    kind = case["kind"]
    if kind in ("batch", "grids"):
        cells = [(w * h, steps) for w, h, _, steps, _ in _sizes(case)]
        return dict(bytes=8 * sum(c for c, _ in cells), flops=sum(c * s for c, s in cells))
    cells = case["w"] * case["h"]
    if kind == "frame":  # light and noise in, colour and light out
        return dict(bytes=cells * (8 + (52 if case["render"] else 0)), flops=cells)
    return dict(bytes=8 * cells, flops=cells * case["steps"])


# ------------------------------------------------------------------ the light of a frame in 64 bits
def _hash_x(ox, oy, frame):
    """First hash word of every block (origins ox by oy)."""
    n = (ox[None, :] * np.int64(461) + oy[:, None] * np.int64(2131) + np.int64(frame) * 4541161) * 213
    h = (n & 0xFFFFFFFF).astype(np.uint32)
    h ^= h >> np.uint32(16)
    h *= np.uint32(0x7FEB352D)
    h ^= h >> np.uint32(15)
    h *= np.uint32(0x846CA68B)
    return h ^ (h >> np.uint32(16))


def _step(grid, frame, mod):
    """One step of the four-material rules: 2x2 blocks at the frame's offset, sand and water falling."""
    h, w = grid.shape
    ox, oy = ((0, 0), (1, 1), (0, 1), (1, 0))[frame % 4]
    nx, ny = (w + ox + 1) // 2, (h + oy + 1) // 2
    pad = np.full((2 * ny, 2 * nx), 2, np.uint32)  # cells outside the world are wall
    pad[oy:oy + h, ox:ox + w] = grid
    a, b, c, d = (pad[y::2, x::2].copy() for y in (0, 1) for x in (0, 1))
    mirror = _hash_x(2 * np.arange(nx, dtype=np.int64) - ox, 2 * np.arange(ny, dtype=np.int64) - oy,
                     frame).astype(np.float32) * np.float32(2.0 ** -32) < np.float32(0.5)

    def swap(p, q, where):
        ok = where & (p != 1) & (p != 2) & (q != 1) & (q != 2)
        t = p[ok].copy()
        p[ok] = q[ok]
        q[ok] = t

    swap(a, b, mirror)
    swap(c, d, mirror)
    is_a = a == 3
    down = is_a & (c == 0)
    right = is_a & ~down & (d == 0)
    swap(a, c, down)
    swap(a, d, right)
    is_a = a == 4
    down = is_a & (c == 0)
    slide = is_a & ~down & (d == 0)
    flow = is_a & ~down & ~slide & (b == 0)
    swap(a, c, down)
    swap(a, d, slide)
    swap(a, b, flow)
    swap(a, b, mirror)
    swap(c, d, mirror)
    for (y, x), v in zip(((0, 0), (0, 1), (1, 0), (1, 1)), (a, b, c, d)):
        pad[y::2, x::2] = v
    new = pad[oy:oy + h, ox:ox + w].copy()
    mx, my, shape, size, mat = mod
    dx, dy = np.abs(np.arange(w) - mx)[None, :], np.abs(np.arange(h) - my)[:, None]
    hit = (dx * dx + dy * dy <= size * size) if shape == 0 else ((dx <= size) & (dy <= size))
    new[hit] = mat
    return new


def _light(prev, light):
    """Light of the next frame: full on row 0, else half the mean and half the maximum of the neighbours' light
    (no material of these rules emits; all but empty cells pass only the falloff)."""
    h, w = prev.shape
    passes = (prev == 0)[..., None]
    term = np.concatenate([np.where(passes, light[..., :3], 0.0) * light[..., 3:], light[..., 3:]], axis=2)
    padded = np.zeros((h + 2, w + 2, 4))
    padded[1:-1, 1:-1] = term
    inside = np.zeros((h + 2, w + 2), bool)
    inside[1:-1, 1:-1] = True
    total, top, n, falloff = np.zeros((h, w, 4)), np.zeros((h, w, 4)), np.zeros((h, w)), np.zeros((h, w))
    for dx, dy in ((0, 1), (0, -1), (-1, 1), (-1, -1), (1, 1), (1, -1), (1, 0), (-1, 0)):
        here = np.s_[1 + dy:1 + dy + h, 1 + dx:1 + dx + w]
        inn, t = inside[here], padded[here].copy()
        t[..., 3] = np.where(t[..., 3] == 0.0, falloff, t[..., 3])
        total += np.where(inn[..., None], t, 0.0)
        top = np.where(inn[..., None], np.maximum(top, t), top)
        falloff = np.where(inn, np.maximum(falloff, t[..., 3]), falloff)
        n += inn
    mean = total / np.maximum(n, 1)[..., None]
    out = mean * 0.5 + top * 0.5
    out[..., 3] = mean[..., 3]
    out[0] = (1.0, 1.0, 1.0, np.float64(np.float32(0.999999)))
    return out


def exact(case, seed):
    """Grids are whole numbers.  The colour has no value in 64 bits: its noise is fract(sin(x) * 43758.5), whose
    digits are those of the 32-bit sine.  The light has one."""
    if case["kind"] != "frame" or not case["render"]:
        return None
    if case["w"] * case["h"] * (case["warm"] + 1) > 10_000_000:
        return None  # numpy would take over ten seconds
    grid, light = _host_fill(case, seed), np.zeros((case["h"], case["w"], 4))
    for k in range(case["warm"] + 1):
        new = _step(grid, k + 2, _brush(case, k))
        light = _light(grid, light)
        grid = new
    return [None, None, torch.from_numpy(light)]
