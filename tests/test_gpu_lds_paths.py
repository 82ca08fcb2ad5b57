"""The LDS kernels on the runs that their defaults now leave to the sliced ones: tile
sleeping and waking, tiles of longer runs and batches of tables that change WALL or have
several hash classes, each with the LDS variant named."""
import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O
from tests import test_gpu_batch as B
from tests import test_gpu_parity as P
from tests import test_gpu_sleep as Z

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["four_materials", "twelve_materials"])
def test_sleeping_lds_tiles_wake(name):
    r = Z.rs(name)
    worlds = {"plain": Z.floor_world(r, 1536, 5), "sleep": Z.floor_world(r, 1536, 5, True),
              "dense": Z.floor_world(r, 1536, 5, False)}
    lds = worlds["sleep"].variant_info(2, 0)[0]
    for label in ("sleep", "dense"):
        worlds[label].set_variant(3, lds)
    for at, (kind, arg) in enumerate(Z.SCRIPT):
        print(f"[gpu] LDS sleep {name} {at}: {kind} {arg}", flush=True)
        for label, w in worlds.items():
            if kind == "blocked":
                w.step(arg) if label == "plain" else w.step_blocked(arg, 8)
            elif kind == "plain":
                w.step(arg)
            elif kind == "mods":
                for m in arg:
                    w.push_modification(*m)
            elif kind == "variant" and label != "plain":
                w.set_variant(3, lds if arg < 0 else arg)
            elif kind == "reupload":
                w.upload(w.download())
        want = worlds["plain"].download()
        for label in ("sleep", "dense"):
            bad = int((worlds[label].download() != want).sum())
            assert bad == 0, f"{label} differs from plain in {bad} cells after {kind} {arg}"
    for w in worlds.values():
        w.close()


@pytest.mark.parametrize("rules", ["_erode_rules", "_three_class_rules"])
def test_tables_in_lds_batches(rules):
    print(f"\n[gpu] LDS batch {rules}", flush=True)
    text = getattr(P, rules)()
    r = S.RuleSet(B.ctx(), text)
    blob = O.compile_ruleset(L.parse_string(text))
    for persistent in (2, 3):
        b, cases = S.Batch(B.ctx()), []
        for i, (W, H, steps) in enumerate([(64, 64, 90), (150, 90, 57), (300, 260, 33), (31, 17, 120)]):
            g = O.fill(70 + i, W, H, [0, 3, 4, 5], [50, 25, 15, 10])
            if i % 2 == 0:
                g[H // 3:H // 3 + 4, W // 4:W // 4 + 6] = 77
            w = S.World(B.ctx(), r, W, H)
            w.frame = 1
            w.upload(g)
            b.add(w, steps)
            cases.append((w, g, steps))
        b.run(mode=persistent, variant=cases[0][0].variant_info(2, 0)[0])
        for w, g, steps in cases:
            np.testing.assert_array_equal(w.download(), O.run(blob, g, 2, steps))
            w.close()
        b.close()


@pytest.mark.parametrize("name", ["four_materials", "twelve_materials"])
@pytest.mark.parametrize("sub", [3, 8])
def test_longer_runs_of_lds_tiles(name, sub):
    print(f"\n[gpu] LDS {name} {sub} sub-steps a launch", flush=True)
    r = B.rs(name)
    blob = O.compile_ruleset(L.parse_string(S.bundled_ruleset(name)))
    for W, H in ((112, 112), (113, 112), (389, 211)):
        g = O.fill(5, W, H, *B.FILLS[name])
        w = S.World(B.ctx(), r, W, H)
        w.upload(g)
        w.frame = 3
        w.set_variant(3, w.variant_info(2, 0)[0])
        w.push_modification(W // 2, H // 3, 0, 9, 3)
        w.step_blocked(29, sub)
        np.testing.assert_array_equal(w.download(), O.run(blob, g, 4, 29, [[W // 2, H // 3, 0, 9, 3]]))
        w.close()
