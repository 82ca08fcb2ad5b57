"""hipGraph capture of a batch's LDS launches: alone, and beside rule sets of the same batch
that take the sliced kernels (submitted directly).  Every run captures and launches a graph
of its own, with eager work and synchronizations between the runs, and is compared with
per-world plain steps."""
import numpy as np
import pytest

import sandengine_amd as S
from tests import test_gpu_batch as B

pytestmark = pytest.mark.gpu


def pairs(spec):
    out = []
    for i, (name, w, h, steps, frame) in enumerate(spec):
        x, y = S.World(B.ctx(), B.rs(name), w, h), S.World(B.ctx(), B.rs(name), w, h)
        for v in (x, y):
            v.frame = frame
            v.fill_seeded(30 + i, *B.FILLS[name])
        out.append((x, y, steps))
    return out


def default_lds(w):
    return w.variant_info(2, 0)[0]


def check(b, worlds, **run):
    for x, _, steps in worlds:
        b.add(x, steps)
    for rep in range(3):
        assert b.run(graph=True, **run) > 0
        for x, y, steps in worlds:
            y.step(steps)
            assert x.frame == y.frame
            np.testing.assert_array_equal(x.download(), y.download(), err_msg=f"run {rep}: {x.W}x{x.H} {steps}")
        worlds[0][0].step(1)  # the plain kernel between two graphs
        worlds[0][1].step(1)
    b.close()
    for x, y, _ in worlds:
        x.close()
        y.close()


def test_graph_of_lds_plans():
    """Both rule sets by their LDS kernels: one-tile worlds, and rounds over the others."""
    print("\n[gpu] batch graph, LDS kernels", flush=True)
    worlds = pairs([(("four_materials", "twelve_materials")[i % 2], w, h, 9 + 17 * i, 1 + i % 5)
                    for i, (w, h) in enumerate([(64, 64), (112, 112), (1, 300), (300, 260), (513, 257), (113, 40)])])
    check(S.Batch(B.ctx()), worlds, mode=2, variant=default_lds(worlds[0][0]))


def test_graph_of_lds_plans_beside_sliced_plans():
    """Four materials run long and take the sliced kernels; twelve run 6 steps."""
    print("\n[gpu] batch graph, LDS kernels beside sliced ones", flush=True)
    worlds = pairs([("four_materials", 200 + 30 * i, 300, 100 + i, 1 + i % 2) for i in range(6)] +
                   [("four_materials", 64, 64, 120, 1)] +
                   [("twelve_materials", 64 + 60 * i, 90, 6, 1 + i) for i in range(5)])
    check(S.Batch(B.ctx()), worlds, mode=1)
