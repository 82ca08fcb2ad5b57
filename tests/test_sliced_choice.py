"""The choice between the LDS and the sliced kernels, on the host: calls on both sides of
the rule whose two paths were timed (us, LDS / sliced, in the comments)."""
import os
import subprocess
import tempfile

import pytest

import sandengine_amd as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include "CSRC/se_sliced.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
using namespace se_rt;
int main(int argc, char** argv) {
    SlicedKernels K;
    K.ok = true;
    K.cost.form = atoi(argv[2]);
    K.cost.wall_kept = atoi(argv[3]) != 0;
    K.cost.tables = atoi(argv[4]);
    K.cost.hash_ops = atoi(argv[5]);
    K.classes = atoi(argv[6]);
    if (atoi(argv[7])) K.step[0] = (hipFunction_t)1;
    const unsigned W = atoi(argv[8]), H = atoi(argv[9]), n = atoi(argv[10]), worlds = atoi(argv[11]), apart = atoi(argv[12]);
    if (!strcmp(argv[1], "one")) {
        printf("%d\n", sliced_pays(K, W, H, n));
    } else {
        std::vector<SlicedLoad> v;
        for (unsigned i = 0; i < worlds; i++) v.push_back({W, H, n, (int)(2 + apart * i)});
        printf("%d\n", sliced_batch_pays(K, v));
    }
    return 0;
}
"""

# form of the LDS kernels, WALL kept, tables, hash instructions, hash planes, one-wavefront tiles
FOUR, TWELVE, FEATURES = (1, 1, 78, 11, 1, 1), (2, 1, 246, 26, 4, 0), (0, 0, 102, 46, 5, 1)
TABLES_618, TABLES_1661 = (1, 0, 618, 22, 2, 1), (1, 0, 1661, 22, 2, 1)
ONE = [
    (FOUR, 2, 2, 9, 0), (FOUR, 2, 2, 24, 0), (FOUR, 2, 2, 128, 1),            # 19 / 27, 25 / 31, 71 / 63
    (FOUR, 32, 32, 16, 0), (FOUR, 32, 32, 48, 1), (FOUR, 64, 64, 9, 0), (FOUR, 64, 64, 16, 1),  # 27 / 28, 50 / 38, 26 / 28, 33 / 29
    (FOUR, 256, 256, 8, 0), (FOUR, 256, 256, 9, 1), (FOUR, 16384, 16384, 9, 1), (FOUR, 200, 40000, 9, 1),  # -, 43 / 30, -, 62 / 54
    (FOUR, 20000, 16, 16, 0), (FOUR, 20000, 16, 64, 1), (FOUR, 300000, 8, 48, 0),  # 28 / 34, 79 / 64, 174 / 202
    (TWELVE, 2, 2, 9, 0), (TWELVE, 64, 64, 12, 1), (TWELVE, 8192, 8192, 9, 1), (TWELVE, 20000, 4, 16, 0),  # 25 / 31, 41 / 33, 345 / 207, 41 / 45
    (FEATURES, 2, 2, 4, 0), (FEATURES, 64, 64, 4, 1), (FEATURES, 1024, 1024, 4, 1),  # 23 / 28, 34 / 29, -
    (FEATURES, 20000, 1, 12, 0), (FEATURES, 300000, 8, 128, 0), (FEATURES, 20000, 128, 4, 1),  # 28 / 44, 643 / 1632, 55 / 39
    (TABLES_618, 4096, 4096, 16, 0), (TABLES_618, 4096, 4096, 96, 1),          # 152 / 179, 849 / 713
    (TABLES_1661, 64, 64, 64, 0), (TABLES_1661, 4096, 4096, 64, 0),            # 87 / 259, 565 / 901
]
BATCH = [  # worlds, all at one first frame (0) or each at its own
    (FOUR, 64, 64, 9, 1000, 0, 0), (FOUR, 64, 64, 100, 1000, 0, 1),            # 122 / 131 (512 worlds), 271 / 182
    (FOUR, 64, 64, 256, 2048, 3, 0), (FOUR, 64, 64, 256, 2048, 0, 1),          # 956 / 2325, 966 / 408
    (FOUR, 300, 300, 100, 64, 3, 1), (FOUR, 120, 120, 128, 512, 3, 1),         # 600 / 290, 1177 / 327
    (TWELVE, 16, 16, 256, 2048, 3, 0), (TWELVE, 120, 120, 64, 512, 3, 1), (TWELVE, 300, 300, 9, 512, 0, 1),  # 1618 / 3432, 1104 / 468, 451 / 278
    (FOUR, 300, 300, 0, 5, 0, 0),
]


@pytest.fixture(scope="module")
def program():
    csrc, pkg = os.path.join(ROOT, "sandengine_amd", "csrc"), os.path.dirname(S.__file__)
    with tempfile.TemporaryDirectory() as d:
        cpp, exe = os.path.join(d, "choice.cpp"), os.path.join(d, "choice")
        with open(cpp, "w") as f:
            f.write(MAIN.replace("CSRC", csrc))
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe, cpp,
                               "-L" + pkg, "-l:libsandengine_hip.so", "-Wl,-rpath," + pkg, "-Wl,--allow-shlib-undefined"])
        yield exe


@pytest.mark.parametrize("case", ONE, ids=[f"{c[0][2]}_{c[1]}x{c[2]}_{c[3]}" for c in ONE])
def test_world(program, case):
    rules, w, h, n, sliced = case
    assert int(subprocess.check_output([program, "one", *map(str, (*rules, w, h, n, 1, 0))])) == sliced


@pytest.mark.parametrize("case", BATCH, ids=[f"{c[0][2]}_{c[4]}x{c[1]}_{c[3]}_{c[5]}" for c in BATCH])
def test_batch(program, case):
    rules, w, h, n, worlds, apart, sliced = case
    assert int(subprocess.check_output([program, "batch", *map(str, (*rules, w, h, n, worlds, apart))])) == sliced


def test_costs_of_the_bundled_sets():
    """What the rule goes by is what the generator says of the rule sets."""
    for name, tables, planes in (("four_materials", 78, 1), ("twelve_materials", 246, 4), ("features", 102, 5)):
        src = S.emit_hip(S.bundled_ruleset(name))
        line = src[src.find("// ---- sliced form"):].split("\n", 1)[0]
        assert f"{planes} hash planes, {tables} tables" in line


def test_a_network_too_large_beside_a_table_is_left_out():
    """Many rules over few materials: a full table, and more than 1000 tables in the network."""
    mats = "abcd"
    rules, names = "", []
    for i in range(150):
        a, b, c = mats[i % 4] * 3, mats[(i // 4) % 4] * 3, ("SELF", "RIGHT", "DOWN", "DOWNRIGHT")
        x, y = c[i % 4], c[(i // 3) % 4 if (i // 3) % 4 != i % 4 else (i + 1) % 4]
        cond = f"{x}.mat != {a} and isType_EMPTY({y})" if i % 3 else f"{x}.mat == {a} and SELF.mat.density > DOWN.mat.density"
        rules += f"  r{i}:\n    if: {cond}\n    probability: 0.5\n    do: {'SWAP ' + x + ' ' + y if i % 2 else 'SET ' + y + ' ' + b}\n"
        names.append(f"r{i}")
    text = ("rules:\n" + rules + "types:\n  base:\n    base_rules: [" + ", ".join(names) + "]\nmaterials:\n" +
            "".join(f"  {m * 3}:\n    type: base\n    color: [0.5, 0.5, 0.5]\n    density: {1 + i}.0\n" for i, m in enumerate(mats)))
    src = S.emit_hip(text)
    assert "#define SE_TBL 1" in src and "// ---- sliced form" not in src
