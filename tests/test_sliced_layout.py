"""Layout of the sliced kernels' hash planes, on the host: for worlds over the range of
sizes, start frames and run lengths, every word that the step kernel reads (its loads
ahead included) lies in the room that the run allocates, and every word used holds the
hash inputs of its blocks.  The addresses are worked out here from the layout's
description, not with the library's code."""
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
using namespace se_rt;
typedef unsigned int u32;
typedef long long i64;
static void offset(i64 f, int& ox, int& oy) { ox = (int)(f & 1); oy = (f & 3) == 1 || (f & 3) == 2; }
static u32 input(i64 x, i64 y, i64 f) { return (u32)(461 * x + 2131 * y + 4541161 * f); }
// word of block row j, block column b (a word's first) in frame f, and its bit
static void locate(const SlicedGrid& g, i64 f, i64 b, i64 j, i64& word, i64& bit) {
    if (!g.hash_shared) {
        word = (f - g.hash_frame0) * (i64)g.hash_words + (b >> 5) * g.hash_pitch + j;
        bit = b & 31;
        return;
    }
    int ox, oy;
    offset(f, ox, oy);
    const int set = (int)((ox + oy + f) & 1);
    const u32 n = input(2 * b - ox - g.xpad, 2 * j + oy - g.ypad, f);
    const i64 m = (u32)(n - (set ? g.hash_n1 : g.hash_n0)) / 2;
    for (i64 a = 0; a < 461; a++)
        if ((m - 2131 * a) % 461 == 0) {
            const i64 c = (m - 2131 * a) / 461 + 2144;
            word = set * (i64)g.hash_words + (c >> 5) * g.hash_pitch + a;
            bit = c & 31;
            return;
        }
    exit(3);
}
int main(int argc, char** argv) {
    const int W = atoi(argv[1]), H = atoi(argv[2]), planes = atoi(argv[3]), classes = atoi(argv[4]);
    const u32 sub = atoi(argv[5]), n = atoi(argv[6]);
    const int frame0 = atoi(argv[7]);
    SlicedKernels K;
    K.step[0] = planes <= 3 ? (hipFunction_t)1 : nullptr;
    SlicedShape s = sliced_one_tile(W, H, true);
    if (!s.nw) {
        int kernel;
        u32 deep;
        sliced_choice(sliced_squares(W, H), K, &kernel, &deep);
        s = sliced_tiles(W, H, kernel, sub ? std::min(sub, deep) : deep);
    }
    SlicedGrid g;
    sliced_geometry(s, W, H, g);
    const SlicedAhead plan = sliced_ahead(s, g, frame0, n, classes);
    const i64 room = (i64)(plan.bytes / 4 / classes);
    int forms = 0;
    for (u32 at = 0; at < n; at += plan.frames) {
        const u32 nf = std::min(plan.frames, n - at);
        const i64 f0 = (i64)frame0 + at, waves = s.threads / 64, nw = s.nw / waves;
        const size_t need = sliced_hash_layout(g, (int)f0, nf, classes);
        forms |= g.hash_shared ? 2 : 1;
        if (need > plan.bytes) { printf("chunk at %u of %u frames needs %zu of %zu bytes\n", at, nf, need, plan.bytes); return 1; }
        if ((i64)g.hash_sets * g.hash_words > room) { printf("planes written past the room\n"); return 1; }
        for (i64 f = f0; f < f0 + nf + 4; f++) {  // four frames past the last are loaded
            if (f > f0 + 3 && f < f0 + nf - 2 && (f - f0) % 61) continue;
            for (int k = 0; k < 9; k++) {  // tiles at the corners, the sides and inside
                const int tx = k % 3 == 0 ? 0 : k % 3 == 1 ? s.tiles_x / 2 : s.tiles_x - 1;
                const int ty = k / 3 == 0 ? 0 : k / 3 == 1 ? s.tiles_y / 2 : s.tiles_y - 1;
                for (i64 wv = 0; wv < waves; wv++) {
                    const i64 b0 = 8 * (tx * (4 * s.nw - 2 * s.side) + 4 * nw * wv);
                    const i64 row0 = ty * (64 * s.r - 2 * s.halo);
                    for (i64 j : {row0 / 2, row0 / 2 + 32 * s.r - 1}) {
                        i64 word, bit;
                        locate(g, f, b0, j, word, bit);
                        const i64 last = word + nw * g.hash_pitch;
                        if (word < 0 || last >= room) {
                            printf("%s form: word %lld of %lld, frame %lld of chunk at %u\n", g.hash_shared ? "shared" : "direct",
                                   last, room, f, at);
                            return 1;
                        }
                        if (f < f0 + nf && last - g.hash_pitch * (bit ? 0 : 1) >= (i64)g.hash_sets * g.hash_words) {
                            printf("a word used is never hashed: %lld\n", last);
                            return 1;
                        }
                        // 32 * nw blocks on, the same place plus nw words
                        i64 w2, bit2;
                        locate(g, f, b0 + 32 * nw, j, w2, bit2);
                        if (f < f0 + nf && (w2 != last || bit2 != bit)) { printf("a block row is no run of bits\n"); return 1; }
                    }
                }
            }
        }
    }
    printf("ok %d\n", forms);
    return 0;
}
"""

# W, H, planes, hash planes, sub-steps a launch (0: the choice), steps, first frame
CASES = [
    (1, 1, 3, 1, 0, 500, 2), (100, 90, 3, 1, 0, 5000, 3), (251, 126, 4, 4, 0, 100, 1), (252, 127, 3, 5, 7, 64, 2),
    (1000, 700, 3, 1, 0, 200, 2), (4096, 4096, 3, 1, 0, 200, 5), (5003, 4999, 4, 4, 0, 45, 3),
    (16384, 16384, 3, 1, 0, 100, 2), (16384, 16384, 3, 8, 0, 900, 2147482000), (9001, 2801, 4, 4, 0, 38, 2147483000),
    # runs whose last chunk takes the other form
    (131039, 106, 3, 5, 16, 45, 2), (104831, 133, 3, 5, 4, 213, 2), (771, 35811, 3, 5, 4, 213, 2),
    (251, 136616, 3, 2, 4, 213, 2), (636558, 195, 4, 5, 0, 17, 9), (922252, 274, 3, 6, 12, 89, 4),
]


@pytest.fixture(scope="module")
def program():
    csrc, pkg = os.path.join(ROOT, "sandengine_amd", "csrc"), os.path.dirname(S.__file__)
    with tempfile.TemporaryDirectory() as d:
        cpp, exe = os.path.join(d, "layout.cpp"), os.path.join(d, "layout")
        with open(cpp, "w") as f:
            f.write(MAIN.replace("CSRC", csrc))
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe, cpp,
                               "-L" + pkg, "-l:libsandengine_hip.so", "-Wl,-rpath," + pkg, "-Wl,--allow-shlib-undefined"])
        yield exe


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c[:2])) + f"_{c[4]}_{c[5]}" for c in CASES])
def test_hash_planes_fit_and_hold_their_blocks(program, case):
    p = subprocess.run([program, *map(str, case)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
