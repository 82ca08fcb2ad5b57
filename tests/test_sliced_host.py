"""The sliced form of a rule set (cells as bit planes, the rule chain as a
network of three-input tables over words of 32 blocks), compiled for the host,
against the oracle's simulate() on every tuple of ids under hash words at both
sides of every threshold: equality, cell for cell."""
import os
import subprocess
import tempfile

import numpy as np
import pytest

import sandengine_amd as S
from oracle import lang_ref as L
from oracle import oracle as O
from tests import test_hip_backend_host as H

MAIN = r"""
static std::vector<char> slurp(const char* p) {
    FILE* f = fopen(p, "rb"); std::vector<char> v;
    if (!f) exit(2);
    char b[65536]; size_t n;
    while ((n = fread(b, 1, sizeof b, f)) > 0) v.insert(v.end(), b, b + n);
    fclose(f); return v;
}
int main(int argc, char** argv) {
    std::vector<char> hb = slurp(argv[1]);
    const uint32_t* hs = (const uint32_t*)hb.data();
    const size_t nh = hb.size() / 16, N = SE_NMAT, nt = N * N * N * N;
    const uint32_t cw[4] = {SE_SL_CODE0, SE_SL_CODE1, SE_SL_CODE2, SE_SL_CODE3};
    const uint32_t iw[4] = {SE_SL_ID0, SE_SL_ID1, SE_SL_ID2, SE_SL_ID3};
    std::vector<uint8_t> out(nt * nh * 4);
    for (size_t t = 0; t < nt; t++)
        for (size_t k0 = 0; k0 < nh; k0 += 32) {
            unsigned c[4][SE_SL_K], h[SE_SL_P];
            size_t id[4] = {t % N, t / N % N, t / N / N % N, t / N / N / N};
            for (int j = 0; j < 4; j++)
                for (int k = 0; k < SE_SL_K; k++)
                    c[j][k] = ((cw[id[j] / 4] >> (8 * (id[j] & 3)) >> k) & 1) ? ~0u : 0u;
            for (int p = 0; p < SE_SL_P; p++) h[p] = 0;
            for (size_t k = k0; k < nh && k < k0 + 32; k++)
                for (int p = 0; p < SE_SL_P; p++)
                    h[p] |= (unsigned)(hs[4 * k + se_sliced_class_lane(p)] <= se_sliced_class_max(p)) << (k - k0);
            se_sliced_block(c[0], c[1], c[2], c[3], h);
            for (size_t k = k0; k < nh && k < k0 + 32; k++)
                for (int j = 0; j < 4; j++) {
                    unsigned code = 0;
                    for (int p = 0; p < SE_SL_K; p++) code |= ((c[j][p] >> (k - k0)) & 1u) << p;
                    out[(t * nh + k) * 4 + j] = (iw[code / 4] >> (8 * (code & 3))) & 0xff;
                }
        }
    FILE* f = fopen(argv[2], "wb"); fwrite(out.data(), 1, out.size(), f); fclose(f);
    return 0;
}
"""

# v_bitop3_b32: bit i of the result is the table's entry (a_i, b_i, c_i), a the high bit
SHIM = r"""
static inline unsigned __builtin_amdgcn_bitop3_b32(unsigned a, unsigned b, unsigned c, int t) {
    unsigned r = 0;
    for (int m = 0; m < 8; m++)
        if ((t >> m) & 1) r |= (m & 4 ? a : ~a) & (m & 2 ? b : ~b) & (m & 1 ? c : ~c);
    return r;
}
"""

# corners of the network builder: conditions over two cells that are not density
# ranks, equal densities compared, a rule that acts on blocks of four EMPTY cells
CORNERS = """
rules:
  number:
    if: SELF.mat.id < RIGHT.mat.type or SELF.mat.density == DOWN.mat.density
    do: SWAP SELF DOWN
  rank:
    if: SELF.mat.density >= RIGHT.mat.density and SELF.mat != silt
    do: SWAP SELF RIGHT
    mirrored: false
  grow:
    if: rand.z >= 0.75
    do: [SET DOWN moss, SWAP DOWN DOWNRIGHT, SET SELF WALL]
    precondition: false
types:
  base:
    base_rules: [number, rank, grow]
materials:
  moss:
    type: base
    color: [0.5, 0.5, 0.5]
    density: 1.5
  clay:
    type: base
    color: [0.5, 0.5, 0.5]
    density: 1.5
  silt:
    type: base
    color: [0.5, 0.5, 0.5]
    density: 0.5
"""


def sets():
    return [(n, t) for n, t in H.cases() if t is not None] + [("corners", CORNERS)]


@pytest.mark.parametrize("name,text", sets(), ids=[c[0] for c in sets()])
def test_sliced_block_matches_oracle(name, text):
    src = S.emit_hip(text)
    a, b = src.find("// ---- sliced form"), src.find("// Sliced kernels")
    assert 0 < a < b, "this rule set has a sliced form"
    res = L.parse_string(text)
    blob, nid = O.compile_ruleset(res), len(res.materials)
    with tempfile.TemporaryDirectory() as d:
        hs = H.hash_words(H.build_harness(d, text), 7)
        cpp, exe = os.path.join(d, "s.cpp"), os.path.join(d, "s")
        with open(cpp, "w") as f:
            f.write(H.SHIM + SHIM + H.generated_part(src) + src[a:b] + MAIN)
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-w", "-o", exe, cpp])
        paths = [os.path.join(d, x) for x in ("hs", "tab")]
        hs.tofile(paths[0])
        subprocess.check_call([exe, *paths])
        got = np.fromfile(paths[1], np.uint8).reshape(nid ** 4, len(hs), 4)
    want = O.block_table(blob, nid, hs)
    bad = np.argwhere((got != want).any(axis=2))
    assert len(bad) == 0, (f"{len(bad)} blocks differ; first: tuple {bad[0][0]} hash {hs[bad[0][1]].tolist()} got "
                           f"{got[bad[0][0], bad[0][1]].tolist()} want {want[bad[0][0], bad[0][1]].tolist()}")
