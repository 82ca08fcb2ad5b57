
// ---------------------------------------------------------------------------
// Sliced kernels: a cell is SE_SL_K bits spread over as many words, a word holds
// one bit of 32 cells.  Appended after se_kernels.hip and the sliced form of the
// rule set (SE_SL_*, se_sliced_block; se_hipgen.cpp).
//
// A row is held as E words (even columns) and O words (odd columns), so bit i of
// E and of O is the block of columns 2i and 2i + 1, and with the row below them a
// word quadruple is 32 blocks, which se_sliced_block advances at once.
//
// Packed grid in memory: 8 bytes [byte column][row], byte k < 4 plane k of E and
// byte 4 + k plane k of O.  A byte column is 16 cells wide, so tiles start at any
// multiple of 16 columns.  Column c and row m of it are the world's x = c - xpad and
// y = m - ypad; everything around the world is WALL.
//
// Hash planes: bits of blocks, 32 blocks of a block row to a word.  The hash input of
// the block with origin (x, y) in frame f depends on n = 461 x + 2131 y + 2131^2 f
// alone.  The planes come in one of two forms:
//   direct: a set of planes per frame, u32 [b / 32][a][plane], bit b % 32, with a the
//     block row and b the block column.
//   shared: two sets, one per parity of n.  Within a set the n used are n0 + 2 m, and
//     m = 2131 a + 461 b with 0 <= a < 461 names each n once; the same layout with
//     these a and b.  A block row is a run along b, the row below it is a + 1 at the
//     same b (from a = 461 on: a - 461, b + 2131), and another frame is another
//     start: four frames on, a + 113 and b + 9 * 2131.  Blocks of different rows and
//     frames with the same n, most of them in a large world, are hashed once.
// At an even x offset the block at bit i of word w is that of columns 64w + 2i and
// 64w + 2i + 1, at an odd offset the block one column to the left; at an odd y offset
// block row j is one row further down (rows 2j + 1 and 2j + 2).
// ---------------------------------------------------------------------------
struct se_slgrid {  // == SlicedGrid (se_sliced.hpp)
    // addresses (as numbers: a pointer read from a record in memory would be generic,
    // and its accesses wait on the LDS counter too)
    u64 in, out;    // the grid (u32 ids)
    u64 pk0, pk1;   // packed grids
    u64 hash;       // hash planes of frames hash_frame0 ...
    int W, H, pitch;
    int xpad, ypad, bcols, rows;  // packed geometry: byte columns, rows (a multiple of 64)
    int brows;                    // block rows
    int hash_frame0, hash_shared, hash_sets;
    int hash_pitch, hash_words;   // values of a, words of a plane
    u32 hash_n0, hash_n1;         // shared: n0 of the sets of even and of odd n
};

template <typename T>
__device__ __forceinline__ T* se_sl_ptr(u64 a) {
    return (T*)(__attribute__((address_space(1))) T*)a;
}

// Codes of four ids < SE_NMAT packed in bytes, and ids of four codes.
__device__ __forceinline__ u32 se_sl_map(u32 q, u32 t0, u32 t1, u32 t2, u32 t3) {
#if SE_SL_K <= 3
    (void)t2; (void)t3;
    return __builtin_amdgcn_perm(t1, t0, q);
#else
    const u32 low = q & 0x07070707u, lo = __builtin_amdgcn_perm(t1, t0, low), hi = __builtin_amdgcn_perm(t3, t2, low);
    const u32 m = ((q >> 3) & 0x01010101u) * 0xffu;
    return (hi & m) | (lo & ~m);
#endif
}
__device__ __forceinline__ u32 se_sl_codes(u32 q) {
    return se_sl_map(q, SE_SL_CODE0, SE_SL_CODE1, SE_SL_CODE2, SE_SL_CODE3);
}
__device__ __forceinline__ u32 se_sl_ids(u32 q) {
    return se_sl_map(q, SE_SL_ID0, SE_SL_ID1, SE_SL_ID2, SE_SL_ID3);
}

// Swaps the bits of x above `m` (a mask of the low bits of each 2s-bit group)
// with the low bits of y: one step of a bit-matrix transpose.
__device__ __forceinline__ void se_sl_swapbits(u32& x, u32& y, int s, u32 m) {
    const u32 t = ((x >> s) ^ y) & m;
    y ^= t;
    x ^= t << s;
}

// 4x4 byte transpose: byte j of output i is byte i of input j.
__device__ __forceinline__ void se_sl_bytes4(u32& q0, u32& q1, u32& q2, u32& q3) {
    const u32 a = __builtin_amdgcn_perm(q1, q0, 0x05010400u), b = __builtin_amdgcn_perm(q3, q2, 0x05010400u);
    const u32 c = __builtin_amdgcn_perm(q1, q0, 0x07030602u), d = __builtin_amdgcn_perm(q3, q2, 0x07030602u);
    q0 = __builtin_amdgcn_perm(b, a, 0x05040100u);
    q1 = __builtin_amdgcn_perm(b, a, 0x07060302u);
    q2 = __builtin_amdgcn_perm(d, c, 0x05040100u);
    q3 = __builtin_amdgcn_perm(d, c, 0x07060302u);
}

// Words of 32 cells of a row: cells d[i] byte j (code < 16) = cell 8j + i  ->  p[k] = plane k.
__device__ __forceinline__ void se_sl_slice(const u32* d, u32* p) {
    u32 u[4];
#pragma unroll
    for (int i = 0; i < 4; i++) u[i] = d[i] | (d[i + 4] << 4);
    se_sl_swapbits(u[0], u[2], 2, 0x33333333u);
    se_sl_swapbits(u[1], u[3], 2, 0x33333333u);
    se_sl_swapbits(u[0], u[1], 1, 0x55555555u);
    se_sl_swapbits(u[2], u[3], 1, 0x55555555u);
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) p[k] = u[k];
}
__device__ __forceinline__ void se_sl_unslice(const u32* p, u32* d) {
    u32 u[4];
#pragma unroll
    for (int k = 0; k < 4; k++) u[k] = k < SE_SL_K ? p[k] : 0u;
    se_sl_swapbits(u[0], u[1], 1, 0x55555555u);
    se_sl_swapbits(u[2], u[3], 1, 0x55555555u);
    se_sl_swapbits(u[0], u[2], 2, 0x33333333u);
    se_sl_swapbits(u[1], u[3], 2, 0x33333333u);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        d[i] = u[i] & 0x0f0f0f0fu;
        d[i + 4] = (u[i] >> 4) & 0x0f0f0f0fu;
    }
}

// ---------------------------------------------------------------------------
// u32 grid -> packed grid.  One wavefront per 64 columns x 64 rows: 16-byte loads
// (4 rows of 64 cells each), four codes to a word, through LDS to one row a lane
// (a stride of 17 words keeps both sides free of bank conflicts), and there the
// bits are transposed into planes.  Bound by HBM: 4 B of ids read per cell, and
// half a byte written.  The second packed grid gets the rows and columns around
// the world too, which the step kernel reads and never writes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint2* se_sl_at(const se_slgrid& g, int which, int bcol, int row) {
    return se_sl_ptr<uint2>(which ? g.pk1 : g.pk0) + ((size_t)bcol * g.rows + row);
}

// The byte column of the world's column 64 * wc: packing and unpacking go by 64
// columns of the world, so that their accesses to the ids are whole cache lines
// (unpacking 16384^2 by 64 columns of the packed grid, 64 bytes off: 253 us for 198).
__device__ __forceinline__ int se_sl_bcol(const se_slgrid& g, int wc) { return 4 * wc + (g.xpad >> 4); }

// Planes of a row's 64 cells <-> its four byte columns.
__device__ __forceinline__ void se_sl_columns(const u32* e, const u32* o, uint2* c) {
    u32 a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        a[k] = k < SE_SL_K ? e[k] : 0u;
        b[k] = k < SE_SL_K ? o[k] : 0u;
    }
    se_sl_bytes4(a[0], a[1], a[2], a[3]);
    se_sl_bytes4(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int q = 0; q < 4; q++) c[q] = make_uint2(a[q], b[q]);
}
__device__ __forceinline__ void se_sl_planes(const uint2* c, u32* e, u32* o) {
    u32 a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        a[q] = c[q].x;
        b[q] = c[q].y;
    }
    se_sl_bytes4(a[0], a[1], a[2], a[3]);
    se_sl_bytes4(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) {
        e[k] = a[k];
        o[k] = b[k];
    }
}

// The code that all 64 x 64 cells of a wavefront's square hold, else 0xff.
__device__ __forceinline__ u32 se_sl_uniform(const u32* e, const u32* o) {
    u32 code = 0u, differ = 0u;
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) {
        const u32 bit = (u32)__builtin_amdgcn_readfirstlane((int)e[k]) & 1u;
        code |= bit << k;
        differ |= (e[k] ^ (0u - bit)) | (o[k] ^ (0u - bit));
    }
    return __builtin_amdgcn_ballot_w64(differ != 0u) ? 0xffu : code;
}

// What a run of one world knows of its 64 x 64 squares (null: nothing is kept).
// same: the code that both grids held all over the square when the last run ended,
// else 0xff; all 0xff when `valid` is 0, which is so once anything else has written a
// grid.  was: the code that the run's first grid held; calm: the same, for tiles that sleep.
// Packing does not read a square whose code it knows, and unpacking does not write one that holds it already: a run of
// 12 steps of a settled 16384^2 world took 540 us, of which 412 were these two passes.
struct se_slknown {
    unsigned char *same, *was, *calm;
    int valid;
};

__device__ __forceinline__ void se_sl_pack_tile(const se_slgrid& g, int wc, int m0, u32* lds, const se_slknown& known,
                                                int sq) {
    const int lane = (int)(threadIdx.x & 63);
    const int x = 16 * se_sl_bcol(g, wc) - g.xpad + 4 * (lane & 15);
    const int y0 = m0 - g.ypad, xw = 16 * se_sl_bcol(g, wc) - g.xpad;
    const bool inside = y0 >= 0 && y0 + 64 <= g.H && xw >= 0 && xw + 64 <= g.W;  // all of the tile inside the world
    const u32 code = known.valid && inside ? known.same[sq] : 0xffu;
    u32 e[SE_SL_K], o[SE_SL_K];
    if (code != 0xffu) {
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) e[k] = o[k] = 0u - ((code >> k) & 1u);
        if (lane == 0) known.was[sq] = known.calm[sq] = (unsigned char)code;
    } else {
        uint4 v[16];
        if (inside) {
            const u32* s = se_sl_ptr<const u32>(g.in) + (size_t)(y0 + (lane >> 4)) * g.pitch + x;
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = se_load_nt(s + (size_t)(4 * i) * g.pitch);
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int y = y0 + 4 * i + (lane >> 4);
                const bool in = y >= 0 && y < g.H && x >= 0 && x < g.W;
                uint4 t = *reinterpret_cast<const uint4*>(se_sl_ptr<const u32>(g.in) + (in ? (size_t)y * g.pitch + x : 0));
                t.x = in ? t.x : SE_WALLID;
                t.y = in && x + 1 < g.W ? t.y : SE_WALLID;
                t.z = in && x + 2 < g.W ? t.z : SE_WALLID;
                t.w = in && x + 3 < g.W ? t.w : SE_WALLID;
                v[i] = t;
            }
        }
        bool exact = true;  // no id beyond the materials: the codes say what the grid holds
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const u32 mx = max(max(v[i].x, v[i].y), max(v[i].z, v[i].w));
            u32 q;
            if (__builtin_expect(mx >= SE_NMAT, 0)) {
                q = se_pack4(se_decode(v[i].x), se_decode(v[i].y), se_decode(v[i].z), se_decode(v[i].w));
                exact = false;
            } else {
                q = se_pack4(v[i].x, v[i].y, v[i].z, v[i].w);
            }
            lds[(4 * i + (lane >> 4)) * 17 + (lane & 15)] = se_sl_codes(q);
        }
        __builtin_amdgcn_wave_barrier();
        u32 q[16], de[8], dd[8];
#pragma unroll
        for (int m = 0; m < 16; m++) q[m] = lds[lane * 17 + m];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            se_sl_bytes4(q[t], q[4 + t], q[8 + t], q[12 + t]);
            de[2 * t] = q[t];
            dd[2 * t] = q[4 + t];
            de[2 * t + 1] = q[8 + t];
            dd[2 * t + 1] = q[12 + t];
        }
        se_sl_slice(de, e);
        se_sl_slice(dd, o);
        if (known.was != nullptr) {
            const u32 all = se_sl_uniform(e, o);
            const bool keep = inside && __builtin_amdgcn_ballot_w64(!exact) == 0;
            if (lane == 0) known.was[sq] = known.calm[sq] = (unsigned char)(keep ? all : 0xffu);
        }
    }
    const int row = m0 + lane;
    const bool around_y = row < g.ypad || row >= g.ypad + g.H;
    uint2 cols[4];
    se_sl_columns(e, o, cols);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int bc = se_sl_bcol(g, wc) + q;
        if (bc < 0 || bc >= g.bcols) continue;
        *se_sl_at(g, 0, bc, row) = cols[q];
        const int c = 16 * bc - g.xpad;
        if (around_y || c < 0 || c + 16 > g.W) *se_sl_at(g, 1, bc, row) = cols[q];
    }
}

// packed grid `from` -> u32 grid (the cells of the world only)
__device__ __forceinline__ void se_sl_unpack_tile(const se_slgrid& g, int from, int wc, int m0, u32* lds,
                                                  const se_slknown& known, int sq) {
    const int lane = (int)(threadIdx.x & 63);
    u32 e[SE_SL_K], o[SE_SL_K], de[8], dd[8], q[16];
    uint2 cols[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        cols[c] = se_sl_bcol(g, wc) + c < g.bcols ? *se_sl_at(g, from, se_sl_bcol(g, wc) + c, m0 + lane)
                                                   : make_uint2(0u, 0u);
    se_sl_planes(cols, e, o);
    if (known.same != nullptr) {
        const u32 was = known.was[sq], all = was != 0xffu ? se_sl_uniform(e, o) : 0xffu;  // 0xff: not all inside the world
        const bool stays = all != 0xffu && was == all;  // the first grid holds it
        const bool held = stays && known.valid && known.same[sq] == all;
        if (lane == 0) known.same[sq] = (unsigned char)(stays ? all : 0xffu);
        if (held) return;
    }
    se_sl_unslice(e, de);
    se_sl_unslice(o, dd);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        q[t] = de[2 * t];
        q[4 + t] = dd[2 * t];
        q[8 + t] = de[2 * t + 1];
        q[12 + t] = dd[2 * t + 1];
        se_sl_bytes4(q[t], q[4 + t], q[8 + t], q[12 + t]);
    }
#pragma unroll
    for (int m = 0; m < 16; m++) lds[lane * 17 + m] = se_sl_ids(q[m]);
    __builtin_amdgcn_wave_barrier();
    const int x = 16 * se_sl_bcol(g, wc) - g.xpad + 4 * (lane & 15);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int y = m0 + 4 * i + (lane >> 4) - g.ypad;
        const u32 p = lds[(4 * i + (lane >> 4)) * 17 + (lane & 15)];
        if (y < 0 || y >= g.H || x < 0 || x >= g.W) continue;
        u32* dst = se_sl_ptr<u32>(g.out) + (size_t)y * g.pitch + x;
        const uint4 v = make_uint4(p & 0xffu, (p >> 8) & 0xffu, (p >> 16) & 0xffu, p >> 24);
        if (x + 3 < g.W) {
            se_store_quad<true>(dst, v);
        } else {
            dst[0] = v.x;
            if (x + 1 < g.W) dst[1] = v.y;
            if (x + 2 < g.W) dst[2] = v.z;
        }
    }
}

// wtiles columns of 64 cells, from the one left of the world on (se_sl_pack: the
// margin is packed too), tiles in all; unpacking leaves that column out
extern "C" __global__ __launch_bounds__(256) void se_sl_pack(se_slgrid g, int wtiles, int tiles, se_slknown known) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), t = (int)blockIdx.x * 4 + wave;
    if (t >= tiles) return;
    se_sl_pack_tile(g, t % wtiles - 1, (t / wtiles) * 64, lds[wave], known, t);
}

extern "C" __global__ __launch_bounds__(256) void se_sl_unpack(se_slgrid g, int from, int wtiles, int tiles, int packed_wtiles,
                                                               se_slknown known) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), t = (int)blockIdx.x * 4 + wave;
    if (t >= tiles) return;
    se_sl_unpack_tile(g, from, t % wtiles, (t / wtiles) * 64, lds[wave], known,
                      (t / wtiles) * packed_wtiles + t % wtiles + 1);
}

// ---------------------------------------------------------------------------
// Hash planes.  A thread makes one word of every plane: lanes are consecutive block
// rows (values of a), so the stores are contiguous, and a thread steps its hash
// inputs along the block row by a constant.  Bound by VALU issue: per block and hash
// lane two 32-bit multiplies, three shifted exclusive ors and the step, and two
// instructions per plane (compare, shift the bit in).  16384^2 and one plane: 1.6 us a
// frame in the shared form, 21 in the direct one; 4096^2 1.0 us (direct).
// ---------------------------------------------------------------------------
#define SE_SL_B0 2144  // keeps b >= 0; a multiple of 32
__device__ __forceinline__ constexpr u32 se_sl_mult(int l) {
    return l == 0 ? 213u : l == 1 ? 2131u : l == 2 ? 21313u : 213132u;
}

// acc = acc << 1 | (h <= t): the compare's carry shifted in
__device__ __forceinline__ void se_sl_push(u32& acc, u32 h, u32 t) {
    __asm__("v_cmp_ge_u32 vcc, %2, %1\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(acc) : "v"(h), "s"(t) : "vcc");
}

// word i of a set
__device__ __forceinline__ void se_sl_hash_word(const se_slgrid& g, int i, int set) {
    const int u = i / g.hash_pitch, a = i - u * g.hash_pitch;
    u32 n;  // of the block at bit 31
    if (g.hash_shared) {
        n = (set ? g.hash_n1 : g.hash_n0) + 2u * (2131u * (u32)a + 461u * (u32)(32 * u + 31 - SE_SL_B0));
    } else {
        const u32 f = (u32)(g.hash_frame0 + set);
        int ox, oy;
        se_offset(f, ox, oy);
        n = 461u * (u32)(64 * u + 62 - ox - g.xpad) + 2131u * (u32)(2 * a + oy - g.ypad) + 4541161u * f;
    }
    u32 in[4], acc[SE_SL_P];
#pragma unroll
    for (int l = 0; l < 4; l++) in[l] = n * se_sl_mult(l);
#pragma unroll
    for (int p = 0; p < SE_SL_P; p++) acc[p] = 0u;
#pragma unroll 4
    for (int k = 0; k < 32; k++) {
        u32 h[4];
#pragma unroll
        for (int l = 0; l < 4; l++) {
            h[l] = 0u;
            if (!se_sliced_lane(l)) continue;
            h[l] = se_lowbias(in[l]);
            in[l] -= 922u * se_sl_mult(l);
        }
#pragma unroll
        for (int p = 0; p < SE_SL_P; p++) se_sl_push(acc[p], h[se_sliced_class_lane(p)], se_sliced_class_max(p));
    }
    u32* out = se_sl_ptr<u32>(g.hash) + ((size_t)set * g.hash_words + i) * SE_SL_P;
#pragma unroll
    for (int p = 0; p < SE_SL_P; p++) out[p] = acc[p];
}

// grid: x over the words of a plane, y over the sets
extern "C" __global__ __launch_bounds__(256) void se_sl_hash(se_slgrid g) {
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i < g.hash_words) se_sl_hash_word(g, i, (int)blockIdx.y);
}

// ---------------------------------------------------------------------------
// Step kernel: S wavefronts advance a tile of S * NW words (64 columns each) by
// 64 * R rows through `nsub` sub-steps entirely in registers.  Lane l holds rows
// R*l .. R*l + R - 1 of every word column.
//   * y offset 1: every lane gives its first row to the lane above it (a wave
//     shift) and the rows move up by one, until the offset returns to 0; the
//     tile's outermost rows take WALL.
//   * x offset 1: the O words move up by one block (alignbit over the word
//     columns) and the blocks are (O, E) instead of (E, O).
// Blocks are never split between lanes otherwise, so one wavefront needs no barriers
// and no LDS; two that share a tile exchange a word column at odd x offsets.  What
// the shifts bring in at the tile's sides is wrong inside the world and right at its
// border (WALL, code 0), so the valid region shrinks by one cell per sub-step on the
// sides that cut into the world: 16 or 32 columns and `halo` rows
// are given up on each side of a tile, none of a world that fits one tile.
// ---------------------------------------------------------------------------
template <int NW, int R>
struct se_sltile {
    u32 e[R][NW][SE_SL_K], o[R][NW][SE_SL_K];
};

// lane i gets lane i + 1 (wave_shl), the last lane 0 (WALL); and the other way round
__device__ __forceinline__ u32 se_sl_from_below(u32 v) {
    return (u32)__builtin_amdgcn_mov_dpp((int)v, 0x130, 0xf, 0xf, true);
}
__device__ __forceinline__ u32 se_sl_from_above(u32 v) {
    return (u32)__builtin_amdgcn_mov_dpp((int)v, 0x138, 0xf, 0xf, true);
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_rows_up(se_sltile<NW, R>& t) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) {
            const u32 e = se_sl_from_below(t.e[0][w][k]), o = se_sl_from_below(t.o[0][w][k]);
#pragma unroll
            for (int r = 0; r + 1 < R; r++) {
                t.e[r][w][k] = t.e[r + 1][w][k];
                t.o[r][w][k] = t.o[r + 1][w][k];
            }
            t.e[R - 1][w][k] = e;
            t.o[R - 1][w][k] = o;
        }
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_rows_down(se_sltile<NW, R>& t) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) {
            const u32 e = se_sl_from_above(t.e[R - 1][w][k]), o = se_sl_from_above(t.o[R - 1][w][k]);
#pragma unroll
            for (int r = R - 1; r > 0; r--) {
                t.e[r][w][k] = t.e[r - 1][w][k];
                t.o[r][w][k] = t.o[r - 1][w][k];
            }
            t.e[0][w][k] = e;
            t.o[0][w][k] = o;
        }
}

// Where the lane's block rows find their hash words: a and b of the tile's first
// block, for one phase of the cycle; stepping four frames on stays in the phase.
template <int NW, int R>
struct se_slwords {  // raw words: a row's bits start at any bit of the first
    u32 v[R / 2][NW + 1][SE_SL_P], shift[R / 2];
};

template <int R>
struct se_slplace {
    u32 a[R / 2], b[R / 2];
    u32 set;  // word offset of the set (direct: of the frame's planes)
};

template <int R>
__device__ __forceinline__ se_slplace<R> se_sl_place(const se_slgrid& g, u32 f, int blk0, int j0) {
    int ox, oy;
    se_offset(f, ox, oy);
    const u32 parity = (u32)(ox + oy + (int)f) & 1u;
    const u32 m = (461u * (u32)(-ox - g.xpad) + 2131u * (u32)(oy - g.ypad) + 4541161u * f -
                   (parity ? g.hash_n1 : g.hash_n0)) >> 1;
    const u32 a0 = m % 461u * 204u % 461u;  // 204 * 2131 = 1 mod 461
    const u32 b0 = (m + 461u * SE_SL_B0 - 2131u * a0) / 461u;
    const bool sh = g.hash_shared != 0;
    se_slplace<R> q;
    q.set = (sh ? parity : f - (u32)g.hash_frame0) * (u32)g.hash_words;
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
        const u32 a = (sh ? a0 : 0u) + (u32)(j0 + i), wrap = sh ? a / 461u : 0u;
        q.a[i] = a - 461u * wrap;
        q.b[i] = (sh ? b0 : 0u) + (u32)blk0 + 2131u * wrap;
    }
    return q;
}

// Loads at the place; the words are shifted into line only where they are used
// (se_sl_hash_of), so nothing waits here.
template <int NW, int R>
__device__ __forceinline__ void se_sl_hash_load(const se_slgrid& g, const se_slplace<R>& q, se_slwords<NW, R>& h) {
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
        const u32 at = (q.set + (q.b[i] >> 5) * (u32)g.hash_pitch + q.a[i]) * (u32)SE_SL_P;
        h.shift[i] = q.b[i];  // alignbit takes it modulo 32
#pragma unroll
        for (int w = 0; w <= NW; w++) {
            const u32* s = se_sl_ptr<const u32>(g.hash) + (size_t)w * (size_t)(g.hash_pitch * SE_SL_P);
#pragma unroll
            for (int p = 0; p < SE_SL_P; p++) h.v[i][w][p] = s[at + (u32)p];
        }
    }
}

template <int R>
__device__ __forceinline__ void se_sl_next_cycle(const se_slgrid& g, se_slplace<R>& q) {
    const u32 da = g.hash_shared ? 113u : 0u, db = g.hash_shared ? 9u * 2131u : 0u;
    const u32 mod = g.hash_shared ? 461u : 0x7fffffffu;
    q.set += g.hash_shared ? 0u : 4u * (u32)g.hash_words;
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
        const u32 a = q.a[i] + da;
        const bool c = a >= mod;
        q.a[i] = c ? a - mod : a;
        q.b[i] += c ? db + 2131u : db;
    }
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_hash_of(const se_slwords<NW, R>& r, u32 (&h)[R / 2][NW][SE_SL_P]) {
#pragma unroll
    for (int i = 0; i < R / 2; i++)
#pragma unroll
        for (int w = 0; w < NW; w++)
#pragma unroll
            for (int p = 0; p < SE_SL_P; p++)
                h[i][w][p] = __builtin_amdgcn_alignbit(r.v[i][w + 1][p], r.v[i][w][p], r.shift[i]);
}

#if !SE_SL_KEEP
// Puts back the WALL outside the world (rules may change it); ysh: rows moved up.
template <int NW, int R>
__device__ __forceinline__ void se_sl_keep_wall(se_sltile<NW, R>& t, const se_slgrid& g, int c0, int y0) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const u32 rm = y0 + r >= 0 && y0 + r < g.H ? 0xffffffffu : 0u;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int x0 = c0 + 64 * w - g.xpad;  // column of bit 0 of E
            const int lo = x0 < 0 ? (-x0 + 1) / 2 : 0, lo1 = x0 < 0 ? -x0 / 2 : 0;
            const int hi = min(32, max(0, (g.W - x0 + 1) / 2)), hi1 = min(32, max(0, (g.W - x0) / 2));
            const u32 me = (u32)((1ull << hi) - 1ull) & ~(u32)((1ull << min(lo, 32)) - 1ull) & rm;
            const u32 mo = (u32)((1ull << hi1) - 1ull) & ~(u32)((1ull << min(lo1, 32)) - 1ull) & rm;
#pragma unroll
            for (int k = 0; k < SE_SL_K; k++) {
                t.e[r][w][k] &= me;
                t.o[r][w][k] &= mo;
            }
        }
    }
}
#endif

// The wavefronts of a tile (S of them side by side, NW word columns each) pass the
// O words at their common side through LDS: lds[side][row][plane][lane], for the
// shift up and for the shift down in turn, one barrier each.  A set is written
// again only after the barrier that follows its reads.
template <int R, int S>
struct se_slshare {
    u32 up[S - 1][R][SE_SL_K][64], down[S - 1][R][SE_SL_K][64];
};
template <int R>
struct se_slshare<R, 1> {};

template <int NW, int R, int S>
__device__ __forceinline__ void se_sl_shift_up(se_sltile<NW, R>& t, se_slshare<R, S>& sh, int wv, int lane) {
    u32 in[R][SE_SL_K];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) in[r][k] = 0u;
    if constexpr (S > 1) {
        if (wv < S - 1)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++) sh.up[wv][r][k][lane] = t.o[r][NW - 1][k];
        __syncthreads();
        if (wv > 0)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++) in[r][k] = sh.up[wv - 1][r][k][lane];
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++)
#pragma unroll
            for (int w = NW - 1; w >= 0; w--)
                t.o[r][w][k] = __builtin_amdgcn_alignbit(t.o[r][w][k], w ? t.o[r][w - 1][k] : in[r][k], 31);
}

template <int NW, int R, int S>
__device__ __forceinline__ void se_sl_shift_down(se_sltile<NW, R>& t, se_slshare<R, S>& sh, int wv, int lane) {
    u32 in[R][SE_SL_K];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) in[r][k] = 0u;
    if constexpr (S > 1) {
        if (wv > 0)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++) sh.down[wv - 1][r][k][lane] = t.o[r][0][k];
        __syncthreads();
        if (wv < S - 1)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++) in[r][k] = sh.down[wv][r][k][lane];
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++)
#pragma unroll
            for (int w = 0; w < NW; w++)
                t.o[r][w][k] = __builtin_amdgcn_alignbit(w + 1 < NW ? t.o[r][w + 1][k] : in[r][k], t.o[r][w][k], 1);
}

// One sub-step at x offset OX with the rows already paired (y offset applied).
template <int NW, int R, int S, bool OX>
__device__ __forceinline__ void se_sl_substep(se_sltile<NW, R>& t, const se_slwords<NW, R>& raw, se_slshare<R, S>& sh,
                                              int wv, int lane) {
    u32 h[R / 2][NW][SE_SL_P];
    se_sl_hash_of<NW, R>(raw, h);
    if (OX) se_sl_shift_up<NW, R, S>(t, sh, wv, lane);
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int b = 0; b < R / 2; b++) {
            if (OX) se_sliced_block(t.o[2 * b][w], t.e[2 * b][w], t.o[2 * b + 1][w], t.e[2 * b + 1][w], h[b][w]);
            else se_sliced_block(t.e[2 * b][w], t.o[2 * b][w], t.e[2 * b + 1][w], t.o[2 * b + 1][w], h[b][w]);
        }
    if (OX) se_sl_shift_down<NW, R, S>(t, sh, wv, lane);
}

// Whole cycles of four frames run in a loop of their own: every offset is a
// constant there, the rows move up once and down once and the moves are register
// names.  Up to three frames before and after them take the general step.  The
// hash words are loaded AHEAD frames before their use: a 2x2 tile's sub-step takes
// 0.3 us, and the words come from beyond the L2.
template <int NW, int R, int S, int AHEAD>
__device__ __forceinline__ void se_sl_advance(se_sltile<NW, R>& t, const se_slgrid& g, int blk0, int row0, int lane,
                                              int frame0, int nsub, se_slshare<R, S>& sh, int wv) {
    static_assert(AHEAD == 2 || AHEAD == 4, "sets of words by phase");
    const int j0 = row0 / 2 + (R / 2) * lane;
    u32 f = (u32)frame0;
    const u32 end = f + (u32)nsub, first = (f + 3u) & ~3u;
#if !SE_SL_KEEP
    const int c0 = 2 * blk0;
    const bool edge = c0 < g.xpad || c0 + 64 * NW > g.xpad + g.W || row0 < g.ypad ||
                      row0 + 64 * R > g.ypad + g.H;
    const int y0 = row0 + R * lane - g.ypad;
#define SE_SL_FIX(up) if (edge) se_sl_keep_wall<NW, R>(t, g, c0, y0 + (up))
#else
#define SE_SL_FIX(up)
#endif
    auto general = [&](u32 fr, const se_slwords<NW, R>& h) {
        int ox, oy;
        se_offset(fr, ox, oy);
        if (oy) se_sl_rows_up(t);
        if (ox) se_sl_substep<NW, R, S, true>(t, h, sh, wv, lane);
        else se_sl_substep<NW, R, S, false>(t, h, sh, wv, lane);
        SE_SL_FIX(oy);
        if (oy) se_sl_rows_down(t);
    };
    for (; f < end && f < first; f++) {
        se_slwords<NW, R> h;
        se_sl_hash_load<NW, R>(g, se_sl_place<R>(g, f, blk0, j0), h);
        general(f, h);
    }
    if (f + 4u <= end) {
        se_slplace<R> q[4];
        se_slwords<NW, R> h[AHEAD];
#pragma unroll
        for (u32 p = 0; p < 4; p++) q[p] = se_sl_place<R>(g, f + p, blk0, j0);
#pragma unroll
        for (int p = 0; p < AHEAD; p++) se_sl_hash_load<NW, R>(g, q[p], h[p]);
#pragma unroll
        for (int p = 0; p < AHEAD; p++) se_sl_next_cycle<R>(g, q[p]);
        // (the last cycle's loads run on into the frames after the last: the planes
        // have room for them)
        do {
            se_sl_substep<NW, R, S, false>(t, h[0], sh, wv, lane);          // offsets (0, 0)
            SE_SL_FIX(0);
            se_sl_hash_load<NW, R>(g, q[AHEAD & 3], h[0]);
            se_sl_next_cycle<R>(g, q[AHEAD & 3]);
            se_sl_rows_up(t);
            se_sl_substep<NW, R, S, true>(t, h[1], sh, wv, lane);           // (1, 1)
            SE_SL_FIX(1);
            se_sl_hash_load<NW, R>(g, q[(AHEAD + 1) & 3], h[1]);
            se_sl_next_cycle<R>(g, q[(AHEAD + 1) & 3]);
            se_sl_substep<NW, R, S, false>(t, h[2 % AHEAD], sh, wv, lane);  // (0, 1)
            SE_SL_FIX(1);
            se_sl_hash_load<NW, R>(g, q[(AHEAD + 2) & 3], h[2 % AHEAD]);
            se_sl_next_cycle<R>(g, q[(AHEAD + 2) & 3]);
            se_sl_rows_down(t);
            se_sl_substep<NW, R, S, true>(t, h[3 % AHEAD], sh, wv, lane);   // (1, 0)
            SE_SL_FIX(0);
            se_sl_hash_load<NW, R>(g, q[(AHEAD + 3) & 3], h[3 % AHEAD]);
            se_sl_next_cycle<R>(g, q[(AHEAD + 3) & 3]);
            f += 4u;
        } while (f + 4u <= end);
    }
    for (; f < end; f++) {
        se_slwords<NW, R> h;
        se_sl_hash_load<NW, R>(g, se_sl_place<R>(g, f, blk0, j0), h);
        general(f, h);
    }
#undef SE_SL_FIX
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_load(se_sltile<NW, R>& t, const se_slgrid& g, int from, int bc0, int row) {
    uint2 c[NW][4][R];
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4* s = reinterpret_cast<const uint4*>(se_sl_at(g, from, bc0 + 4 * w + q, row));
#pragma unroll
            for (int r = 0; r < R; r += 2) {  // row is even: two rows are 16 aligned bytes
                const uint4 v = s[r / 2];
                c[w][q][r] = make_uint2(v.x, v.y);
                c[w][q][r + 1] = make_uint2(v.z, v.w);
            }
        }
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint2 col[4] = {c[w][0][r], c[w][1][r], c[w][2][r], c[w][3][r]};
            se_sl_planes(col, t.e[r][w], t.o[r][w]);
        }
}

// byte columns first .. last of the NW word columns
template <int NW, int R>
__device__ __forceinline__ void se_sl_store(const se_sltile<NW, R>& t, const se_slgrid& g, int to, int bc0, int row,
                                            int first, int last) {
#pragma unroll
    for (int w = 0; w < NW; w++) {
        uint2 col[R][4];
#pragma unroll
        for (int r = 0; r < R; r++) se_sl_columns(t.e[r][w], t.o[r][w], col[r]);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (4 * w + q < first || 4 * w + q > last) continue;
            uint4* d = reinterpret_cast<uint4*>(se_sl_at(g, to, bc0 + 4 * w + q, row));
#pragma unroll
            for (int r = 0; r < R; r += 2)
                d[r / 2] = make_uint4(col[r][q].x, col[r][q].y, col[r + 1][q].x, col[r + 1][q].y);
        }
    }
}

// `from`: the packed grid read, the other is written.  side: byte columns given up
// on each side (1 or 2, for up to 16 or 32 sub-steps), halo: rows; both 0: the
// world fits the one tile, all of which is stored.
template <int NW, int R, int S, int AHEAD>
__device__ __forceinline__ void se_sl_tile(const se_slgrid& g, int from, int tx, int ty, int frame0, int nsub,
                                           int side, int halo, se_slshare<R, S>& sh) {
    const int lane = (int)(threadIdx.x & 63), wv = S > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    const int bc0 = tx * (4 * NW * S - 2 * side) + 4 * NW * wv, row0 = ty * (64 * R - 2 * halo);
    const int row = row0 + R * lane;
    se_sltile<NW, R> t;
    se_sl_load<NW, R>(t, g, from, bc0, row);
    se_sl_advance<NW, R, S, AHEAD>(t, g, 8 * bc0, row0, lane, frame0, nsub, sh, wv);
    if (R * lane < halo || R * lane >= 64 * R - halo) return;
    se_sl_store<NW, R>(t, g, from ^ 1, bc0, row, side - 4 * NW * wv, 4 * NW * S - 1 - side - 4 * NW * wv);
}

// A world and how it is cut into tiles.  In a batch (device memory, filled by the
// host) the hash fields are those of its group: worlds that start at the same frame
// read the same planes.
struct se_slworld {  // == SlicedWorld (se_sliced.hpp)
    se_slgrid g;
    int frame0, steps, tiles_x, side, halo, group;
    int result;  // packed grid that holds the world after its last launch
    u32 stable;  // codes of tiles that may sleep (se_sl_sleeps); 0 in a batch
    u64 calm;    // squares' codes
    int calm_cols, pad;
};

// Does the tile sleep through the launch?  Then its kept cells are written as they are.
// A change travels a cell a step: a tile where all squares within `done` cells of it (it has
// the launch's halo in it) held one code when the run began (calm, by packing; a
// modification ends it), and no rule changes a block of four such cells, is as it was.
// Others are mostly found out by the square at their middle, one scalar load.  Kept apart
// from the tile's own loads and registers: a test of the cells once they are here, or one
// path to the stores for both, cost a launch of a dense 16384^2 world 3 to 8 %.
template <int NW, int R, int S>
__device__ __forceinline__ bool se_sl_sleeps(const se_slworld& v, int from, int tx, int ty, int done) {
    constexpr int W = 64 * NW * S, H = 64 * R;
    const int bc0 = tx * (4 * NW * S - 2 * v.side), row0 = ty * (H - 2 * v.halo), x = 16 * bc0 - v.g.xpad;
    const int mid = ((row0 + H / 2) >> 6) * v.calm_cols + ((x + W / 2) >> 6) + 1;  // inside the packed grid
    const u32 code = ((const __attribute__((address_space(4))) u32*)v.calm)[mid >> 2] >> (8 * (mid & 3)) & 0xffu;
    if (code == 0xffu || !((v.stable >> code) & 1u)) return false;
    const int ca = (x - done) >> 6, cb = (x + W - 1 + done) >> 6, ra = (row0 - done) >> 6, rb = (row0 + H - 1 + done) >> 6;
    if (ca < 0 || cb + 1 >= v.calm_cols || ra < 0 || 64 * rb >= v.g.rows) return false;
    const unsigned char* calm = se_sl_ptr<const unsigned char>(v.calm);
    const int wide = cb - ca + 1, n = wide * (rb - ra + 1);
    bool other = false;
    for (int i = (int)(threadIdx.x & 63); i < n; i += 64) other |= calm[(ra + i / wide) * v.calm_cols + ca + i % wide + 1] != code;
    if (__builtin_amdgcn_ballot_w64(other)) return false;
    u32 planes = 0u;
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) planes |= (code >> k) & 1u ? 0xffu << (8 * k) : 0u;
    const int pairs = H / 2 - v.halo, columns = 4 * NW * S - 2 * v.side;  // pairs of rows
    for (int i = (int)threadIdx.x; i < columns * pairs; i += 64 * S)
        *reinterpret_cast<uint4*>(se_sl_at(v.g, from ^ 1, bc0 + v.side + i / pairs, row0 + v.halo + 2 * (i % pairs))) =
            make_uint4(planes, planes, planes, planes);
    return true;
}

// Steps [done, done + k) of `one` (n = 0), or of worlds [0, n) (longest first, their
// tiles counted by prefix); one workgroup per tile.
#define SE_SL_STEP(NW, R, S, AHEAD, WAVES, SLEEP, NAME)                                                                       \
    extern "C" __global__ __launch_bounds__(64 * S, WAVES) void se_sl_step_##NAME(                                 \
        se_slworld one, const se_slworld* __restrict__ worlds, const int* __restrict__ prefix, int n,          \
        const se_slgrid* __restrict__ groups, int from, int done, int k) {                                     \
        __shared__ se_slshare<R, S> sh;                                                                        \
        if (S > 1) __builtin_amdgcn_s_setprio(3); /* a chain of steps beside the planes of a later chunk */    \
        se_slworld v = one;                                                                                    \
        int tile;                                                                                              \
        if (n == 0) {                                                                                          \
            tile = se_xcd_tile((int)blockIdx.x, (int)gridDim.x);                                               \
            if (SLEEP && one.stable != 0u &&                                                                   \
                se_sl_sleeps<NW, R, S>(one, from, tile % one.tiles_x, tile / one.tiles_x, done)) return;       \
        } else {                                                                                               \
            const int w = se_owner(prefix, n, (int)blockIdx.x);                                                \
            tile = (int)blockIdx.x - prefix[w];                                                                \
            v = worlds[w];                                                                                     \
            const se_slgrid& G = groups[v.group];                                                              \
            v.g.hash = G.hash;                                                                                 \
            v.g.hash_frame0 = G.hash_frame0;                                                                   \
            v.g.hash_shared = G.hash_shared;                                                                   \
            v.g.hash_pitch = G.hash_pitch;                                                                     \
            v.g.hash_words = G.hash_words;                                                                     \
            v.g.hash_n0 = G.hash_n0;                                                                           \
            v.g.hash_n1 = G.hash_n1;                                                                           \
        }                                                                                                      \
        se_sl_tile<NW, R, S, AHEAD>(v.g, from, tile % v.tiles_x, tile / v.tiles_x, v.frame0 + done,               \
                                 min(k, v.steps - done), v.side, v.halo, sh);                                      \
    }
// By two and by four wavefronts: half the instructions in a sub-step's chain, which
// is what a world of few tiles waits for (us a call without the fill, one wavefront for 2x2: 100x90 500
// steps 229 / 162, 1000x700 200 steps 141 / 113, twelve materials 800x800 150 steps
// 201 / 152); the wider tile gives up a smaller share of its columns.
SE_SL_STEP(1, 2, 2, 4, 1, false, 2x2s)
SE_SL_STEP(1, 2, 4, 4, 1, false, 4x2s)
// By one: no barriers, for worlds that fill the SIMDs many times over (16384^2, 100
// steps without the fill: 1.37 ms with 4x2, 1.39 with 4x2s; 4096^2, 200 steps: 445 and 455 us).  With
// four planes one wavefront's registers leave two or three a SIMD and the
// split tiles are faster (8192^2, twelve materials, 64 steps: 646 us with 4x2s, 758).
// Only the kernels of large worlds sleep: with se_sl_sleeps in them the split tiles' main
// loops came out with other registers and moves (us a call, split tiles with / without: feature
// rules 1296x67 557 steps 417 / 409, 618x119 107 steps 104 / 103).
#if SE_SL_K <= 3
SE_SL_STEP(2, 2, 1, 4, 3, true, 2x2)
SE_SL_STEP(4, 2, 1, 2, 3, true, 4x2)
#else
SE_SL_STEP(1, 2, 2, 4, 1, true, 2x2z)
SE_SL_STEP(1, 2, 4, 4, 1, true, 4x2z)
#endif

// ---------------------------------------------------------------------------
// Modifications of a run's first step, on packed grid `to` after that step (one launch of
// one sub-step).  blockIdx.y is a modification; a thread takes 16 cells of a row at a time
// of its box, unless an earlier one's box has them too, and looks all modifications up for
// each cell as the plain kernel does.  12 steps of a settled 16384^2 world with a brush take
// 178 us, with the first step by the plain kernel instead, a pass over the ids that ends
// what is known of them, 852, and with the LDS kernels 211.
// ---------------------------------------------------------------------------
struct se_slbrush_args {  // the arguments as they lie in the kernel's argument segment
    se_slgrid g;
    int to;
    const se_mod* mods;
    int nmods;
    unsigned char* calm;
    int cols;
    se_few few;
};

extern "C" __global__ __launch_bounds__(256) void se_sl_brush(se_slgrid g, int to, const se_mod* __restrict__ list,
                                                              int nmods, unsigned char* calm, int cols, se_few) {
    const se_cmods few = (se_cmods)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() +
                                    __builtin_offsetof(se_slbrush_args, few));
    const se_cmods mods = nmods <= SE_PLAIN_MODS ? few : (se_cmods)list;
    const int i = (int)blockIdx.y;
    const long r = max(mods[i].size, 0), mx = mods[i].x, my = mods[i].y;
    const long xa = max(mx - r, 0l), xb = min(mx + r, (long)g.W - 1), ya = max(my - r, 0l), yb = min(my + r, (long)g.H - 1);
    if (xa > xb || ya > yb) return;
    const int first = ((int)xa + g.xpad) >> 4, wide = (((int)xb + g.xpad) >> 4) - first + 1;
    const u64 units = (u64)wide * (u64)(yb - ya + 1);
    for (u64 u = (u64)blockIdx.x * 256 + threadIdx.x; u < units; u += (u64)gridDim.x * 256) {
        const int bc = first + (int)(u % (u64)wide), y = (int)ya + (int)(u / (u64)wide), x0 = 16 * bc - g.xpad;
        if (se_mods_touch(mods, i, x0, x0 + 15, y, y)) continue;
        uint2* p = se_sl_at(g, to, bc, y + g.ypad);
        uint2 v = *p;
#pragma unroll 1
        for (int c = 0; c < 16; c++) {
            const int x = x0 + c;
            const int id = x >= 0 && x < g.W ? se_mod_override(mods, nmods, x, y) : -1;
            if (id < 0) continue;
            const u32 code = se_sl_codes((u32)id) & 0xffu;
            u32 w = c & 1 ? v.y : v.x;
#pragma unroll
            for (int k = 0; k < SE_SL_K; k++) {
                const u32 bit = 1u << (8 * k + (c >> 1));
                w = (code >> k) & 1u ? w | bit : w & ~bit;
            }
            if (c & 1) v.y = w;
            else v.x = w;
        }
        *p = v;
        if (calm != nullptr) calm[((y + g.ypad) >> 6) * cols + (x0 >> 6) + 1] = 0xffu;  // 16 cells of one square
    }
}

// Batch forms of the other kernels: prefix sums count 64 x 64 tiles (pack, unpack).
extern "C" __global__ __launch_bounds__(256) void se_sl_bpack(const se_slworld* __restrict__ worlds,
                                                              const int* __restrict__ prefix, int n) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), t = (int)blockIdx.x * 4 + wave;
    if (t >= prefix[n]) return;
    const int w = se_owner(prefix, n, t), i = t - prefix[w];
    const se_slgrid g = worlds[w].g;
    const int cols = 1 + (g.bcols - (g.xpad >> 4) + 3) / 4;
    se_sl_pack_tile(g, i % cols - 1, (i / cols) * 64, lds[wave], se_slknown{nullptr, nullptr, nullptr, 0}, 0);
}

extern "C" __global__ __launch_bounds__(256) void se_sl_bunpack(const se_slworld* __restrict__ worlds,
                                                                const int* __restrict__ prefix, int n) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), t = (int)blockIdx.x * 4 + wave;
    if (t >= prefix[n]) return;
    const int w = se_owner(prefix, n, t), i = t - prefix[w];
    const se_slgrid g = worlds[w].g;
    const int cols = 1 + (g.bcols - (g.xpad >> 4) + 3) / 4;  // as packing: the first column holds no cells
    if (i % cols > 0) se_sl_unpack_tile(g, worlds[w].result, i % cols - 1, (i / cols) * 64, lds[wave], se_slknown{nullptr, nullptr, nullptr, 0}, 0);
}

// The words of all groups in one row of workgroups (prefix counts 256 of them): a grid
// over the largest group's extents would be mostly empty workgroups (25 groups of a
// 48-world batch: 103 us a launch, and the work in it some 15).
extern "C" __global__ __launch_bounds__(256) void se_sl_bhash(const se_slgrid* __restrict__ groups,
                                                              const int* __restrict__ prefix, int n) {
    const int w = se_owner(prefix, n, (int)blockIdx.x);
    const se_slgrid g = groups[w];
    const u32 t = (u32)((int)blockIdx.x - prefix[w]) * 256u + threadIdx.x, set = t / (u32)g.hash_words;
    if (set < (u32)g.hash_sets) se_sl_hash_word(g, (int)(t - set * (u32)g.hash_words), (int)set);
}
