
// ---------------------------------------------------------------------------
// Sliced kernels: a cell is SE_SL_K bits spread over as many words, a word holds
// one bit of 32 cells.  Appended after se_kernels.hip and the sliced form of the
// rule set (SE_SL_*, se_sliced_block; se_hipgen.cpp).
//
// A row is held as E words (even columns) and O words (odd columns), so bit i of
// E and of O is the block of columns 2i and 2i + 1, and with the row below them a
// word quadruple is 32 blocks, which se_sliced_block advances at once.
//
// Packed grid in memory: u16 [half column][row][2K].  A half column is 32 cells
// wide; the entries of a row are E planes 0..K-1, then O planes.  Column c and
// row m of it are the world's x = c - xpad and y = m - ypad; everything around
// the world is WALL.
//
// Hash planes: u32 [frame][plane][word column][block row]; bit i of word w is the
// block whose columns at an even x offset are 64w + 2i and 64w + 2i + 1.  At an
// odd offset bit i is the block one column to the left, and at an odd y offset
// block row j is one row further down (rows 2j + 1 and 2j + 2).
// ---------------------------------------------------------------------------
typedef unsigned short u16;
typedef unsigned short se_u16x4 __attribute__((ext_vector_type(4)));

struct se_slgrid {  // == SlicedGrid (se_sliced.hpp)
    u32* in;        // the grid (u32 ids)
    u32* out;
    u16* pk[2];     // packed grids
    u32* hash;      // hash planes of frames hash_frame0 ...
    int W, H, pitch;
    int xpad, ypad, hcols, rows;  // packed geometry: columns of 32 cells, rows (a multiple of 64)
    int wcols, brows;             // hash planes: word columns, block rows (even)
    int hash_frame0;
};

__device__ __forceinline__ u32 se_sl_alignbit(u32 hi, u32 lo, int n) { return __builtin_amdgcn_alignbit(hi, lo, n); }

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
#if SE_SL_REMAP
    return se_sl_map(q, SE_SL_CODE0, SE_SL_CODE1, SE_SL_CODE2, SE_SL_CODE3);
#else
    return q;
#endif
}
__device__ __forceinline__ u32 se_sl_ids(u32 q) {
#if SE_SL_REMAP
    return se_sl_map(q, SE_SL_ID0, SE_SL_ID1, SE_SL_ID2, SE_SL_ID3);
#else
    return q;
#endif
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
// K/8 B written.  The second packed grid gets the rows and half columns around
// the world too, which the step kernel reads and never writes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ u16* se_sl_at(u16* p, const se_slgrid& g, int hcol, int row) {
    return p + ((size_t)hcol * g.rows + row) * (2 * SE_SL_K);
}

__device__ __forceinline__ void se_sl_put(u16* p, const u32* e, const u32* o, int half) {
    u16 v[2 * SE_SL_K];
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) {
        v[k] = (u16)(e[k] >> (16 * half));
        v[SE_SL_K + k] = (u16)(o[k] >> (16 * half));
    }
    u32* q = reinterpret_cast<u32*>(p);
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) q[k] = (u32)v[2 * k] | ((u32)v[2 * k + 1] << 16);
}

__device__ __forceinline__ void se_sl_pack_tile(const se_slgrid& g, int wc, int m0, u32* lds) {
    const int lane = (int)(threadIdx.x & 63);
    const int x = 64 * wc - g.xpad + 4 * (lane & 15);
    constexpr u32 WALL4 = SE_SL_WALL * 0x01010101u;
    uint4 v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int y = m0 + 4 * i + (lane >> 4) - g.ypad;
        v[i] = make_uint4(SE_WALLID, SE_WALLID, SE_WALLID, SE_WALLID);
        if (y >= 0 && y < g.H && x >= 0 && x < g.W)
            v[i] = *reinterpret_cast<const uint4*>(g.in + (size_t)y * g.pitch + x);
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const u32 mx = max(max(v[i].x, v[i].y), max(v[i].z, v[i].w));
        u32 q;
        if (__builtin_expect(mx >= SE_NMAT, 0))
            q = se_pack4(se_decode(v[i].x), se_decode(v[i].y), se_decode(v[i].z), se_decode(v[i].w));
        else
            q = se_pack4(v[i].x, v[i].y, v[i].z, v[i].w);
        q = se_sl_codes(q);
        const int in = g.W - x;  // cells of the quad inside the world
        if (in < 4 && in > 0) {
            const u32 keep = 0xffffffffu >> (8 * (4 - in));
            q = (q & keep) | (WALL4 & ~keep);
        }
        lds[(4 * i + (lane >> 4)) * 17 + (lane & 15)] = q;
    }
    __builtin_amdgcn_wave_barrier();
    u32 q[16], e[SE_SL_K], o[SE_SL_K], de[8], dd[8];
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
    const int row = m0 + lane;
    const bool around_y = row < g.ypad || row >= g.ypad + g.H;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int hc = 2 * wc + half;
        if (hc >= g.hcols || row >= g.rows) continue;
        se_sl_put(se_sl_at(g.pk[0], g, hc, row), e, o, half);
        const int c = 32 * hc - g.xpad;
        if (around_y || c < 0 || c + 32 > g.W) se_sl_put(se_sl_at(g.pk[1], g, hc, row), e, o, half);
    }
}

// packed grid `from` -> u32 grid (the cells of the world only)
__device__ __forceinline__ void se_sl_unpack_tile(const se_slgrid& g, int from, int wc, int m0, u32* lds) {
    const int lane = (int)(threadIdx.x & 63);
    u32 e[SE_SL_K], o[SE_SL_K], de[8], dd[8], q[16];
#pragma unroll
    for (int k = 0; k < SE_SL_K; k++) e[k] = o[k] = 0u;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int hc = 2 * wc + half, row = m0 + lane;
        if (hc >= g.hcols || row >= g.rows) continue;
        const u32* p = reinterpret_cast<const u32*>(se_sl_at(g.pk[from], g, hc, row));
        u32 v[SE_SL_K];
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) v[k] = p[k];
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) {
            const u32 ev = (v[k / 2] >> (16 * (k & 1))) & 0xffffu;
            const u32 ov = (v[(SE_SL_K + k) / 2] >> (16 * ((SE_SL_K + k) & 1))) & 0xffffu;
            e[k] |= ev << (16 * half);
            o[k] |= ov << (16 * half);
        }
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
    const int x = 64 * wc - g.xpad + 4 * (lane & 15);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int y = m0 + 4 * i + (lane >> 4) - g.ypad;
        const u32 p = lds[(4 * i + (lane >> 4)) * 17 + (lane & 15)];
        if (y < 0 || y >= g.H || x < 0 || x >= g.W) continue;
        u32* dst = g.out + (size_t)y * g.pitch + x;
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

extern "C" __global__ __launch_bounds__(256) void se_sl_pack(se_slgrid g, int wtiles, int tiles) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = (int)(threadIdx.x >> 6), t = (int)blockIdx.x * 4 + wave;
    if (t >= tiles) return;
    se_sl_pack_tile(g, t % wtiles, (t / wtiles) * 64, lds[wave]);
}

extern "C" __global__ __launch_bounds__(256) void se_sl_unpack(se_slgrid g, int from, int wtiles, int tiles) {
    __shared__ u32 lds[4][64 * 17];
    const int wave = (int)(threadIdx.x >> 6), t = (int)blockIdx.x * 4 + wave;
    if (t >= tiles) return;
    se_sl_unpack_tile(g, from, t % wtiles, (t / wtiles) * 64, lds[wave]);
}

// ---------------------------------------------------------------------------
// Hash planes of `nf` frames from hash_frame0 on.  A thread makes the words of one
// (frame, word column, block row): lanes are consecutive block rows, so the
// stores are contiguous, and a thread steps its hash inputs along x by a constant.
// Bound by VALU issue: per block and hash lane two 32-bit multiplies and three
// shifted exclusive ors, and two instructions per plane (compare, shift it in).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void se_sl_hash_word(const se_slgrid& g, int fi, int wc, int j) {
    const u32 f = (u32)(g.hash_frame0 + fi);
    int ox, oy;
    se_offset(f, ox, oy);
    const int y = 2 * j + oy - g.ypad, x = 64 * wc + 62 - ox - g.xpad;  // block of bit 31
    u32 in[4], acc[SE_SL_P];
#pragma unroll
    for (int l = 0; l < 4; l++)
        in[l] = (u32)x * se_hash_ka(l) + (u32)y * se_hash_kb(l) + f * se_hash_kf(l);
#pragma unroll
    for (int p = 0; p < SE_SL_P; p++) acc[p] = 0u;
#pragma unroll 4
    for (int i = 0; i < 32; i++) {
        u32 h[4];
        bool c[SE_SL_P];
#pragma unroll
        for (int l = 0; l < 4; l++) h[l] = se_sliced_lane(l) ? se_lowbias(in[l]) : 0u;
        se_sliced_classes(h, c);
#pragma unroll
        for (int p = 0; p < SE_SL_P; p++) acc[p] = acc[p] + acc[p] + (c[p] ? 1u : 0u);
#pragma unroll
        for (int l = 0; l < 4; l++) in[l] -= 2u * se_hash_ka(l);
    }
#pragma unroll
    for (int p = 0; p < SE_SL_P; p++)
        g.hash[(((size_t)fi * SE_SL_P + p) * g.wcols + wc) * g.brows + j] = acc[p];
}

extern "C" __global__ __launch_bounds__(256) void se_sl_hash(se_slgrid g, int nf) {
    const int j = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (j >= g.brows) return;
    for (int c = (int)blockIdx.y; c < nf * g.wcols; c += (int)gridDim.y) se_sl_hash_word(g, c / g.wcols, c % g.wcols, j);
}

// ---------------------------------------------------------------------------
// Step kernel: one wavefront advances a tile of NW words (64 * NW columns) by
// 64 * R rows through `nsub` sub-steps entirely in registers.  Lane l holds rows
// R*l .. R*l + R - 1 of every word column.
//   * y offset 1: every lane gives its first row to the lane above it (a wave
//     shift) and the rows move up by one, until the offset returns to 0; the
//     tile's outermost rows take WALL.
//   * x offset 1: the O words move up by one block (alignbit over the word
//     columns) and the blocks are (O, E) instead of (E, O).
// Blocks are never split between lanes otherwise, so there are no barriers and no
// LDS.  What the shifts bring in at the tile's sides is wrong inside the world and
// right at its border (WALL), so the valid region shrinks by one cell per
// sub-step on the sides that cut into the world: 32 columns and `halo` rows are
// given up on each side of a tile, none of a world that fits one tile.
// ---------------------------------------------------------------------------
template <int NW, int R>
struct se_sltile {
    u32 e[R][NW][SE_SL_K], o[R][NW][SE_SL_K];
};

__device__ __forceinline__ constexpr u32 se_sl_wall(int k) { return (SE_SL_WALL >> k) & 1u ? 0xffffffffu : 0u; }

// lane i gets lane i + 1 (wave_shl), the last lane `fill`; and the other way round
__device__ __forceinline__ u32 se_sl_from_below(u32 v, u32 fill) {
    return (u32)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ u32 se_sl_from_above(u32 v, u32 fill) {
    return (u32)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x138, 0xf, 0xf, false);
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_rows_up(se_sltile<NW, R>& t) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int k = 0; k < SE_SL_K; k++) {
            const u32 e = se_sl_from_below(t.e[0][w][k], se_sl_wall(k)), o = se_sl_from_below(t.o[0][w][k], se_sl_wall(k));
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
            const u32 e = se_sl_from_above(t.e[R - 1][w][k], se_sl_wall(k)),
                      o = se_sl_from_above(t.o[R - 1][w][k], se_sl_wall(k));
#pragma unroll
            for (int r = R - 1; r > 0; r--) {
                t.e[r][w][k] = t.e[r - 1][w][k];
                t.o[r][w][k] = t.o[r - 1][w][k];
            }
            t.e[0][w][k] = e;
            t.o[0][w][k] = o;
        }
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_hash_load(const se_slgrid& g, int fi, int wc0, int j0,
                                                u32 (&h)[NW][R / 2][SE_SL_P]) {
#pragma unroll
    for (int p = 0; p < SE_SL_P; p++)
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const u32* s = g.hash + (((size_t)fi * SE_SL_P + p) * g.wcols + wc0 + w) * g.brows + j0;
#pragma unroll
            for (int b = 0; b < R / 2; b++) h[w][b][p] = s[b];
        }
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_advance(se_sltile<NW, R>& t, const se_slgrid& g, int wc0, int row0, int lane,
                                              int frame0, int nsub) {
    const int j0 = row0 / 2 + (R / 2) * lane;
    int ysh = 0;
    u32 h[NW][R / 2][SE_SL_P];
    se_sl_hash_load<NW, R>(g, frame0 - g.hash_frame0, wc0, j0, h);
#if !SE_SL_KEEP
    const bool edge = 64 * wc0 < g.xpad || 64 * (wc0 + NW) > g.xpad + g.W || row0 < g.ypad ||
                      row0 + 64 * R > g.ypad + g.H;
#endif
    for (int s = 0; s < nsub; s++) {
        int ox, oy;
        se_offset((u32)(frame0 + s), ox, oy);
        u32 hn[NW][R / 2][SE_SL_P];  // the next sub-step's hash planes are in flight during this one
        se_sl_hash_load<NW, R>(g, frame0 - g.hash_frame0 + min(s + 1, nsub - 1), wc0, j0, hn);
        if (oy != ysh) {
            if (oy) se_sl_rows_up(t);
            else se_sl_rows_down(t);
            ysh = oy;
        }
        if (ox) {
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++)
#pragma unroll
                    for (int w = NW - 1; w >= 0; w--)
                        t.o[r][w][k] = se_sl_alignbit(t.o[r][w][k], w ? t.o[r][w - 1][k] : se_sl_wall(k), 31);
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int b = 0; b < R / 2; b++)
                    se_sliced_block(t.o[2 * b][w], t.e[2 * b][w], t.o[2 * b + 1][w], t.e[2 * b + 1][w], h[w][b]);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int k = 0; k < SE_SL_K; k++)
#pragma unroll
                    for (int w = 0; w < NW; w++)
                        t.o[r][w][k] = se_sl_alignbit(w + 1 < NW ? t.o[r][w + 1][k] : se_sl_wall(k), t.o[r][w][k], 1);
        } else {
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int b = 0; b < R / 2; b++)
                    se_sliced_block(t.e[2 * b][w], t.o[2 * b][w], t.e[2 * b + 1][w], t.o[2 * b + 1][w], h[w][b]);
        }
#if !SE_SL_KEEP
        if (edge) {  // rules may change the WALL outside the world: it is put back
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int y = row0 + R * lane + r + ysh - g.ypad;
                const u32 rm = y >= 0 && y < g.H ? 0xffffffffu : 0u;
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    const int x0 = 64 * (wc0 + w) - g.xpad;  // column of bit 0 of E
                    const int lo = x0 < 0 ? (-x0 + 1) / 2 : 0, lo1 = x0 < 0 ? -x0 / 2 : 0;
                    const int hi = min(32, max(0, (g.W - x0 + 1) / 2)), hi1 = min(32, max(0, (g.W - x0) / 2));
                    const u32 me = (u32)((1ull << hi) - 1ull) & ~(u32)((1ull << min(lo, 32)) - 1ull) & rm;
                    const u32 mo = (u32)((1ull << hi1) - 1ull) & ~(u32)((1ull << min(lo1, 32)) - 1ull) & rm;
#pragma unroll
                    for (int k = 0; k < SE_SL_K; k++) {
                        t.e[r][w][k] = (t.e[r][w][k] & me) | (se_sl_wall(k) & ~me);
                        t.o[r][w][k] = (t.o[r][w][k] & mo) | (se_sl_wall(k) & ~mo);
                    }
                }
            }
        }
#endif
#pragma unroll
        for (int w = 0; w < NW; w++)
#pragma unroll
            for (int b = 0; b < R / 2; b++)
#pragma unroll
                for (int p = 0; p < SE_SL_P; p++) h[w][b][p] = hn[w][b][p];
    }
    if (ysh) se_sl_rows_down(t);
}

// Rows of two neighbouring half columns <-> words (R rows x 2K planes each).
template <int NW, int R>
__device__ __forceinline__ void se_sl_load(se_sltile<NW, R>& t, u16* pk, const se_slgrid& g, int hc0, int row) {
    constexpr int D = R * SE_SL_K;  // u32 of a lane's rows in one half column
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const u32* a = reinterpret_cast<const u32*>(se_sl_at(pk, g, hc0 + 2 * w, row));
        const u32* b = reinterpret_cast<const u32*>(se_sl_at(pk, g, hc0 + 2 * w + 1, row));
        u32 va[D], vb[D];
#pragma unroll
        for (int i = 0; i < D; i += 2) {
            *reinterpret_cast<uint2*>(va + i) = *reinterpret_cast<const uint2*>(a + i);
            *reinterpret_cast<uint2*>(vb + i) = *reinterpret_cast<const uint2*>(b + i);
        }
#pragma unroll
        for (int i = 0; i < 2 * D; i++) {
            const int r = i / (2 * SE_SL_K), k = i % (2 * SE_SL_K);
            const u32 v = __builtin_amdgcn_perm(vb[i / 2], va[i / 2], i & 1 ? 0x07060302u : 0x05040100u);
            if (k < SE_SL_K) t.e[r][w][k] = v;
            else t.o[r][w][k - SE_SL_K] = v;
        }
    }
}

template <int NW, int R>
__device__ __forceinline__ void se_sl_store(const se_sltile<NW, R>& t, u16* pk, const se_slgrid& g, int hc0, int row,
                                            int first, int last) {
    constexpr int D = R * SE_SL_K;
#pragma unroll
    for (int hc = 0; hc < 2 * NW; hc++) {
        if (hc < first || hc > last) continue;
        u32* a = reinterpret_cast<u32*>(se_sl_at(pk, g, hc0 + hc, row));
        u32 v[D];
#pragma unroll
        for (int i = 0; i < D; i++) {
            u32 lo, hi;
            {
                const int r = 2 * i / (2 * SE_SL_K), k = 2 * i % (2 * SE_SL_K);
                lo = k < SE_SL_K ? t.e[r][hc / 2][k] : t.o[r][hc / 2][k - SE_SL_K];
            }
            {
                const int r = (2 * i + 1) / (2 * SE_SL_K), k = (2 * i + 1) % (2 * SE_SL_K);
                hi = k < SE_SL_K ? t.e[r][hc / 2][k] : t.o[r][hc / 2][k - SE_SL_K];
            }
            v[i] = __builtin_amdgcn_perm(hi, lo, hc & 1 ? 0x07060302u : 0x05040100u);
        }
#pragma unroll
        for (int i = 0; i < D; i += 2) *reinterpret_cast<uint2*>(a + i) = *reinterpret_cast<uint2*>(v + i);
    }
}

// `from`: the packed grid read, the other is written.  halo 0: the world fits the
// one tile, all of which is stored.
template <int NW, int R>
__device__ __forceinline__ void se_sl_tile(const se_slgrid& g, int from, int tx, int ty, int frame0, int nsub,
                                           int halo) {
    const int lane = (int)(threadIdx.x & 63);
    const int hc0 = tx * (2 * NW - 2), row0 = ty * (64 * R - 2 * halo);
    const int row = row0 + R * lane;
    se_sltile<NW, R> t;
    se_sl_load<NW, R>(t, g.pk[from], g, hc0, row);
    se_sl_advance<NW, R>(t, g, hc0 / 2, row0, lane, frame0, nsub);
    if (R * lane < halo || R * lane >= 64 * R - halo) return;
    if (halo == 0) se_sl_store<NW, R>(t, g.pk[from ^ 1], g, hc0, row, 0, 2 * NW - 1);
    else se_sl_store<NW, R>(t, g.pk[from ^ 1], g, hc0, row, 1, 2 * NW - 2);
}

#define SE_SL_STEP(NW, R)                                                                                     \
    extern "C" __global__ __launch_bounds__(64) void se_sl_step_##NW##x##R(se_slgrid g, int from, int tiles_x, \
                                                                           int frame0, int nsub, int halo) {   \
        const int tile = se_xcd_tile((int)blockIdx.x, (int)gridDim.x);                                         \
        se_sl_tile<NW, R>(g, from, tile % tiles_x, tile / tiles_x, frame0, nsub, halo);                        \
    }
SE_SL_STEP(2, 2)
SE_SL_STEP(4, 2)
SE_SL_STEP(4, 4)
