// Advancing one world with the sliced kernels (se_sliced.hip).
//
// A call packs the grid into bit planes once, advances the planes in launches of
// up to 32 sub-steps -- a packed cell is K bits, so the passes between the first
// and the last one move an eighth of what a pass over ids moves -- and writes ids
// back once.  The hash planes of the frames ahead are made by a kernel of their
// own, which hashes every block of the world once and not once per tile that
// covers it.
#include "se_sliced.hpp"

#include <algorithm>
#include <cmath>

using se_rt::DeviceGuard;
using se_rt::fail;

namespace {

constexpr size_t kKnownSquares = 1024;      // from so many 64 x 64 squares on a world keeps what is known of them
constexpr size_t kFewSquares = 2048;        // up to so many a run is a chain of sub-steps, beyond its tiles can sleep
constexpr size_t kHashBudget = 128u << 20;  // hash planes made ahead, unless one launch needs more

struct Tile {
    int nw, r, waves;
};
constexpr Tile kTiles[4] = {{2, 2, 1}, {4, 2, 1}, {2, 2, 2}, {4, 2, 4}};  // as instantiated in se_sliced.hip

void set_tile(se_rt::SlicedShape& s, int kernel) {
    s.kernel = kernel;
    s.nw = kTiles[kernel].nw;
    s.r = kTiles[kernel].r;
    s.threads = 64u * kTiles[kernel].waves;
}

template <typename... A>
int launch2(hipFunction_t f, unsigned gx, unsigned gy, unsigned block, hipStream_t s, A... args) {
    void* p[] = {(void*)&args...};
    hipError_t e = hipModuleLaunchKernel(f, gx, gy, 1, block, 1, 1, 0, s, p, nullptr);
    if (e != hipSuccess) return fail(SE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
    return SE_OK;
}

// Workgroups a modification for se_sl_brush: the largest box of `list` at 16 cells a
// thread, or a fixed number where the list is in device memory; they stride over more.
unsigned brush_blocks(const se_world& w, const se_modification* list, int n) {
    uint64_t most = list ? 1 : 64;
    for (int i = 0; list && i < n; i++) {
        const uint64_t side = 2ull * (uint64_t)std::max(list[i].mod_size, 0) + 1;
        most = std::max(most, (std::min<uint64_t>(side, w.W) / 16 + 2) * std::min<uint64_t>(side, w.H) / 256 + 1);
    }
    return (unsigned)std::min<uint64_t>(most, 4096);
}

}  // namespace

// A world with its WALL border inside one tile needs no halo: one column and one row
// more than the world has to the right and below (the wave shifts bring WALL in from
// the other sides).
se_rt::SlicedShape se_rt::sliced_one_tile(uint32_t W, uint32_t H, bool wide) {
    SlicedShape s;
    for (int i = 2; i < (wide ? 4 : 3) && !s.nw; i++) {
        if (W + 4 > 64u * kTiles[i].nw - 1 || H + 2 > 64u * kTiles[i].r) continue;
        set_tile(s, i);
        s.tiles_x = s.tiles_y = 1;
        s.max_sub = 1u << 20;
    }
    return s;
}

// The tile and the depth of a launch, by how many squares of 64 x 64 cells the worlds
// make.  While those leave SIMDs idle a launch is a serial chain of sub-steps: split
// tiles, the small one first, and the deepest launch.  Beyond that the rows and
// columns given up count (16 columns a side up to 16 sub-steps, 32 beyond), and
// where one wavefront a tile has the registers for it, the barriers.  us a call without
// the seeded fill (2x2s 32 deep / 4x2s 32 / 2x2 16 / 4x2s 16, and from the third on 4x2 12):
//   1000x700   200 steps  113 / 120 / 160 / 138
//   2000x1900  200 steps  184 / 186 / 209 / 183 / 299
//   4096^2     200 steps  544 / 476 / 445 / 455 / 511
//   16384^2    100 steps     -      / 1505 / 1477 / 1367
// and with four planes (2x2s 32 / 4x2s 32 / 2x2s 16 / 4x2s 16)
//   800^2      150 steps  152 / 161 / 168 / 176
//   1537x1111  150 steps  221 / 191 / 199 / 203
//   4096^2      64 steps  433 / 366 / 338 / 341
//   8192^2      64 steps    -  /  -  / 703 / 646
// The deepest launch of one wavefront is 12 sub-steps; a run of up to 16 takes them in one
// launch and not in two (settled 16384^2: 201 us a call, 236 in two).
void se_rt::sliced_choice(size_t few, const SlicedKernels& K, int* kernel, uint32_t* deep) {
    const bool one_wave = K.step[0] != nullptr;
    if (few <= kFewSquares) {
        *kernel = few <= 256 ? 2 : 3;
        *deep = 32;
    } else if (few <= 8192) {
        *kernel = one_wave ? 0 : 2;
        *deep = 16;
    } else {
        *kernel = one_wave ? 1 : 3;
        *deep = one_wave ? 12 : 16;
    }
}

se_rt::SlicedShape se_rt::sliced_tiles(uint32_t W, uint32_t H, int kernel, uint32_t max_sub) {
    SlicedShape s;
    set_tile(s, kernel);
    s.max_sub = std::min(max_sub, 32u);
    s.halo = (int)(s.max_sub + 3) & ~3;
    s.side = s.max_sub > 16 ? 2 : 1;
    const uint32_t ux = 64u * s.nw - 32u * s.side, uy = 64u * s.r - 2u * s.halo;  // useful columns and rows of a tile
    s.tiles_x = (int)((W + ux - 1) / ux);
    s.tiles_y = (int)((H + uy - 1) / uy);
    return s;
}

// Packing covers the margins (one column of 64 more on the left); unpacking the
// world's columns.
int se_rt::sliced_pack_tiles(const SlicedGrid& g) { return (1 + (g.bcols - g.xpad / 16 + 3) / 4) * (g.rows / 64); }
int se_rt::sliced_unpack_columns(const SlicedGrid& g) { return (g.W + (g.xpad & 15) + 63) / 64; }

void se_rt::sliced_geometry(const SlicedShape& s, uint32_t W, uint32_t H, SlicedGrid& g) {
    g.W = (int)W;
    g.H = (int)H;
    if (s.halo == 0) {
        g.xpad = 4;  // keeps the 16-byte loads of ids aligned
        g.ypad = 2;
    } else {
        g.xpad = 16 * s.side;
        g.ypad = s.halo;
    }
    g.bcols = (s.tiles_x - 1) * (4 * s.nw - 2 * s.side) + 4 * s.nw;
    g.rows = ((s.tiles_y - 1) * (64 * s.r - 2 * s.halo) + 64 * s.r + 63) & ~63;
    g.brows = g.rows / 2;
}

size_t se_rt::sliced_packed_bytes(const SlicedGrid& g) {
    return ((size_t)g.bcols * g.rows * 8 + 255) & ~(size_t)255;
}

size_t se_rt::sliced_hash_layout(SlicedGrid& g, int32_t frame0, uint32_t nf, int classes) {
    const int wcols = (g.bcols + 3) / 4;
    g.hash_frame0 = frame0;
    // shared form: the range of n of each parity over the frames, and the words of b
    // that cover it (one more than a tile's last word, for the shifted read).  n grows by
    // 4.5 M a frame and the offsets change it by some thousands, and any four frames hold
    // both parities, so the first four and the last four frames bound it.
    int64_t lo[2] = {0, 0}, hi[2] = {-1, -1};
    for (uint32_t i = 0; i < nf; i = i == 3 && nf > 8 ? nf - 4 : i + 1) {
        const int64_t f = (int64_t)frame0 + i;
        const int ox = (int)(f & 1), oy = (f & 3) == 1 || (f & 3) == 2;
        const int64_t n = 461ll * (-ox - g.xpad) + 2131ll * (oy - g.ypad) + 4541161ll * f;
        const int c = (int)((ox + oy + f) & 1);
        if (hi[c] < lo[c]) lo[c] = hi[c] = n;
        lo[c] = std::min(lo[c], n);
        hi[c] = std::max(hi[c], n);
    }
    int64_t words = 0;
    for (int c = 0; c < 2; c++) {
        const int64_t m = (hi[c] - lo[c]) / 2 + 2131ll * g.brows + 461ll * 32 * (wcols + 1);
        words = std::max(words, (m / 461 + 2144) / 32 + 2);
    }
    g.hash_n0 = (uint32_t)lo[0];
    g.hash_n1 = (uint32_t)lo[1];
    // The shared form where it hashes less: its sets hold every n between the first
    // and the last, 4.5 M more with each frame, used or not.  16384^2 (67 M blocks a
    // frame) takes 1.6 us a frame and 21 direct, 8192^2 with twelve materials (17 M) 4
    // and 13; at 4096^2 (4.2 M) the direct form hashes less.
    const int64_t shared = 2 * words * 464, direct = (int64_t)nf * wcols * g.brows;
    g.hash_shared = shared < direct && words * 464 < (1ll << 26) ? 1 : 0;
    g.hash_pitch = g.hash_shared ? 464 : g.brows;
    g.hash_words = (int)(g.hash_shared ? words * 464 : (int64_t)wcols * g.brows);
    // The step kernel loads up to four frames past the last one and a word past a
    // row's last: 4 * 4541161 / 2 / 461 bits further on, or four more frames.
    g.hash_sets = g.hash_shared ? 2 : (int)nf;
    const size_t past = g.hash_shared ? (size_t)(4 * 4541161 / 2 / 461 / 32 + 70) * 464
                                      : 4 * (size_t)g.hash_words + g.brows;
    return ((size_t)g.hash_sets * g.hash_words + past) * classes * sizeof(uint32_t);
}

// As many whole launches at a time as the budget holds, at least one.  A later chunk
// can need more room than the first: it may be shorter and take the direct form, whose
// frames loaded ahead are larger than the shared form's.
se_rt::SlicedAhead se_rt::sliced_ahead(const SlicedShape& s, SlicedGrid g, int32_t frame0, uint32_t n, int classes) {
    const uint32_t per_launch = std::min(s.max_sub, n);
    SlicedAhead a;
    a.frames = std::min(n, kSlicedMostFrames);
    while (sliced_hash_layout(g, frame0, a.frames, classes) > kHashBudget && a.frames > (s.halo ? per_launch : 1u)) {
        a.frames = a.frames / 2;
        if (s.halo) a.frames = std::max(a.frames / per_launch, 1u) * per_launch;
    }
    for (uint32_t at = 0; at < n; at += a.frames)
        a.bytes = std::max(a.bytes, sliced_hash_layout(g, frame0 + (int32_t)at, std::min(a.frames, n - at), classes));
    return a;
}

// ---------------------------------------------------------------- LDS or sliced kernels
// Packing, hashing and unpacking cost three launches more than the LDS kernels have, and
// from the largest worlds a pass over the grid.  The LDS kernels' default tile advances 8
// steps in one launch and stays for those; the generated chain, where no table fits, does a
// step in the time of ten (measured per call, LDS against sliced, us: four materials 4096^2
// 8 steps 46 and 55, 12 steps 83 and 64; 16384^2 427 and 567, 831 and 607; twelve at 8192^2
// 226 and 223, 368 and 261; feature rules 4096^2 2 steps 52 and 53, 4 steps 88 and 66).
// From there on the sliced kernels are ahead in worlds of at least 128 cells a side with
// networks of up to 300 tables (1500^2 to 12000^2, 3000x8192, 200x40000 and the like, 9 to 32
// steps: 1.1 to 2.2 times faster with four and twelve materials).  Elsewhere the path is the
// one of the smaller estimate, which goes by times like these:
//   * worlds inside one LDS tile take all their steps in one launch (four materials, LDS /
//     sliced: 2x2 9 steps 19 / 27 us, 96 steps 56 / 53; 32x32 16 steps 27 / 28, 24 33 / 31;
//     64x64 9 steps 26 / 28, 12 29 / 28; 90x90 9 steps 31 / 28);
//   * worlds a few rows high fill a tenth of the sliced tiles, whose planes are hashed all
//     the same (20000x16 16 steps 28 / 34, 32 45 / 43; chain form 20000x1 128 steps 172 / 219);
//   * large networks beside a table (586 tables, 4096^2, 64 steps 487 / 475; 1661 565 / 901);
//   * batches whose worlds all start at different frames share no planes (2048 worlds of 64^2,
//     256 steps 956 / 2325 us, and 966 / 408 at one frame).
// Fitted to some 700 calls of seven rule sets; the estimates' choice costs at most a third
// more than the better path there, mostly in worlds a few rows high.
namespace {

bool one_lds_tile(uint32_t W, uint32_t H) { return W <= 112 && H <= 112; }

// The generated chain grows with the rules, as the network does.
double chain_scale(const se_rt::StepCost& c) { return c.form == 0 ? (c.tables + 100) / 200.0 : 1.0; }

// us a step of a world alone: a serial chain of LDS reads and barriers, longer by the tile's rows
double lds_latency(const se_rt::StepCost& c, uint32_t W, uint32_t H) {
    static const double one[3][2] = {{.75, .060}, {.40, .0105}, {1.05, .0145}};
    static const double many[3][2] = {{1.2, .056}, {.85, .0155}, {1.7, .018}};
    const double t = one_lds_tile(W, H) ? one[c.form][0] + one[c.form][1] * std::sqrt((double)W * H)
                                        : many[c.form][0] + many[c.form][1] * std::min(H, 112u);
    return chain_scale(c) * (c.form == 1 && !c.wall_kept ? 1.15 : 1.0) * t;
}

// us a step of a world that shares a full device with others
double lds_work(const se_rt::StepCost& c, uint32_t W, uint32_t H) {
    static const double tile[3][2] = {{.004, 8e-7}, {.0008, 2.0e-7}, {.0027, 2.6e-7}};
    const double* t = tile[c.form];
    if (one_lds_tile(W, H)) return chain_scale(c) * (t[0] + t[1] * W * H);
    return chain_scale(c) * (t[0] + t[1] * 16384) * ((W + 111) / 112) * ((H + 111) / 112);
}

// n steps, in steps of a long run: beyond one tile they come in launches of up to 8, and two
// fifths of a full one's time are the launch's own
double lds_steps(uint32_t W, uint32_t H, uint32_t n) {
    return one_lds_tile(W, H) ? n : 3.2 * ((n + 7) / 8) + .6 * n;
}

double sliced_latency(const se_rt::StepCost& c, bool one) {
    return (one ? .16 : .24) + .0021 * c.tables + (c.form == 0 && !c.wall_kept ? .06 : 0);
}

// us to hash a frame for planes of that geometry, n frames together
double hash_time(const se_rt::StepCost& c, se_rt::SlicedGrid g, uint32_t n) {
    n = std::min(n, 256u);
    se_rt::sliced_hash_layout(g, 1, n, 1);
    return .028e-6 * c.hash_ops * 32.0 * g.hash_words * g.hash_sets / n;
}

}  // namespace

bool se_rt::sliced_pays(const SlicedKernels& K, uint32_t W, uint32_t H, uint32_t n) {
    const StepCost& c = K.cost;
    if (!K.ok || n < sliced_least_steps(K)) return false;
    if (std::min(W, H) >= 128 && (c.form == 0 || c.tables <= 300)) return true;
    const SlicedShape s = sliced_shape(K, W, H, n, 0);
    SlicedGrid g;
    sliced_geometry(s, W, H, g);
    const double cells = 1e-6 * W * H, area = 16e-6 * g.bcols * g.rows;
    const double tiles = 12544e-6 * ((W + 111) / 112) * ((H + 111) / 112) * (std::min(H, 112u) + 16) / 128;
    const double work[3] = {1.0, c.wall_kept ? .20 : .42, .42};  // LDS kernels, us a step and M cells of its tiles
    const double alone = lds_latency(c, W, H), full = chain_scale(c) * work[c.form] * tiles;
    const double lds = (one_lds_tile(W, H) ? 15 : 12) + lds_steps(W, H, n) * (one_lds_tile(W, H) ? alone : std::hypot(alone, full));
    const double step = std::max(sliced_latency(c, !s.halo), (.0003 * c.tables + .006) * area);
    return 25 + (s.halo ? 2 : 0) + n * (step + hash_time(c, g, n)) + 1.55 * cells < lds;
}

bool se_rt::sliced_batch_pays(const SlicedKernels& K, const std::vector<SlicedLoad>& worlds) {
    const StepCost& c = K.cost;
    uint32_t most = 0;
    size_t squares = 0;
    for (auto& w : worlds) {
        most = std::max(most, w.n);
        if (w.n) squares += sliced_squares(w.W, w.H);
    }
    if (!K.ok || most < sliced_least_steps(K)) return false;
    int kernel;
    uint32_t deep;
    sliced_choice(squares, K, &kernel, &deep);
    // The lists that advance side by side: worlds beyond one tile, and the others.  Worlds
    // that start at the same frame share planes, as large as the largest needs.
    struct List {
        SlicedGrid most;      // extents
        uint32_t n = 0;       // steps
        size_t worlds = 0, groups = 0;
        double hash = 0;  // us, were each world's planes its own
    } lists[2];
    size_t slots = 64;
    while (slots < 4 * worlds.size()) slots *= 2;
    std::vector<int32_t> seen[2];  // first frames, a hash table
    SlicedLoad last{0, 0, 0, 0};
    SlicedGrid g;
    bool one = false;
    double t = 0, work = 0, chain = 0, sliced = 0, cells = 0, lds_all = 0, lds_chain = 0, sliced_all = 0, sliced_chain = 0, count = 0;
    for (auto& w : worlds) {
        if (!w.n) continue;
        if (w.W != last.W || w.H != last.H || w.n != last.n) {  // runs of equal worlds
            last = w;
            SlicedShape s = sliced_one_tile(w.W, w.H, false);
            one = s.nw != 0;
            if (!one) s = sliced_tiles(w.W, w.H, kernel, deep);
            g = SlicedGrid();
            sliced_geometry(s, w.W, w.H, g);
            t = hash_time(c, g, w.n);
            const double steps = lds_steps(w.W, w.H, w.n);
            work = steps * lds_work(c, w.W, w.H);
            chain = steps * lds_latency(c, w.W, w.H);
            sliced = w.n * c.tables * (one ? 3.9e-6 : 3.5e-6 * sliced_squares(w.W, w.H));
        }
        List& l = lists[one];
        if (!l.worlds) l.most = g;
        l.most.bcols = std::max(l.most.bcols, g.bcols);
        l.most.brows = std::max(l.most.brows, g.brows);
        l.n = std::max(l.n, w.n);
        l.worlds++;
        l.hash += w.n * t;
        std::vector<int32_t>& at = seen[one];
        if (at.empty()) at.assign(slots, INT32_MIN);
        size_t i = (uint32_t)w.frame * 2654435761u & (slots - 1);
        while (at[i] != INT32_MIN && at[i] != w.frame) i = (i + 1) & (slots - 1);
        l.groups += at[i] == INT32_MIN;
        at[i] = w.frame;
        count++;
        cells += 1e-6 * w.W * w.H;
        lds_all += work;
        lds_chain = std::max(lds_chain, chain);
        sliced_all += sliced;
        sliced_chain = std::max(sliced_chain, w.n * sliced_latency(c, one));
    }
    double host = 0;
    for (int k = 0; k < 2; k++) {
        const List& l = lists[k];
        if (!l.worlds) continue;
        const double us = l.groups == 1 ? l.n * hash_time(c, l.most, l.n) : l.hash * l.groups / l.worlds;
        sliced_all += us * (k ? 1.5 : 1.0);  // one tile: few words a set, waiting workgroups
        const double bytes = us / (.028e-6 * c.hash_ops) / 8 * K.classes;
        const double chunks = k ? std::max(1.0, bytes / (64 << 20)) : l.n <= 64 ? 1 : l.n <= 192 ? 2 : 2 + (l.n + 63) / 256;
        host += l.groups * (.08 + .12 * chunks) + (k ? 0 : 12 * (chunks - 1));
    }
    return 88 + .07 * count + host + std::max(sliced_chain, sliced_all) + 1.5 * cells <
           76 + .045 * count + std::hypot(lds_chain, lds_all);
}

se_rt::SlicedShape se_rt::sliced_shape(const SlicedKernels& K, uint32_t W, uint32_t H, uint32_t n, uint32_t sub) {
    SlicedShape s = sliced_one_tile(W, H, true);
    if (s.nw) {
        if (sub) s.max_sub = sub;
        return s;
    }
    int kernel;
    uint32_t deep;
    sliced_choice(sliced_squares(W, H), K, &kernel, &deep);
    if (deep < n && n <= 16) deep = 16;
    return sliced_tiles(W, H, kernel, sub ? std::min(sub, deep) : deep);
}

// A launch of one sub-step and se_sl_brush take some 10 us and a pass over the packed
// grid, a plain step 5 us and a pass over the ids, and it ends what is known of the
// grids (us a call of 12 steps with a brush, plain step / packed, dense worlds: twelve materials
// 2304x2112 54 / 58, 2816x2880 73 / 74, 4096^2 115 / 105, 8192^2 292 / 236; feature rules 62 / 65,
// 85 / 85, 131 / 121, 301 / 247; settled four materials 40 / 39, 52 / 45, 84 / 57, 222 / 87).
bool se_rt::sliced_takes_mods(const se_world* w, uint32_t n) {
    return n > 1 && sliced_squares(w->W, w->H) > kFewSquares;
}

bool se_rt::sliced_sleeps(const se_world* w, int kernel) {
    return w->sleep_enabled && sliced_squares(w->W, w->H) > kFewSquares && w->mod->sliced.sleep_step[kernel];
}

int se_rt::sliced_steps(se_world* w, uint32_t n, uint32_t sub, bool* done) {
    *done = false;
    const SlicedKernels& K = w->mod->sliced;
    const SlicedShape shape = sliced_shape(K, w->W, w->H, n, sub);
    SlicedWorld one;
    SlicedGrid& g = one.g;
    sliced_geometry(shape, w->W, w->H, g);
    g.pitch = (int)w->pitch;
    const size_t packed = sliced_packed_bytes(g);
    const SlicedAhead plan = sliced_ahead(shape, g, w->frame + 1, n, K.classes);
    const uint32_t ahead = plan.frames;
    const size_t bytes = 2 * packed + plan.bytes;

    const int ptiles = sliced_pack_tiles(g), pcols = ptiles / (g.rows / 64);
    const int ucols = sliced_unpack_columns(g), utiles = ucols * (g.rows / 64);
    // From some 4 M cells on known squares are not packed or unpacked, and from twice that on
    // settled tiles are only written (below, a call is a chain of launches and steps that a
    // settled tile does not shorten).  us a call of 12 steps of a settled world (stone below,
    // nothing above), sleeping LDS tiles / sliced kernels without / with this: four materials
    // 2816x2880 46 / 41 / 35, 4096^2 61 / 76 / 57, 8192^2 88 / 166 / 80, 16384^2 174 / 540 / 139,
    // twelve at 16384^2 312 / 748 / 240; a dense world pays up to 1 % (8192^2 twelve 749 / 756).
    // A caller who holds a grid's address may write it between two calls: nothing is known
    // from one to the next then.
    SlicedKnown known;
    hipFunction_t step = K.step[shape.kernel];
    const int variant = (int)w->mod->lds.size() - 1, layout = (g.xpad << 8 | g.ypad) << 16 | pcols;
    const size_t each = ((size_t)ptiles + 255) & ~(size_t)255;  // calm is read by whole words
    if (w->sleep_enabled && sliced_squares(w->W, w->H) >= kKnownSquares && sleep_room(w, 2 * each) == SE_OK) {
        if (!w->exposed) known.same = w->d_sleep[0];
        known.was = w->d_sleep[1];
        known.calm = w->d_sleep[1] + each;
        known.valid = known.same && w->sleep_variant == variant && w->sleep_layout == layout;
        if (sliced_sleeps(w, shape.kernel)) {
            step = K.sleep_step[shape.kernel];
            one.stable = K.stable;
            one.calm = known.calm;
            one.calm_cols = pcols;
        }
    }

    // The scratch belongs to the context: its worlds share one stream, and the
    // launches of one call are enqueued together under the lock.
    se_ctx* ctx = w->ctx;
    std::lock_guard<std::mutex> lk(ctx->pool->mu);
    Pool::Block& scratch = ctx->pool->scratch;
    if (bytes > scratch.bytes) {
        if (scratch.mem) Pool::drop(scratch);  // waits for the work that uses it
        if (hipMalloc(&scratch.mem, bytes) != hipSuccess) {
            (void)hipGetLastError();
            scratch.mem = nullptr;
            return SE_OK;
        }
        scratch.bytes = bytes;
    }
    ModsArg mods;
    FewMods few{};
    int rc = take_mods(w, mods, &few);
    if (rc) return rc;
    *done = true;
    one.frame0 = w->frame + 1;
    one.steps = (int)n;
    one.tiles_x = shape.tiles_x;
    one.side = shape.side;
    one.halo = shape.halo;
    g.in = w->buf[w->cur];
    g.out = w->buf[w->cur ^ 1];
    g.pk0 = scratch.mem;
    g.pk1 = (char*)scratch.mem + packed;
    g.hash = (uint32_t*)((char*)scratch.mem + 2 * packed);

    sleep_reset(w);  // until the run is enqueued
    rc = launch2(K.pack, (unsigned)(ptiles + 3) / 4, 1, 256, w->stream, g, pcols, ptiles, known);
    int from = 0;
    for (uint32_t at = 0; at < n && !rc;) {
        const uint32_t nf = std::min(ahead, n - at);
        sliced_hash_layout(g, w->frame + 1 + (int)at, nf, K.classes);
        rc = launch2(K.hash, (unsigned)(g.hash_words + 255) / 256, (unsigned)g.hash_sets, 256, w->stream, g);
        for (uint32_t d = 0; d < nf && !rc;) {
            // a launch after the first starts at the head of a cycle where that costs
            // no further launch
            const uint32_t lead = (uint32_t)(g.hash_frame0 + (int)d + (int)shape.max_sub) & 3u;
            uint32_t m = std::min(shape.max_sub, nf - d);
            if (m < nf - d && lead < m && (nf - d - (m - lead) + shape.max_sub - 1) / shape.max_sub ==
                                              (nf - d - m + shape.max_sub - 1) / shape.max_sub)
                m -= lead;
            if (at + d == 0 && mods.n > 0) m = 1;  // modifications follow the first step
            rc = launch2(step, (unsigned)(shape.tiles_x * shape.tiles_y), 1, shape.threads, w->stream, one,
                         (const SlicedWorld*)nullptr, (const int*)nullptr, 0, (const SlicedGrid*)nullptr, from,
                         (int)(at + d), (int)m);
            from ^= 1;
            if (at + d == 0 && mods.n > 0 && !rc) {
                const unsigned blocks = brush_blocks(*w, mods.n <= kFewMods ? few.m : nullptr, mods.n);
                rc = launch2(K.brush, blocks, (unsigned)mods.n, 256, w->stream, g, from, (const void*)mods.ptr, mods.n,
                             (void*)known.calm, pcols, few);
            }
            d += m;
        }
        at += nf;
    }
    if (!rc) rc = launch2(K.unpack, (unsigned)(utiles + 3) / 4, 1, 256, w->stream, g, from, ucols, utiles, pcols, known);
    if (rc) return rc;
    if (known.same) {
        w->sleep_variant = variant;
        w->sleep_layout = layout;
    }
    w->frame += (int32_t)n;
    w->cur ^= 1;
    return SE_OK;
}
