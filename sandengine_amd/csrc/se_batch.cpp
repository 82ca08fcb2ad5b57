// Batched multi-world execution (se_batch_* in include/sandengine_hip.h).
//
// Many independent worlds advance together.  Worlds are grouped by rule set
// (one JIT module each).  Within a group:
//   * a world that fits one LDS tile keeps its WALL border in LDS, so one work
//     item advances it through all of its steps in a single launch;
//   * larger worlds advance in rounds of k sub-steps (k <= the tile halo): round
//     r covers every world with more than r*k steps; worlds are ordered by step
//     count (longest first) so the active set of a round is a prefix, and one
//     launch per round covers all of their tiles.
// Groups of a rule set with a sliced form run these two lists with the sliced kernels
// where that is estimated to be faster (SlicedPlan below).
// The single-tile launch and the rounds of every group go to their own streams
// and overlap on the device; these launches can be captured in one hipGraph, the sliced
// plans' are submitted beside it.  The reference has no batched mode: each Simulation is one world
// (sandengine-core/src/simulation.rs:97-126); the per-world step is the same.
#include <algorithm>
#include <cstdio>

#include "se_internal.hpp"
#include "se_sliced.hpp"

using se_rt::DeviceGuard;
using se_rt::fail;
using se_rt::launch_ex;

namespace {

// == se_bworld in se_kernels.hip
struct BWorld {
    uint32_t* buf[2];
    int W, H, pitch, tiles_x, ntiles;
    int frame0;
    int steps;
    int cur0;
    const void* mods;
    int nmods;
    int pad;
};
static_assert(sizeof(BWorld) == 64, "se_bworld layout");

struct DevArray {
    void* p = nullptr;
    ~DevArray() {
        if (p) (void)hipFree(p);
    }
};

// Events, a captured graph and its executable, released on every exit path.
struct RunResources {
    std::vector<hipEvent_t> events;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<hipStream_t> streams;  // drained first: launches may still read the plans' arrays
    RunResources() = default;
    RunResources(const RunResources&) = delete;
    RunResources& operator=(const RunResources&) = delete;
    ~RunResources() {
        for (auto s : streams)
            if (s) (void)hipStreamSynchronize(s);
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (auto e : events) (void)hipEventDestroy(e);
    }
    int event(hipEvent_t* out, unsigned flags) {
        HIPCHECK(hipEventCreateWithFlags(out, flags));
        events.push_back(*out);
        return SE_OK;
    }
};

}  // namespace

struct se_batch {
    se_ctx* ctx = nullptr;
    std::vector<std::pair<se_world*, uint32_t>> items;
    struct Tuned {
        int vi;           // LDS variant index
        uint32_t k;       // sub-steps per round
        bool persistent;  // launch shape (see enqueue_plan)
    };
    std::map<se_module*, Tuned> tuned;
    hipStream_t streams[8] = {};
    // records, packed grids and hash planes of the sliced plans, kept from run to run
    // (which end with the device idle), freed by se_batch_clear or when another allocation
    // of the device fails
    std::shared_ptr<se_rt::Pool> pool;
    se_rt::Pool::Block arena;
    ~se_batch() {
        if (pool) {
            std::lock_guard<std::mutex> lk(pool->mu);
            pool->arenas.erase(std::find(pool->arenas.begin(), pool->arenas.end(), &arena));
            se_rt::Pool::drop(arena);
        }
        for (auto s : streams)
            if (s) (void)hipStreamDestroy(s);
    }
};

namespace {

struct Plan {
    se_module* mod = nullptr;
    int vi = 0;
    uint32_t k = 8;
    std::vector<std::pair<se_world*, uint32_t>> small, large;  // (world, steps), steps descending
    std::vector<int> n_active;                                  // per round, large list
    DevArray d_small, d_large, d_pre_small, d_pre_large;
    std::vector<int> pre_small, pre_large;                      // host copies of the tile prefix sums
    bool persistent = false;                                     // launch shape (see enqueue_plan)
};

bool fits_one_tile(const se_world* w, const se::LdsVariant& v) {
    return w->W <= (uint32_t)v.tw && w->H <= (uint32_t)v.th;
}

int upload_list(const std::vector<std::pair<se_world*, uint32_t>>& list, const se::LdsVariant& v, DevArray& dw,
                DevArray& dp, std::vector<int>& pre) {
    std::vector<BWorld> recs;
    pre.assign(1, 0);
    for (auto& it : list) {
        se_world* w = it.first;
        BWorld b;
        b.buf[0] = w->buf[0];
        b.buf[1] = w->buf[1];
        b.W = (int)w->W;
        b.H = (int)w->H;
        b.pitch = (int)w->pitch;
        b.tiles_x = (int)((w->W + v.tw - 1) / v.tw);
        b.ntiles = b.tiles_x * (int)((w->H + v.th - 1) / v.th);
        b.frame0 = w->frame + 1;
        b.steps = (int)it.second;
        b.cur0 = w->cur;
        b.mods = nullptr;
        b.nmods = 0;
        b.pad = 0;
        recs.push_back(b);
        pre.push_back(pre.back() + b.ntiles);
    }
    if (recs.empty()) return SE_OK;
    HIPCHECK(hipMalloc(&dw.p, recs.size() * sizeof(BWorld)));
    HIPCHECK(hipMalloc(&dp.p, pre.size() * sizeof(int)));
    HIPCHECK(hipMemcpy(dw.p, recs.data(), recs.size() * sizeof(BWorld), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(dp.p, pre.data(), pre.size() * sizeof(int), hipMemcpyHostToDevice));
    return SE_OK;
}

int make_plan(se_ctx* ctx, se_module* mod, int vi, uint32_t k, const std::vector<std::pair<se_world*, uint32_t>>& ws,
              Plan& P) {
    const se::LdsVariant& v = mod->lds[vi].first;
    if (k == 0 || k > (uint32_t)v.hb) k = (uint32_t)v.hb;
    P.mod = mod;
    P.vi = vi;
    P.k = k;
    for (auto& it : ws) {
        if (it.second == 0) continue;
        (fits_one_tile(it.first, v) ? P.small : P.large).push_back(it);
    }
    auto by_steps = [](const std::pair<se_world*, uint32_t>& a, const std::pair<se_world*, uint32_t>& b) {
        return a.second > b.second;
    };
    std::stable_sort(P.small.begin(), P.small.end(), by_steps);
    std::stable_sort(P.large.begin(), P.large.end(), by_steps);
    if (!P.large.empty()) {
        uint32_t rounds = (P.large[0].second + k - 1) / k;
        for (uint32_t r = 0; r < rounds; r++) {
            int n = 0;
            while (n < (int)P.large.size() && P.large[n].second > r * k) n++;
            P.n_active.push_back(n);
        }
    }
    int rc = upload_list(P.small, v, P.d_small, P.d_pre_small, P.pre_small);
    if (!rc) rc = upload_list(P.large, v, P.d_large, P.d_pre_large, P.pre_large);
    return rc;
}

// Enqueues a plan's launches: single-tile worlds on `s_small`, rounds on `s_large`.
// Two launch shapes of the same kernel:
//   * one workgroup per work item (the kernel's item loop runs once);
//     workgroups that start as others retire keep the loads and compute of
//     different items overlapped, and the longest-first order makes the
//     dispatch order a longest-first schedule;
//   * persistent: as many workgroups as are resident at once, each striding
//     over the items.
// The autotuner measures both.
int enqueue_plan(Plan& P, hipStream_t s_small, hipStream_t s_large) {
    const se::LdsVariant& v = P.mod->lds[P.vi].first;
    hipFunction_t f = P.mod->batch[P.vi];
    const unsigned shmem = 0;  // the LDS kernels' LDS is static
    const uint32_t* tbl = P.mod->table;
    auto grid = [&](int items) {
        return (unsigned)(P.persistent ? std::min(items, P.mod->lds_grid[P.vi]) : items);
    };
    if (!P.small.empty()) {
        int n = (int)P.small.size();
        int rc = launch_ex(f, grid(P.pre_small.back()), (unsigned)v.nt, shmem, s_small, (const void*)P.d_small.p,
                           (const int*)P.d_pre_small.p, n, 0, (int)(1 << 30), tbl);
        if (rc) return rc;
    }
    for (size_t r = 0; r < P.n_active.size(); r++) {
        int rc = launch_ex(f, grid(P.pre_large[P.n_active[r]]), (unsigned)v.nt, shmem, s_large,
                           (const void*)P.d_large.p, (const int*)P.d_pre_large.p, P.n_active[r], (int)r, (int)P.k,
                           tbl);
        if (rc) return rc;
    }
    return SE_OK;
}

void finish_plan(Plan& P) {
    for (auto& it : P.small) se_rt::sleep_reset(it.first);
    for (auto& it : P.large) se_rt::sleep_reset(it.first);
    for (auto& it : P.small) {
        it.first->frame += (int32_t)it.second;
        it.first->cur ^= 1;
    }
    for (auto& it : P.large) {
        uint32_t rounds = (it.second + P.k - 1) / P.k;
        it.first->frame += (int32_t)it.second;
        it.first->cur ^= (int)(rounds & 1);
    }
}

// ---------------------------------------------------------------- sliced plans
// The worlds of a rule set whose list is `single` (each fits one 2x2 tile with its
// border) or not, longest first: packed once, advanced in launches of up to k steps
// over the worlds that have steps left, unpacked once.  Worlds that start at the
// same frame -- all of them in the usual batch -- form a group that shares hash
// planes, made for the group's largest extents.  They are made a chunk of frames at a
// time on a stream of their own, while the steps of the chunk before run (which
// leave most of the device idle when the worlds are few): two sets of planes a plan,
// and events both ways.  A chunk's end costs some 10 us of waiting on events, and
// nothing runs beside the first chunk's planes: chunks start at 64 frames and double.
// Worlds inside one tile have small planes, made for the whole run where they fit.
// Bound by vector instructions, about half of them the planes' (no two frames of small
// worlds share a plane), at the occupancy that a few hundred tiles give.  48 worlds of
// 64 to 1024 cells a side, two rule sets, 100 to 1000 steps each: 5.6 to 6.3 ms a run with the LDS
// kernels, 1.9 ms so; 2.0 to 2.1 with the one-tile worlds last, or queued behind planes.
constexpr size_t kBatchHashBudget = 256u << 20, kBatchHashMost = 1024u << 20;
constexpr uint32_t kBatchChunk = 64, kBatchChunkMost = 256;  // frames

struct SlicedPlan {
    se_module* mod = nullptr;
    std::vector<std::pair<se_world*, uint32_t>> list;
    se_rt::SlicedShape shape;  // kernel, side, halo and depth of every world's tiles
    std::vector<se_rt::SlicedWorld> recs;
    std::vector<int> tiles, packs;                // prefix sums over the list
    std::vector<se_rt::SlicedGrid> groups;        // [chunk][group]: hash fields
    std::vector<int> words;                       // [chunk]: prefix sums over its groups, in 256 hash words
    size_t n_groups = 0, hash_bytes = 0, packed_bytes = 0, meta_bytes = 0;
    struct Launch {
        uint32_t done, k;
        int n, from;
    };
    std::vector<std::vector<Launch>> chunks;
    char* base = nullptr;  // device: records, prefix sums, groups, packed grids, hash planes

    size_t off_tiles() const { return (recs.size() * sizeof(se_rt::SlicedWorld) + 255) & ~(size_t)255; }
    size_t off_packs() const { return off_tiles() + ((tiles.size() * sizeof(int) + 255) & ~(size_t)255); }
    size_t off_groups() const { return off_packs() + ((packs.size() * sizeof(int) + 255) & ~(size_t)255); }
    size_t off_words() const { return off_groups() + ((groups.size() * sizeof(se_rt::SlicedGrid) + 255) & ~(size_t)255); }
};

// Everything but the addresses.  squares: of the whole batch (sliced_choice).  False when the hash planes would take too much
// memory (many worlds at different frames).
bool make_sliced(SlicedPlan& P, bool single, uint32_t k, size_t squares) {
    const se_rt::SlicedKernels& K = P.mod->sliced;
    std::stable_sort(P.list.begin(), P.list.end(),
                     [](const std::pair<se_world*, uint32_t>& a, const std::pair<se_world*, uint32_t>& b) {
                         return a.second > b.second;
                     });
    int kernel = 0;
    uint32_t deep = 1u << 20;
    if (!single) {
        se_rt::sliced_choice(squares, K, &kernel, &deep);
        if (k) deep = std::min(k, 32u);
    }
    std::map<int32_t, size_t> at;  // first frame -> group
    std::vector<se_rt::SlicedGrid> extent;  // per group: pads, largest extents
    std::vector<uint32_t> steps;
    std::vector<int> frame;
    P.tiles.assign(1, 0);
    P.packs.assign(1, 0);
    for (auto& it : P.list) {
        se_world* w = it.first;
        const se_rt::SlicedShape s = single ? se_rt::sliced_one_tile(w->W, w->H, false)
                                            : se_rt::sliced_tiles(w->W, w->H, kernel, deep);
        P.shape = s;
        se_rt::SlicedWorld r;
        se_rt::sliced_geometry(s, w->W, w->H, r.g);
        r.g.in = w->buf[w->cur];
        r.g.out = w->buf[w->cur ^ 1];
        r.g.pitch = (int)w->pitch;
        r.frame0 = w->frame + 1;
        r.steps = (int)it.second;
        r.tiles_x = s.tiles_x;
        r.side = s.side;
        r.halo = s.halo;
        auto found = at.find(r.frame0);
        if (found == at.end()) {
            found = at.emplace(r.frame0, extent.size()).first;
            extent.push_back(r.g);
            steps.push_back(0);
            frame.push_back(r.frame0);
        }
        r.group = (int)found->second;
        se_rt::SlicedGrid& e = extent[found->second];
        e.bcols = std::max(e.bcols, r.g.bcols);
        e.brows = std::max(e.brows, r.g.brows);
        steps[found->second] = std::max(steps[found->second], it.second);
        P.tiles.push_back(P.tiles.back() + s.tiles_x * s.tiles_y);
        P.packs.push_back(P.packs.back() + se_rt::sliced_pack_tiles(r.g));
        P.packed_bytes += 2 * se_rt::sliced_packed_bytes(r.g);
        P.recs.push_back(r);
    }
    // the first launch ends at the head of a cycle where all worlds start in one phase
    bool in_phase = true;
    for (auto& r : P.recs) in_phase = in_phase && ((r.frame0 ^ P.recs[0].frame0) & 3) == 0;
    const uint32_t most = P.list[0].second;
    uint32_t first = std::min(deep, most);
    const uint32_t lead = (uint32_t)(P.recs[0].frame0 + (int)first) & 3u;
    if (in_phase && !single && first < most && lead < first) first -= lead;
    // Frames hashed at a time (a chunk): all of them within the budget, else fewer, at
    // least one launch's.  Each group's planes lie where its largest chunk has room.
    P.n_groups = extent.size();
    const uint32_t least = std::min(single ? 32u : deep, most);
    for (uint32_t ahead = single ? std::min(most, se_rt::kSlicedMostFrames) : std::max(1u, kBatchChunkMost / deep) * deep;;) {
        uint32_t length = std::min(ahead, single ? ahead : std::max(1u, kBatchChunk / deep) * deep);
        P.groups.clear();
        P.words.clear();
        P.chunks.clear();
        std::vector<size_t> need(P.n_groups, 0), offset(P.n_groups, 0);
        int from = 0;
        for (uint32_t done = 0; done < most;) {
            const uint32_t stop = std::min(most, done + length);
            length = std::min(ahead, 2 * length);
            P.words.push_back(0);
            for (size_t i = 0; i < P.n_groups; i++) {
                se_rt::SlicedGrid g = extent[i];
                if (done < steps[i])
                    need[i] = std::max(need[i], se_rt::sliced_hash_layout(g, frame[i] + (int)done,
                                                                          std::min(stop, steps[i]) - done, K.classes));
                P.groups.push_back(g);
                P.words.push_back(P.words.back() + (int)(((size_t)g.hash_words * g.hash_sets + 255) / 256));
            }
            P.chunks.emplace_back();
            while (done < stop) {
                const uint32_t m = std::min(done == 0 ? first : deep, stop - done);
                int n = 0;
                while (n < (int)P.recs.size() && P.recs[n].steps > (int)done) P.recs[n++].result ^= 1;
                P.chunks.back().push_back({done, m, n, from});
                from ^= 1;
                done += m;
            }
        }
        size_t set = 0;
        for (size_t i = 0; i < P.n_groups; i++) {
            offset[i] = set;
            set += (need[i] + 255) & ~(size_t)255;
        }
        P.hash_bytes = P.chunks.size() > 1 ? 2 * set : set;
        for (size_t j = 0; j < P.groups.size(); j++)  // offsets until the arena is known
            P.groups[j].hash = (uint32_t*)(offset[j % P.n_groups] + (j / P.n_groups & 1) * set);
        if (P.hash_bytes <= (single ? kBatchHashBudget / 4 : kBatchHashBudget) || ahead <= least) break;
        ahead = std::max(least, ahead / 2);
        if (!single) ahead = std::max(1u, ahead / deep) * deep;
        for (auto& r : P.recs) r.result = 0;
    }
    P.meta_bytes = P.off_words() + ((P.words.size() * sizeof(int) + 255) & ~(size_t)255);
    return P.hash_bytes <= kBatchHashMost;
}

// Device addresses from `base` on, and the records there.
int place_sliced(SlicedPlan& P, char* base) {
    P.base = base;
    char* p = base + P.meta_bytes;
    for (auto& r : P.recs) {
        const size_t bytes = se_rt::sliced_packed_bytes(r.g);
        r.g.pk0 = p;
        r.g.pk1 = p + bytes;
        p += 2 * bytes;
    }
    for (auto& g : P.groups) g.hash = (uint32_t*)(p + (size_t)g.hash);
    std::vector<char> meta(P.meta_bytes);
    std::memcpy(meta.data(), P.recs.data(), P.recs.size() * sizeof(P.recs[0]));
    std::memcpy(meta.data() + P.off_tiles(), P.tiles.data(), P.tiles.size() * sizeof(int));
    std::memcpy(meta.data() + P.off_packs(), P.packs.data(), P.packs.size() * sizeof(int));
    std::memcpy(meta.data() + P.off_groups(), P.groups.data(), P.groups.size() * sizeof(P.groups[0]));
    std::memcpy(meta.data() + P.off_words(), P.words.data(), P.words.size() * sizeof(int));
    HIPCHECK(hipMemcpy(base, meta.data(), meta.size(), hipMemcpyHostToDevice));
    return SE_OK;
}

int sliced_pack(SlicedPlan& P, hipStream_t s) {
    return launch_ex(P.mod->sliced.bpack, (unsigned)(P.packs.back() + 3) / 4, 256, 0u, s, (const void*)P.base,
                     (const int*)(P.base + P.off_packs()), (int)P.recs.size());
}
int sliced_unpack(SlicedPlan& P, hipStream_t s) {
    return launch_ex(P.mod->sliced.bunpack, (unsigned)(P.packs.back() + 3) / 4, 256, 0u, s, (const void*)P.base,
                     (const int*)(P.base + P.off_packs()), (int)P.recs.size());
}

// Chunk c: its planes on hs, then its steps on s.  events: two per chunk, planes made
// and steps done.
int sliced_chunk(SlicedPlan& P, size_t c, hipStream_t s, hipStream_t hs, const std::vector<hipEvent_t>& events) {
    const se_rt::SlicedGrid* g = (const se_rt::SlicedGrid*)(P.base + P.off_groups()) + c * P.n_groups;
    const size_t row = c * (P.n_groups + 1);
    if (c >= 2) HIPCHECK(hipStreamWaitEvent(hs, events[2 * (c - 2) + 1], 0));  // the set's planes have been read
    int rc = launch_ex(P.mod->sliced.bhash, (unsigned)P.words[row + P.n_groups], 256, 0u, hs, (const void*)g,
                       (const int*)(P.base + P.off_words()) + row, (int)P.n_groups);
    if (rc) return rc;
    HIPCHECK(hipEventRecord(events[2 * c], hs));
    HIPCHECK(hipStreamWaitEvent(s, events[2 * c], 0));
    for (auto& l : P.chunks[c]) {
        rc = launch_ex(P.mod->sliced.step[P.shape.kernel], (unsigned)P.tiles[l.n], P.shape.threads, 0u, s,
                       se_rt::SlicedWorld(), (const void*)P.base, (const int*)(P.base + P.off_tiles()), l.n,
                       (const void*)g, l.from, (int)l.done, (int)l.k);
        if (rc) return rc;
    }
    HIPCHECK(hipEventRecord(events[2 * c + 1], s));
    return SE_OK;
}

void finish_sliced(SlicedPlan& P) {
    for (auto& it : P.list) {
        se_rt::sleep_reset(it.first);
        it.first->frame += (int32_t)it.second;
        it.first->cur ^= 1;
    }
}

int ensure_streams(se_batch* b, int n) {
    for (int i = 0; i < n && i < 8; i++)
        if (!b->streams[i]) HIPCHECK(hipStreamCreateWithFlags(&b->streams[i], hipStreamNonBlocking));
    return SE_OK;
}

// Runs the batch: plans are built for every rule-set group, then all launches
// are submitted (optionally through a hipGraph) between two events.
// launch: 0 one workgroup per item, 1 persistent, -1 the tuned choice (else one per item)
int run_batched(se_batch* b, const std::vector<std::pair<se_world*, uint32_t>>& work, int32_t variant, uint32_t k,
                int launch, int graph, float* gpu_ms) {
    se_ctx* ctx = b->ctx;
    std::map<se_module*, std::vector<std::pair<se_world*, uint32_t>>> groups;
    for (auto& it : work) groups[it.first->mod.get()].push_back(it);
    struct Release {  // after the streams are drained: the arena may be given back again
        se_batch* b;
        ~Release() {
            std::lock_guard<std::mutex> lk(b->pool->mu);
            b->arena.busy = false;
        }
    } release{b};
    std::vector<std::unique_ptr<Plan>> plans;
    std::vector<std::unique_ptr<SlicedPlan>> sliced;
    size_t squares = 0;  // of the whole batch: its lists run side by side
    for (auto& it : work)
        if (it.second) squares += se_rt::sliced_squares(it.first->W, it.first->H);
    for (auto& g : groups) {
        se_module* mod = g.first;
        int vi = variant;
        uint32_t kk = k;
        int la = launch;
        auto t = b->tuned.find(mod);
        bool chosen = vi >= 0;
        if (vi < 0) {
            if (t != b->tuned.end()) {
                vi = t->second.vi;
                chosen = true;
                if (kk == 0) kk = t->second.k;
            } else {
                vi = se_rt::default_lds_index(mod);
            }
        }
        if (la < 0) la = t != b->tuned.end() ? (int)t->second.persistent : 0;
        if (vi < 0 || vi >= (int)mod->lds.size()) return fail(SE_ERR_ARG, "LDS variant out of range");
        uint32_t most = 0;
        for (auto& it : g.second) most = std::max(most, it.second);
        bool want = mod->lds[vi].first.sliced;
        if (!want && !chosen && la != 1 && mod->sliced.ok && most >= se_rt::sliced_least_steps(mod->sliced)) {
            std::vector<se_rt::SlicedLoad> loads;
            loads.reserve(g.second.size());
            for (auto& it : g.second) loads.push_back({it.first->W, it.first->H, it.second, it.first->frame});
            want = se_rt::sliced_batch_pays(mod->sliced, loads);
        }
        if (want && most > 0) {
            std::unique_ptr<SlicedPlan> one(new SlicedPlan()), many(new SlicedPlan());
            one->mod = many->mod = mod;
            for (auto& it : g.second)
                if (it.second)
                    (se_rt::sliced_one_tile(it.first->W, it.first->H, false).nw ? one : many)->list.push_back(it);
            if ((one->list.empty() || make_sliced(*one, true, kk, squares)) && (many->list.empty() || make_sliced(*many, false, kk, squares))) {
                if (!many->list.empty()) sliced.push_back(std::move(many));
                if (!one->list.empty()) sliced.push_back(std::move(one));
                continue;
            }
        }
        if (mod->lds[vi].first.sliced) vi = se_rt::default_lds_index(mod);
        plans.emplace_back(new Plan());
        plans.back()->persistent = la == 1;
        int rc = make_plan(ctx, mod, vi, kk, g.second, *plans.back());
        if (rc) return rc;
    }
    if (!sliced.empty()) {
        size_t bytes = 0;
        for (auto& p : sliced) bytes += p->meta_bytes + p->packed_bytes + p->hash_bytes;
        {
            std::lock_guard<std::mutex> lk(b->pool->mu);
            if (bytes > b->arena.bytes) {
                bytes += bytes / 8;  // worlds that drift apart in frames take a little more each run
                se_rt::Pool::drop(b->arena);
                if (hipMalloc(&b->arena.mem, bytes) != hipSuccess) {
                    (void)hipGetLastError();
                    b->arena.mem = nullptr;
                } else {
                    b->arena.bytes = bytes;
                }
            }
            b->arena.busy = b->arena.mem != nullptr;
        }
        if (b->arena.mem) {
            char* p = (char*)b->arena.mem;
            for (auto& q : sliced) {
                int rc = place_sliced(*q, p);
                if (rc) return rc;
                p += q->meta_bytes + q->packed_bytes + q->hash_bytes;
            }
        } else {  // no memory for them: the LDS kernels
            std::map<se_module*, std::vector<std::pair<se_world*, uint32_t>>> back;
            for (auto& q : sliced) back[q->mod].insert(back[q->mod].end(), q->list.begin(), q->list.end());
            sliced.clear();
            for (auto& g : back) {
                plans.emplace_back(new Plan());
                int rc = make_plan(ctx, g.first, se_rt::default_lds_index(g.first), 0, g.second, *plans.back());
                if (rc) return rc;
            }
        }
    }
    // Sliced plans: worlds beyond one tile on a stream per plan, two at most, the longest
    // chain first; their hash planes on the context's stream, idle until the joins; and all
    // worlds inside one tile, a few long launches with planes of their own, on a third
    // stream ahead of everything.
    std::vector<int> lane(sliced.size());
    {
        auto chain = [](const SlicedPlan& p) { return (double)p.list[0].second * p.mod->sliced.planes; };
        std::stable_sort(sliced.begin(), sliced.end(),
                         [&](const std::unique_ptr<SlicedPlan>& x, const std::unique_ptr<SlicedPlan>& y) {
                             return chain(*x) > chain(*y);
                         });
        double sum[2] = {0, 0};
        for (size_t i = 0; i < sliced.size(); i++) {
            lane[i] = !sliced[i]->shape.halo ? 2 : sum[0] <= sum[1] ? 0 : 1;
            if (lane[i] < 2) sum[lane[i]] += chain(*sliced[i]);
        }
    }
    const size_t n_streams = 2 * plans.size() + (sliced.empty() ? 0 : 3);
    // A stream more only for a graph beside sliced plans: a process has four hardware queues,
    // which its streams take in the order of their creation, idle ones too (48 worlds of 64 to
    // 1024 a side, several such batches alive: 1.92 ms a run, 2.08 with an idle stream each)
    int rc = ensure_streams(b, (int)n_streams + (graph && !plans.empty() && !sliced.empty() ? 1 : 0));
    if (rc) return rc;
    RunResources res;  // declared after `plans`: destroyed (and the stream drained) first
    res.streams.assign(b->streams, b->streams + 8);
    res.streams.push_back(ctx->stream);
    hipEvent_t e0, e1, fork;
    std::vector<hipEvent_t> joins(n_streams);
    rc = res.event(&e0, hipEventDefault);
    if (!rc) rc = res.event(&e1, hipEventDefault);
    if (!rc) rc = res.event(&fork, hipEventDisableTiming);
    for (auto& j : joins)
        if (!rc) rc = res.event(&j, hipEventDisableTiming);
    std::vector<std::vector<hipEvent_t>> chunk_events(sliced.size());
    for (size_t i = 0; i < sliced.size(); i++) {
        chunk_events[i].resize(2 * sliced[i]->chunks.size());
        for (auto& e : chunk_events[i])
            if (!rc) rc = res.event(&e, hipEventDisableTiming);
    }
    if (rc) return rc;
    auto submit_plans = [&]() -> int {  // forks from the context's stream and joins it
        HIPCHECK(hipEventRecord(fork, ctx->stream));
        for (size_t i = 0; i < plans.size(); i++) {
            hipStream_t sa = b->streams[(2 * i) % 8], sb = b->streams[(2 * i + 1) % 8];
            HIPCHECK(hipStreamWaitEvent(sa, fork, 0));
            HIPCHECK(hipStreamWaitEvent(sb, fork, 0));
            int r2 = enqueue_plan(*plans[i], sa, sb);
            if (r2) return r2;
            HIPCHECK(hipEventRecord(joins[2 * i], sa));
            HIPCHECK(hipEventRecord(joins[2 * i + 1], sb));
        }
        return SE_OK;
    };
    auto submit_sliced = [&](hipEvent_t begin) -> int {
        if (!sliced.empty()) {
            hipStream_t st[3];
            for (int i = 0; i < 3; i++) {
                st[i] = b->streams[(2 * plans.size() + i) % 8];
                HIPCHECK(hipStreamWaitEvent(st[i], begin, 0));
            }
            for (size_t i = 0; i < sliced.size(); i++) {
                if (lane[i] < 2) continue;
                int r2 = sliced_pack(*sliced[i], st[2]);
                for (size_t c = 0; !r2 && c < sliced[i]->chunks.size(); c++)
                    r2 = sliced_chunk(*sliced[i], c, st[2], st[2], chunk_events[i]);
                if (!r2) r2 = sliced_unpack(*sliced[i], st[2]);
                if (r2) return r2;
            }
            // the others two at a time, chunk by chunk
            for (size_t next[2] = {0, 0};;) {
                int at[2] = {-1, -1};
                size_t chunks = 0;
                for (int l = 0; l < 2; l++) {
                    while (next[l] < sliced.size() && lane[next[l]] != l) next[l]++;
                    if (next[l] == sliced.size()) continue;
                    at[l] = (int)next[l]++;
                    int r2 = sliced_pack(*sliced[at[l]], st[l]);
                    if (r2) return r2;
                    chunks = std::max(chunks, sliced[at[l]]->chunks.size());
                }
                if (at[0] < 0 && at[1] < 0) break;
                for (size_t c = 0; c < chunks; c++)
                    for (int l = 0; l < 2; l++) {
                        if (at[l] < 0 || c >= sliced[at[l]]->chunks.size()) continue;
                        int r2 = sliced_chunk(*sliced[at[l]], c, st[l], ctx->stream, chunk_events[at[l]]);
                        if (r2) return r2;
                    }
                for (int l = 0; l < 2; l++) {
                    int r2 = at[l] < 0 ? SE_OK : sliced_unpack(*sliced[at[l]], st[l]);
                    if (r2) return r2;
                }
            }
            for (int i = 0; i < 3; i++) HIPCHECK(hipEventRecord(joins[2 * plans.size() + i], st[i]));
        }
        return SE_OK;
    };
    auto join = [&](size_t from, size_t to) -> int {
        for (size_t i = from; i < to; i++) HIPCHECK(hipStreamWaitEvent(ctx->stream, joins[i], 0));
        return SE_OK;
    };
    // A graph holds the LDS plans' launches, hundreds in their rounds.  Sliced plans make some
    // forty and are submitted directly, beside the graph: a run that captured them ended in
    // a host abort ("free(): invalid next size") under one HIP runtime, whose cause was not
    // found.
    const size_t n_plan_joins = 2 * plans.size();
    hipStream_t beside = nullptr;  // of the graph, where sliced plans run too
    hipEvent_t begin = nullptr, end = nullptr;
    if (graph && !plans.empty()) {
        HIPCHECK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        int r2 = submit_plans();
        if (!r2) r2 = join(0, n_plan_joins);
        hipError_t ce = hipStreamEndCapture(ctx->stream, &res.graph);
        if (r2) return r2;
        if (ce != hipSuccess) return fail(SE_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(ce));
        HIPCHECK(hipGraphInstantiate(&res.exec, res.graph, nullptr, nullptr, 0));
        if (!sliced.empty()) {
            beside = b->streams[(n_plan_joins + 3) % 8];
            rc = res.event(&begin, hipEventDisableTiming);
            if (!rc) rc = res.event(&end, hipEventDisableTiming);
            if (rc) return rc;
        }
    }
    HIPCHECK(hipEventRecord(e0, ctx->stream));
    if (beside) {
        HIPCHECK(hipEventRecord(begin, ctx->stream));
        HIPCHECK(hipStreamWaitEvent(beside, begin, 0));
        HIPCHECK(hipGraphLaunch(res.exec, beside));
        HIPCHECK(hipEventRecord(end, beside));
        rc = submit_sliced(begin);
        if (!rc) rc = join(n_plan_joins, joins.size());
        if (rc) return rc;
        HIPCHECK(hipStreamWaitEvent(ctx->stream, end, 0));
    } else if (res.exec) {
        HIPCHECK(hipGraphLaunch(res.exec, ctx->stream));
    } else {
        rc = submit_plans();
        if (!rc) rc = submit_sliced(fork);
        if (!rc) rc = join(0, joins.size());
        if (rc) return rc;
    }
    HIPCHECK(hipEventRecord(e1, ctx->stream));
    HIPCHECK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
    for (auto& p : plans) finish_plan(*p);
    for (auto& p : sliced) finish_sliced(*p);
    if (gpu_ms) *gpu_ms = ms;
    return SE_OK;
}

// Worlds whose next step is the clearing frame, or that carry queued
// modifications, take that one step with the plain kernel first.
int pre_steps(std::vector<std::pair<se_world*, uint32_t>>& work) {
    for (auto& it : work) {
        se_world* w = it.first;
        if (it.second == 0) continue;
        if (w->frame + 1 == 1 || !w->pending.empty()) {
            int rc = se_rt::plain_step(w);
            if (rc) return rc;
            it.second--;
        }
    }
    return SE_OK;
}

}  // namespace

extern "C" {

int se_batch_create(se_ctx* ctx, se_batch** out) {
    if (!ctx || !out) return fail(SE_ERR_ARG, "null argument");
    auto* b = new se_batch();
    b->ctx = ctx;
    {
        std::lock_guard<std::mutex> lk(ctx->pool->mu);
        ctx->pool->arenas.push_back(&b->arena);
    }
    b->pool = ctx->pool;
    *out = b;
    return SE_OK;
}

void se_batch_destroy(se_batch* b) {
    if (!b) return;
    DeviceGuard dg(b->pool->device);
    delete b;
}

int se_batch_add(se_batch* b, se_world* w, uint32_t nsteps) {
    if (!b || !w) return fail(SE_ERR_ARG, "null argument");
    if (w->ctx != b->ctx) return fail(SE_ERR_ARG, "world belongs to another context");
    if ((int64_t)w->frame + nsteps > INT32_MAX) return fail(SE_ERR_ARG, "frame counter would overflow");
    if (w->color) return fail(SE_ERR_STATE, "a world with render outputs steps alone (one step per launch)");
    for (auto& it : b->items)
        if (it.first == w) return fail(SE_ERR_ARG, "world already in the batch");
    b->items.push_back({w, nsteps});
    return SE_OK;
}

int se_batch_clear(se_batch* b) {
    if (!b) return fail(SE_ERR_ARG, "null batch");
    b->items.clear();
    DeviceGuard dg(b->pool->device);
    std::lock_guard<std::mutex> lk(b->pool->mu);
    se_rt::Pool::drop(b->arena);
    return SE_OK;
}

int se_batch_run(se_batch* b, int mode, int32_t lds_variant, uint32_t k, int graph, float* gpu_ms) {
    if (!b) return fail(SE_ERR_ARG, "null batch");
    DeviceGuard dg(b->ctx->device);
    std::vector<std::pair<se_world*, uint32_t>> work = b->items;
    // every run advances the worlds again: the frame check of se_batch_add holds
    // for the first run only
    for (auto& it : work)
        if ((int64_t)it.first->frame + it.second > INT32_MAX)
            return fail(SE_ERR_ARG, "frame counter would overflow for a world of the batch");
    if (mode == 0) {  // loop the plain kernel world by world, one launch per step
        RunResources res;
        hipEvent_t e0, e1;
        int rc = res.event(&e0, hipEventDefault);
        if (!rc) rc = res.event(&e1, hipEventDefault);
        if (rc) return rc;
        HIPCHECK(hipEventRecord(e0, b->ctx->stream));
        for (auto& it : work)
            for (uint32_t s = 0; s < it.second; s++) {
                rc = se_rt::plain_step(it.first);
                if (rc) return rc;
            }
        HIPCHECK(hipEventRecord(e1, b->ctx->stream));
        HIPCHECK(hipEventSynchronize(e1));
        float ms = 0;
        HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
        if (gpu_ms) *gpu_ms = ms;
        return SE_OK;
    }
    if (mode < 1 || mode > 3)
        return fail(SE_ERR_ARG, "mode must be 0 (looped plain), 1 (batched, tuned launch), 2 (batched, one "
                                "workgroup per item) or 3 (batched, persistent)");
    int rc = pre_steps(work);
    if (rc) return rc;
    HIPCHECK(hipStreamSynchronize(b->ctx->stream));
    return run_batched(b, work, lds_variant, k, mode == 1 ? -1 : mode - 2, graph, gpu_ms);
}

int se_batch_tuned(const se_batch* b, const se_ruleset* rs, int32_t* variant, uint32_t* k, int32_t* persistent) {
    if (!b || !rs) return fail(SE_ERR_ARG, "null argument");
    auto it = b->tuned.find(rs->mod.get());
    if (it == b->tuned.end()) return fail(SE_ERR_STATE, "this rule set's group has not been tuned");
    if (variant) *variant = it->second.vi;
    if (k) *k = it->second.k;
    if (persistent) *persistent = it->second.persistent ? 1 : 0;
    return SE_OK;
}

int se_batch_autotune(se_batch* b, uint32_t rounds, int32_t* best_variant, uint32_t* best_k,
                      int32_t* best_persistent, float* best_ns_per_kcell) {
    if (!b || rounds == 0) return fail(SE_ERR_ARG, "bad arguments");
    DeviceGuard dg(b->ctx->device);
    int rc = SE_OK;
    // trial runs must leave the worlds untouched: worlds whose next step needs
    // the plain kernel (clearing frame, queued modifications) sit out
    std::map<se_module*, std::vector<std::pair<se_world*, uint32_t>>> groups;
    for (auto& it : b->items)
        if (it.second > 0 && it.first->frame + 1 != 1 && it.first->pending.empty())
            groups[it.first->mod.get()].push_back(it);
    for (auto& g : groups) {
        se_module* mod = g.first;
        // snapshot the group's grids and frames
        std::vector<std::pair<void*, size_t>> snaps;
        std::vector<std::pair<int32_t, int>> state;
        for (auto& it : g.second) {
            se_world* w = it.first;
            size_t bytes = (size_t)w->pitch * w->H * 4;
            void* p = nullptr;
            if (se_rt::device_alloc(b->ctx->device, &p, bytes) != hipSuccess) {
                for (auto& s : snaps) (void)hipFree(s.first);
                return fail(SE_ERR_OOM, "autotune snapshot allocation failed");
            }
            HIPCHECK(hipMemcpyAsync(p, w->buf[w->cur], bytes, hipMemcpyDeviceToDevice, b->ctx->stream));
            snaps.push_back({p, bytes});
            state.push_back({w->frame, w->cur});
        }
        HIPCHECK(hipStreamSynchronize(b->ctx->stream));
        double best = 1e300;
        int bv = 0;
        uint32_t bk = 0;
        bool bp = false;
        for (int vi = 0; vi < (int)mod->lds.size(); vi++) {
            const int hb = mod->lds[vi].first.hb;
            for (uint32_t kk : {(uint32_t)hb, (uint32_t)std::max(2, hb / 2)})
            for (int la = 0; la < (mod->lds[vi].first.sliced ? 1 : 2); la++) {
                std::vector<std::pair<se_world*, uint32_t>> trial;
                double cells = 0;
                for (auto& it : g.second) {
                    uint32_t st = std::min<uint32_t>(it.second, rounds * kk);
                    trial.push_back({it.first, st});
                    cells += (double)it.first->W * it.first->H * st;
                }
                float ms = 0;
                rc = run_batched(b, trial, vi, kk, la, 0, &ms);
                // restore
                for (size_t i = 0; i < g.second.size(); i++) {
                    se_world* w = g.second[i].first;
                    w->frame = state[i].first;
                    w->cur = state[i].second;
                    HIPCHECK(hipMemcpyAsync(w->buf[w->cur], snaps[i].first, snaps[i].second,
                                            hipMemcpyDeviceToDevice, b->ctx->stream));
                }
                HIPCHECK(hipStreamSynchronize(b->ctx->stream));
                if (rc) {
                    for (auto& s : snaps) (void)hipFree(s.first);
                    return rc;
                }
                double score = cells > 0 ? ms * 1e6 / (cells / 1e3) : 0;  // ns per 1000 cell-updates
                if (score < best) {
                    best = score;
                    bv = vi;
                    bk = kk;
                    bp = la == 1;
                }
            }
        }
        for (auto& s : snaps) (void)hipFree(s.first);
        b->tuned[mod] = {bv, bk, bp};
        if (best_variant) *best_variant = bv;
        if (best_k) *best_k = bk;
        if (best_persistent) *best_persistent = bp ? 1 : 0;
        if (best_ns_per_kcell) *best_ns_per_kcell = (float)best;
    }
    return SE_OK;
}

}  // extern "C"
