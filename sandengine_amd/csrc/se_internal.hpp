// Internal types and helpers shared by the runtime translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/sandengine_hip.h"
#include "se_hipgen.hpp"
#include "se_lang.hpp"

namespace se_rt {

// Records the message for se_last_error() and returns `code`.
int fail(int code, const std::string& msg);

#define HIPCHECK(expr)                                                                                 \
    do {                                                                                               \
        hipError_t _e = (expr);                                                                        \
        if (_e != hipSuccess) return se_rt::fail(SE_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

// Launches `f` on a 1-D grid of 256-thread workgroups; each argument is passed
// by address (kernelParams), so its C++ type must match the kernel parameter.
template <typename... A>
int launch(hipFunction_t f, unsigned grid, hipStream_t s, A... args) {
    void* p[] = {(void*)&args...};
    hipError_t e = hipModuleLaunchKernel(f, grid, 1, 1, 256, 1, 1, 0, s, p, nullptr);
    if (e != hipSuccess) return se_rt::fail(SE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
    return SE_OK;
}

template <typename... A>
int launch_ex(hipFunction_t f, unsigned grid, unsigned block, unsigned shmem, hipStream_t s, A... args) {
    void* p[] = {(void*)&args...};
    hipError_t e = hipModuleLaunchKernel(f, grid, 1, 1, block, 1, 1, shmem, s, p, nullptr);
    if (e != hipSuccess) return se_rt::fail(SE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
    return SE_OK;
}

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        hipGetDevice(&prev);
        if (prev != dev) hipSetDevice(dev);
    }
    ~DeviceGuard() {
        int now;
        hipGetDevice(&now);
        if (prev >= 0 && now != prev) hipSetDevice(prev);
    }
};

struct FillSpec {  // == se_fillspec in se_kernels.hip
    int n, stone_rows;
    uint32_t stone_id, pad;
    uint32_t ids[16], thr[16];
};

// Device memory that a context keeps from call to call.  Its worlds hold it too: they may
// outlive the context.
struct Pool {
    struct Block {
        void* mem = nullptr;
        size_t bytes = 0;
        bool busy = false;  // a batch's run is under way
    };
    int device = 0;
    std::mutex mu;
    // packed grids and hash planes of the sliced kernels (se_sliced.cpp), as large as the
    // largest call needed, in use while mu is held and by what that enqueued
    Block scratch;
    int worlds = 0;              // live worlds made by se_world_create
    std::vector<Block*> arenas;  // of the context's batches
    // Frees a block that nothing uses (hipFree waits for the device); mu held.
    static void drop(Block& b) {
        (void)hipFree(b.mem);
        b.mem = nullptr;
        b.bytes = 0;
    }
    ~Pool();
};
// A context's pool, known to device_alloc while it lives.
std::shared_ptr<Pool> make_pool(int device);
// hipMalloc on the current device, `device`; where that fails, once more after the pools of
// all contexts there gave back what is not in use.  The caller holds no pool's mu.
hipError_t device_alloc(int device, void** p, size_t bytes);

// What the choice between a rule set's kernels goes by (se_sliced.cpp).
struct StepCost {
    int form = 0;           // of the LDS kernels: 0 generated chain, 1 full table, 2 coded table
    bool wall_kept = true;  // no block changes a WALL cell
    int tables = 0;         // three-input tables of the sliced form
    int hash_ops = 0;       // instructions that hash a block: 9 a lane, 2 a plane
    bool one_wave = true;   // tiles of one wavefront are there (up to three planes)
};

// The sliced kernels of a module (se_sliced.hip); ok false where the rule set has
// no sliced form.
struct SlicedKernels {
    bool ok = false;
    StepCost cost;
    int planes = 0, classes = 0;  // bit planes of a cell, hash planes of a frame
    uint32_t stable = 0;          // SlicedInfo::stable
    hipFunction_t pack = nullptr, unpack = nullptr, hash = nullptr, brush = nullptr;
    hipFunction_t bpack = nullptr, bunpack = nullptr, bhash = nullptr;  // the worlds of a batch
    hipFunction_t step[4] = {};  // 2x2 and 4x2 tiles by one wavefront (up to three planes), 2x2 by two, 4x2 by four
    hipFunction_t sleep_step[4] = {};  // those of large worlds, whose tiles sleep
};

}  // namespace se_rt

// ------------------------------------------------------------------ internal types
struct se_module {
    hipModule_t mod = nullptr;
    uint32_t* table = nullptr;       // transition table (SE_TBL), device memory
    size_t table_entries = 0;        // 0 when the rule set runs the generated chain
    int table_form = 0;              // 0 generated chain, 1 full table, 2 coded table
    bool wall_kept = false;          // full table: no entry changes a WALL cell
    uint32_t stable_mask = 0;        // bit c: a block of four cells of LDS code c never changes
    std::vector<unsigned> lds_bytes; // dynamic LDS per LDS variant
    std::vector<int> lds_grid;       // resident workgroups per LDS variant at full occupancy (multiple of 8)
    std::vector<int> lds_waves;      // resident wavefronts per CU per LDS variant
    int default_lds = 0;             // LDS variant of se_world_step_blocked when none is set
    int wide_lds = 0;  // of the default's tile and halo, the variant with the most threads
    int cus = 0;
    hipFunction_t plain = nullptr, fill = nullptr, fill_seeded = nullptr, copy = nullptr, fill_spec = nullptr, fill_narrow = nullptr;
    hipFunction_t frame[2] = {};   // se_frame_b1/2: plain step with its colour and light
    hipFunction_t render = nullptr;  // se_render: colour and light alone
    hipFunction_t noise_fill = nullptr;  // se_noise_fill: the colour noise image
    hipFunction_t plain_v[6] = {};  // se_step_plain_r{1,2,4}_nt{0,1}
    std::vector<std::pair<se::LdsVariant, hipFunction_t>> lds;
    std::vector<hipFunction_t> batch;  // se_batch_lds_* parallel to `lds`
    se_rt::SlicedKernels sliced;
    int device = 0;
    ~se_module() {
        if (mod) {
            int prev;
            hipGetDevice(&prev);
            hipSetDevice(device);
            hipFree(table);
            hipModuleUnload(mod);
            hipSetDevice(prev);
        }
    }
};

struct se_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::mutex mu;
    std::map<uint64_t, std::pair<std::string, std::shared_ptr<se_module>>> cache;
    // se_grids_step_noalloc: the device's scratch array, a pinned staging buffer
    // of its size, and the event after the last copy out of that buffer
    void* scratch = nullptr;
    void* staging = nullptr;
    hipEvent_t staging_done = nullptr;
    std::mutex staging_mu;
    std::shared_ptr<se_rt::Pool> pool;
};

struct se_ruleset {
    se_ctx* ctx = nullptr;
    se::ParsingResult pr;
    std::shared_ptr<se_module> mod;
    int nmat = 0;
};

struct se_world {
    se_ctx* ctx = nullptr;
    const se_ruleset* rs = nullptr;
    std::shared_ptr<se_module> mod;
    uint32_t W = 0, H = 0, pitch = 0;
    uint32_t* buf[2] = {nullptr, nullptr};
    int cur = 0;
    int32_t frame = 0;
    std::shared_ptr<se_rt::Pool> pool;  // of the context (worlds from se_world_create)
    std::vector<se_modification> pending;
    void* d_mods = nullptr;
    hipStream_t stream = nullptr;
    bool owns = true;       // buffers from hipMalloc (false: carved from a serving arena)
    int plain_variant = 3;  // index into se_module::plain_v (default: 1 row pair, non-temporal stores)
    int lds_variant = -1;   // index into se_module::lds, -1 = default choice
    // render side-outputs (se_world_set_render): RGBA f32 per cell, row pitch `pitch`
    void* light[2] = {nullptr, nullptr};  // ping-pong: light[lcur] holds the last step's light
    float* noise = nullptr;                // colour noise per cell (position only), filled once
    void* color = nullptr;
    int lcur = 0;
    // tile sleeping of the LDS kernel (se_tile_sleeps): per tile of variant
    // sleep_variant, the settled code in the last launch or 0xff; of the sliced kernels
    // (se_slknown), whose variant is the last: per 64 x 64 square, laid out as
    // sleep_layout says.  Valid only while nothing but those kernels has written either
    // grid buffer (sleep_variant -1 otherwise)
    unsigned char* d_sleep[2] = {nullptr, nullptr};
    size_t sleep_cap = 0;
    int sleep_variant = -1;
    int sleep_layout = 0;
    int sleep_p = 0;
    bool exposed = false;  // the caller has a grid's address and may write through it at any time
    bool sleep_enabled = true;
};


namespace se_rt {
constexpr int kFewMods = 8;  // SE_PLAIN_MODS of the kernel source
struct FewMods {             // == se_few
    se_modification m[kFewMods];
};
struct ModsArg {
    void* ptr;
    int n;
};
// Takes the queued modifications (cut at the first size-0 entry, as the
// kernel's loop stops there, falling_sand.glsl:139-141) and clears the queue: up to
// kFewMods go to `few`, if given, where the kernel takes them by value, more to device
// memory.
int take_mods(se_world* w, ModsArg& m, FewMods* few = nullptr);
// One Simulation::run of `w` with the plain kernel (frame += 1, mods, step).
int plain_step(se_world* w);
// The grids of `w` were written by something other than the LDS kernel: its
// tile-sleeping record no longer describes them.
inline void sleep_reset(se_world* w) { w->sleep_variant = -1; }
// Room for n bytes in each of w->d_sleep.
int sleep_room(se_world* w, size_t n);
// Index of the default LDS tile variant of a module (batches and serving use it
// unless tuned).
int default_lds_index(const se_module* m);
// Enqueues the seeded fill of a grid of w.
int fill_spec(const se_world* w, uint32_t* grid, uint64_t seed, const FillSpec& fs);
// Device address of the no-allocation scratch array on `device` (current).
int noalloc_scratch(int device, void** out);
}  // namespace se_rt
