// Host side of the sliced kernels (se_sliced.hip): geometry of the packed grid
// and the launches that advance one world.
#pragma once
#include <cstdint>

#include "se_internal.hpp"

namespace se_rt {

// == se_slgrid in se_sliced.hip
struct SlicedGrid {
    uint32_t* in = nullptr;
    uint32_t* out = nullptr;
    void* pk0 = nullptr;
    void* pk1 = nullptr;
    uint32_t* hash = nullptr;
    int W = 0, H = 0, pitch = 0;
    int xpad = 0, ypad = 0, bcols = 0, rows = 0;
    int brows = 0;
    int hash_frame0 = 0, hash_shared = 0, hash_sets = 0;
    int hash_pitch = 0, hash_words = 0;
    uint32_t hash_n0 = 0, hash_n1 = 0;
};
static_assert(sizeof(SlicedGrid) == 104, "se_slgrid layout");

// == se_slworld in se_sliced.hip
struct SlicedWorld {
    SlicedGrid g;
    int frame0 = 0, steps = 0, tiles_x = 0, side = 0, halo = 0, group = 0;
    int result = 0;
    uint32_t stable = 0;
    unsigned char* calm = nullptr;
    int calm_cols = 0, pad = 0;
};
static_assert(sizeof(SlicedWorld) == 152, "se_slworld layout");

struct SlicedKnown {  // == se_slknown in se_sliced.hip
    unsigned char *same = nullptr, *was = nullptr, *calm = nullptr;
    int valid = 0;
};

// How a world is cut into tiles of one step kernel.
struct SlicedShape {
    int kernel = 0;            // index into SlicedKernels::step
    int nw = 0, r = 0;         // words of a tile, rows of a lane
    unsigned threads = 0;      // of a workgroup (one tile)
    int side = 0, halo = 0;    // byte columns and rows given up on each side; 0: the world fits one tile
    int tiles_x = 0, tiles_y = 0;
    uint32_t max_sub = 0;      // sub-steps of one launch (any number when the world fits one tile)
};

// The one tile that holds a W x H world with its border, if there is one (nw 0 else):
// the 2x2 tile or, with `wide`, the 4x2 one.
SlicedShape sliced_one_tile(uint32_t W, uint32_t H, bool wide);
// Tiles of step kernel `kernel` for launches of up to max_sub (at most 32) sub-steps.
SlicedShape sliced_tiles(uint32_t W, uint32_t H, int kernel, uint32_t max_sub);
// Step kernel and depth of a launch for worlds of `few` 64 x 64 squares in all.
void sliced_choice(size_t few, const SlicedKernels& K, int* kernel, uint32_t* deep);
// What a run of n steps takes, in launches of up to `sub` (0: the choice).
SlicedShape sliced_shape(const SlicedKernels& K, uint32_t W, uint32_t H, uint32_t n, uint32_t sub);
inline size_t sliced_squares(uint32_t W, uint32_t H) { return (size_t)((W + 63) / 64) * ((H + 63) / 64); }
// Fills the geometry fields of g for that shape.
void sliced_geometry(const SlicedShape& s, uint32_t W, uint32_t H, SlicedGrid& g);
size_t sliced_packed_bytes(const SlicedGrid& g);  // of one packed grid
constexpr uint32_t kSlicedMostFrames = 32768;  // hashed in one launch (a grid's most in y is 65535)
// Sets up the hash planes of frames [frame0, frame0 + nf) in g (all but the pointer):
// the form and its sizes; returns their bytes, with room for the words that the step
// kernel loads ahead.
size_t sliced_hash_layout(SlicedGrid& g, int32_t frame0, uint32_t nf, int classes);

// How a run of n steps of one world hashes its frames: so many at a time, and the bytes
// that the planes of every such chunk fit.
struct SlicedAhead {
    uint32_t frames = 0;
    size_t bytes = 0;
};
SlicedAhead sliced_ahead(const SlicedShape& s, SlicedGrid g, int32_t frame0, uint32_t n, int classes);

// The fewest steps that may leave the LDS kernels.
inline uint32_t sliced_least_steps(const SlicedKernels& K) { return K.cost.form == 0 ? 4 : 9; }
// Is the sliced path taken for n steps of a world whose caller chose no variant?
bool sliced_pays(const SlicedKernels& K, uint32_t W, uint32_t H, uint32_t n);
// And for the worlds of a batch that share the rule set?
struct SlicedLoad {
    uint32_t W, H, n;
    int32_t frame;
};
bool sliced_batch_pays(const SlicedKernels& K, const std::vector<SlicedLoad>& worlds);
// Wavefronts (64 columns x 64 rows each) that pack and that unpack a world.
int sliced_pack_tiles(const SlicedGrid& g);
int sliced_unpack_columns(const SlicedGrid& g);
// Do the modifications of a run's first step go into the packed grid (else that step is
// for the plain kernel)?
bool sliced_takes_mods(const se_world* w, uint32_t n);
// Do the step kernel's tiles sleep (K.sleep_step in place of K.step)?
bool sliced_sleeps(const se_world* w, int kernel);
// Advances w by n steps (no clearing frame among them; queued modifications follow the
// first), launches of up to `sub` sub-steps.  *done = false and nothing enqueued
// when the scratch memory cannot be had.
int sliced_steps(se_world* w, uint32_t n, uint32_t sub, bool* done);

}  // namespace se_rt
