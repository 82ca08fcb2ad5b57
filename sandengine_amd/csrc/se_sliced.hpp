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
    void* pk[2] = {nullptr, nullptr};
    uint32_t* hash = nullptr;
    int W = 0, H = 0, pitch = 0;
    int xpad = 0, ypad = 0, bcols = 0, rows = 0;
    int brows = 0;
    int hash_frame0 = 0, hash_shared = 0;
    int hash_pitch = 0, hash_words = 0;
    uint32_t hash_n0[2] = {0, 0};
};
static_assert(sizeof(SlicedGrid) == 96, "se_slgrid layout");

// How a world is cut into tiles of one step kernel.
struct SlicedShape {
    int kernel = 0;            // index into SlicedKernels::step
    int nw = 0, r = 0;         // words and rows of a lane
    int side = 0, halo = 0;    // byte columns and rows given up on each side; 0: the world fits one tile
    int tiles_x = 0, tiles_y = 0;
    uint32_t max_sub = 0;      // sub-steps of one launch (any number when the world fits one tile)
};

// The tiles for W x H cells in launches of up to `sub` sub-steps (0: no limit but the kernel's).
SlicedShape sliced_shape(uint32_t W, uint32_t H, uint32_t sub);
// Fills the geometry fields of g for that shape.
void sliced_geometry(const SlicedShape& s, uint32_t W, uint32_t H, SlicedGrid& g);
size_t sliced_packed_bytes(const SlicedGrid& g);  // of one packed grid
// Sets up the hash planes of frames [frame0, frame0 + nf) in g (all but the pointer):
// the form and its sizes; returns their bytes, with room for the words that the step
// kernel loads ahead.
size_t sliced_hash_layout(SlicedGrid& g, int32_t frame0, uint32_t nf, int classes);

// Is the sliced path taken for n steps of a world whose caller chose no variant?
bool sliced_pays(const se_world* w, uint32_t n);
// Advances w by n steps (no clearing frame and no queued modifications among
// them), launches of up to `sub` sub-steps.  *done = false and nothing enqueued
// when the scratch memory cannot be had.
int sliced_steps(se_world* w, uint32_t n, uint32_t sub, bool* done);

}  // namespace se_rt
