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

using se_rt::DeviceGuard;
using se_rt::fail;

namespace {

constexpr size_t kHashBudget = 128u << 20;  // hash planes made ahead, unless one launch needs more

struct Tile {
    int nw, r;
};
constexpr Tile kTiles[3] = {{2, 2}, {4, 2}, {4, 4}};  // as instantiated in se_sliced.hip

template <typename... A>
int launch2(hipFunction_t f, unsigned gx, unsigned gy, unsigned block, hipStream_t s, A... args) {
    void* p[] = {(void*)&args...};
    hipError_t e = hipModuleLaunchKernel(f, gx, gy, 1, block, 1, 1, 0, s, p, nullptr);
    if (e != hipSuccess) return fail(SE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
    return SE_OK;
}

}  // namespace

se_rt::SlicedShape se_rt::sliced_shape(uint32_t W, uint32_t H, uint32_t sub) {
    SlicedShape s;
    // A world with its WALL border inside one tile needs no halo: one column and
    // one row more than the world has to the right and below (the wave shifts
    // bring WALL in from the other sides).
    for (int i = 0; i < 2; i++) {
        if (W + 4 > 64u * kTiles[i].nw - 1 || H + 2 > 64u * kTiles[i].r) continue;
        s.kernel = i;
        s.nw = kTiles[i].nw;
        s.r = kTiles[i].r;
        s.tiles_x = s.tiles_y = 1;
        s.max_sub = sub ? sub : 1u << 20;
        return s;
    }
    // The tile and the depth of a launch, by how many 2x2 tiles (64 useful columns and
    // rows at 32 sub-steps) the world makes.  Up to one a SIMD the launches are a
    // serial chain of sub-steps: the smallest tile and the deepest launch
    // (1000x700: 162 us for 200 steps, 249 with 4x2, 178 with 16 sub-steps).  Beyond
    // that the rows given up count, and from 8 a SIMD on the columns too
    // (4096^2, 200 steps: 541 us with 2x2 and 16, 563 with either 4x2 or 32;
    // 16384^2, 100 steps: 3.35 ms with 4x2 and 16, 3.52 with 2x2).
    const size_t few = (size_t)((W + 63) / 64) * ((H + 63) / 64);
    const int i = few > 8192 ? 1 : 0;
    const uint32_t deep = few > 1024 ? 16 : 32;
    s.kernel = i;
    s.nw = kTiles[i].nw;
    s.r = kTiles[i].r;
    s.max_sub = sub ? std::min(sub, deep) : deep;
    s.halo = (int)(s.max_sub + 3) & ~3;
    s.tiles_x = (int)(W + 64 * s.nw - 65) / (64 * s.nw - 64);
    s.tiles_y = (int)(H + 64 * s.r - 2 * s.halo - 1) / (64 * s.r - 2 * s.halo);
    return s;
}

void se_rt::sliced_geometry(const SlicedShape& s, uint32_t W, uint32_t H, SlicedGrid& g) {
    g.W = (int)W;
    g.H = (int)H;
    if (s.halo == 0) {
        g.xpad = 4;  // keeps the 16-byte loads of ids aligned
        g.ypad = 2;
    } else {
        g.xpad = 32;
        g.ypad = s.halo;
    }
    g.hcols = (s.tiles_x - 1) * (2 * s.nw - 2) + 2 * s.nw;
    g.rows = ((s.tiles_y - 1) * (64 * s.r - 2 * s.halo) + 64 * s.r + 63) & ~63;
    g.wcols = g.hcols / 2;
    g.brows = g.rows / 2;
}

size_t se_rt::sliced_packed_bytes(const SlicedGrid& g, int planes) {
    return ((size_t)g.hcols * g.rows * 2 * planes * sizeof(uint16_t) + 255) & ~(size_t)255;
}
size_t se_rt::sliced_frame_bytes(const SlicedGrid& g, int classes) {
    return (size_t)g.wcols * g.brows * classes * sizeof(uint32_t);
}

// Packing, hashing and unpacking cost three launches more than the LDS kernels
// have, and from the largest worlds a pass over the grid: the LDS kernels stay for
// short runs (measured per call, LDS against sliced: 256^2 8 steps 23 and 20 us, 12
// steps 37 and 24; 4096^2 8 steps 46 and 56, 12 steps 82 and 67; 16384^2 16 steps
// 836 and 921, 24 steps 1208 and 1146).
bool se_rt::sliced_pays(const se_world* w, uint32_t n) {
    return w->mod->sliced.ok && n >= ((size_t)w->W * w->H > (64u << 20) ? 24u : 12u);
}

int se_rt::sliced_steps(se_world* w, uint32_t n, uint32_t sub, bool* done) {
    *done = false;
    const SlicedKernels& K = w->mod->sliced;
    const SlicedShape shape = sliced_shape(w->W, w->H, sub);
    SlicedGrid g;
    sliced_geometry(shape, w->W, w->H, g);
    g.pitch = (int)w->pitch;
    const size_t packed = sliced_packed_bytes(g, K.planes), frame = sliced_frame_bytes(g, K.classes);
    const uint32_t per_launch = std::min(shape.max_sub, n);
    // frames hashed at a time: whole launches within the budget
    uint32_t ahead = (uint32_t)std::min<size_t>(n, std::max<size_t>(1, kHashBudget / frame));
    if (shape.halo) ahead = std::min(n, std::max(ahead / per_launch, 1u) * per_launch);
    const size_t bytes = 2 * packed + ahead * frame;

    // The scratch belongs to the context: its worlds share one stream, and the
    // launches of one call are enqueued together under the lock.
    se_ctx* ctx = w->ctx;
    std::lock_guard<std::mutex> lk(ctx->sliced_mu);
    if (bytes > ctx->sliced_bytes) {
        if (ctx->sliced_mem) HIPCHECK(hipFree(ctx->sliced_mem));  // waits for the work that uses it
        ctx->sliced_mem = nullptr;
        ctx->sliced_bytes = 0;
        if (hipMalloc(&ctx->sliced_mem, bytes) != hipSuccess) {
            (void)hipGetLastError();
            ctx->sliced_mem = nullptr;
            return SE_OK;
        }
        ctx->sliced_bytes = bytes;
    }
    *done = true;
    g.in = w->buf[w->cur];
    g.out = w->buf[w->cur ^ 1];
    g.pk[0] = (uint16_t*)ctx->sliced_mem;
    g.pk[1] = (uint16_t*)((char*)ctx->sliced_mem + packed);
    g.hash = (uint32_t*)((char*)ctx->sliced_mem + 2 * packed);

    const int wtiles = g.hcols / 2, ctiles = wtiles * (g.rows / 64);
    int rc = launch2(K.pack, (unsigned)(ctiles + 3) / 4, 1, 256, w->stream, g, wtiles, ctiles);
    int from = 0;
    for (uint32_t at = 0; at < n && !rc;) {
        const uint32_t nf = std::min(ahead, n - at);
        g.hash_frame0 = w->frame + 1 + (int)at;
        rc = launch2(K.hash, (unsigned)(g.brows + 255) / 256, std::min(nf * (uint32_t)g.wcols, 65535u), 256, w->stream,
                     g, (int)nf);
        for (uint32_t d = 0; d < nf && !rc;) {
            const uint32_t m = std::min(shape.max_sub, nf - d);
            rc = launch2(K.step[shape.kernel], (unsigned)(shape.tiles_x * shape.tiles_y), 1, 64, w->stream, g, from,
                         shape.tiles_x, g.hash_frame0 + (int)d, (int)m, shape.halo);
            from ^= 1;
            d += m;
        }
        at += nf;
    }
    if (!rc) rc = launch2(K.unpack, (unsigned)(ctiles + 3) / 4, 1, 256, w->stream, g, from, wtiles, ctiles);
    if (rc) return rc;
    sleep_reset(w);
    w->frame += (int32_t)n;
    w->cur ^= 1;
    return SE_OK;
}
