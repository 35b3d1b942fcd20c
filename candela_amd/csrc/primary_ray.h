// Primary ray of pixel (x, y) as in TraverseBVHStackless.glsl:371-378
// (uv = pixel / dims, GetRayDirectionAt of :143-148, normalize).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "device_math.h"
#include "trace_launch.h"

#pragma clang fp contract(off)

namespace crt {
namespace dm {

__device__ __forceinline__ crt_ray primary_ray(const Camera& cam, int32_t width, int32_t height, int32_t x, int32_t y,
                                               uint32_t id) {
    const float u = float(x) / float(width), v = float(y) / float(height);
    const float cx = u * 2.0f - 1.0f, cy = v * 2.0f - 1.0f;
    const float* ip = cam.inv_proj;
    const float ex = ip[0] * cx + ip[4] * cy + ip[8] * -1.0f + ip[12] * 1.0f;
    const float ey = ip[1] * cx + ip[5] * cy + ip[9] * -1.0f + ip[13] * 1.0f;
    const f3 d = xform(cam.inv_view, mk(ex, ey, -1.0f), 0.0f);
    const float il = 1.0f / sqrtf(dot(d, d));
    crt_ray r;
    r.org[0] = cam.inv_view[12];
    r.org[1] = cam.inv_view[13];
    r.org[2] = cam.inv_view[14];
    r.tmax = cam.tmax;
    r.dir[0] = d.x * il;
    r.dir[1] = d.y * il;
    r.dir[2] = d.z * il;
    r.id = id;
    return r;
}

__device__ __forceinline__ void store_ray(crt_ray* out, const crt_ray& r) {
    float4* p = reinterpret_cast<float4*>(out);
    p[0] = make_float4(r.org[0], r.org[1], r.org[2], r.tmax);
    p[1] = make_float4(r.dir[0], r.dir[1], r.dir[2], __uint_as_float(r.id));
}

// Pixel of a workgroup's lane: waves take blocks of pixels, 8 x 8 when full
// (rays_per_wave_log2), and a workgroup 2 x 2 of them; they share more of their
// walk than pixels of one row do.  Images narrower or lower than 8 pixels are
// taken in row order.  Runs of kTileRun workgroups go to one XCD (consecutive
// tiles share nodes in its L2), runs in turn so that cheap and costly bands of
// the image are spread over all eight.
constexpr int32_t kTileRun = 32;

struct ImageTiles {
    int32_t width, height;
    int32_t log2;       // pixels of a wave
    int32_t tiles_x;    // workgroups across; 0: row order
    int64_t blocks;
};

inline ImageTiles image_tiles(int32_t width, int32_t height) {
    ImageTiles t;
    t.width = width;
    t.height = height;
    t.log2 = rays_per_wave_log2(int64_t(width) * height);
    const int32_t w = 2 << ((t.log2 + 1) / 2), h = 2 << (t.log2 / 2);
    t.tiles_x = width >= 8 && height >= 8 ? (width + w - 1) / w : 0;
    t.blocks = t.tiles_x ? int64_t(t.tiles_x) * ((height + h - 1) / h)
                         : ((int64_t(width) * height + (4 << t.log2) - 1) >> (t.log2 + 2));
    return t;
}

// Workgroups to launch: whole rounds of runs.
inline unsigned image_grid(const ImageTiles& t) {
    const int64_t round = 8 * kTileRun;
    return unsigned(t.blocks <= round ? t.blocks : (t.blocks + round - 1) / round * round);
}

struct Pixel {
    int32_t x, y;
    int64_t i;   // -1: none
};

__device__ __forceinline__ Pixel image_pixel(const ImageTiles& t) {
    int64_t b = blockIdx.x;
    if (gridDim.x > 8 * kTileRun) {
        const uint32_t k = blockIdx.x / 8u;
        b = (int64_t(k / kTileRun) * 8 + blockIdx.x % 8u) * kTileRun + k % kTileRun;
    }
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63u;
    Pixel p{0, 0, -1};
    if (l >> t.log2 || b >= t.blocks) return p;
    if (t.tiles_x) {
        const int32_t lx = (t.log2 + 1) / 2, ly = t.log2 / 2;
        const int64_t ty = b / t.tiles_x;
        p.x = (int32_t(b - ty * t.tiles_x) << (lx + 1)) + int32_t(((w & 1u) << lx) + (l & ((1u << lx) - 1u)));
        p.y = (int32_t(ty) << (ly + 1)) + int32_t(((w >> 1) << ly) + (l >> lx));
        if (p.x < t.width && p.y < t.height) p.i = int64_t(p.y) * t.width + p.x;
    } else {
        const int64_t i = ((b * 4 + w) << t.log2) + l;
        if (i >= int64_t(t.width) * t.height) return p;
        p.i = i;
        p.y = int32_t(i / t.width);
        p.x = int32_t(i - int64_t(p.y) * t.width);
    }
    return p;
}

}  // namespace dm
}  // namespace crt
