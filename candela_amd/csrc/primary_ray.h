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

// Pixel of a workgroup's lane: waves take 8 x 8 pixels (a workgroup 16 x 16),
// whose rays share more of their walk than 64 pixels of one row do.  Images
// narrower or lower than a tile are taken in row order.  Runs of kTileRun
// workgroups go to one XCD (consecutive tiles share nodes in its L2), runs in
// turn so that cheap and costly bands of the image are spread over all eight.
constexpr int32_t kTileRun = 32;

struct Pixel {
    int32_t x, y;
    int64_t i;   // -1: none
};

__host__ __device__ inline bool image_tiled(int32_t width, int32_t height) { return width >= 8 && height >= 8; }

inline int64_t image_blocks(int32_t width, int32_t height) {
    return image_tiled(width, height) ? int64_t((width + 15) / 16) * ((height + 15) / 16)
                                      : (int64_t(width) * height + 255) / 256;
}

// Grid of image_blocks(...) workgroups, padded to whole rounds of runs.
inline int64_t image_grid(int64_t blocks) {
    const int64_t round = 8 * kTileRun;
    return blocks <= round ? blocks : (blocks + round - 1) / round * round;
}

__device__ __forceinline__ Pixel image_pixel(int32_t width, int32_t height) {
    int64_t b = blockIdx.x;
    if (gridDim.x > 8 * kTileRun) {
        const uint32_t k = blockIdx.x / 8u;
        b = (int64_t(k / kTileRun) * 8 + blockIdx.x % 8u) * kTileRun + k % kTileRun;
    }
    Pixel p;
    if (image_tiled(width, height)) {
        const int32_t tiles = (width + 15) / 16;
        const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63u;
        const int64_t ty = b / tiles;
        p.x = int32_t(b - ty * tiles) * 16 + int32_t((w & 1u) * 8 + (l & 7u));
        const int64_t y = ty * 16 + int64_t((w >> 1) * 8 + (l >> 3));
        p.y = int32_t(y);
        p.i = p.x < width && y < height ? y * width + p.x : -1;
    } else {
        p.i = b * 256 + threadIdx.x;
        if (p.i >= int64_t(width) * height) p.i = -1;
        p.y = int32_t(p.i / width);
        p.x = int32_t(p.i - int64_t(p.y) * width);
    }
    return p;
}

}  // namespace dm
}  // namespace crt
