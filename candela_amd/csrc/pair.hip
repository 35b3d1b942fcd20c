// Launchers of the pair walk (pair_walk.h) over a context's stackless scene:
// a ray batch, or an image's primary rays.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "pair_walk.h"
#include "primary_ray.h"
#include "trace_launch.h"

#pragma clang fp contract(off)

namespace crt {
namespace pair {

template <bool ANY, bool TOGETHER, int D, int I, int LB>
__global__ void __launch_bounds__(256) pair_grid(PairScene s, const crt_ray* rays, crt_hit* __restrict__ hits,
                                                 int64_t n, uint32_t flags, int32_t max_iter, int32_t log2,
                                                 int32_t blocks) {
    __shared__ typename PairStack<D>::Entry lds[D * 256];
    const int64_t i = grid_ray(n, log2, blocks);
    typename PairStack<D>::Entry spill[spill_entries<D>()];
    PairStack<D> st{lds + threadIdx.x, 256, spill};
    PairWave<ANY, D, I, LB> w;
    if constexpr (TOGETHER)
        w.run_together(s, rays, hits, i, flags, max_iter, st);
    else
        w.run(s, rays, hits, i, flags, max_iter, st);
}

template <int D, int I, int LB>
__global__ void __launch_bounds__(256) pair_primary(PairScene s, Camera cam, crt_ray* rays, crt_hit* __restrict__ hits,
                                                    ImageTiles image, uint32_t flags, int32_t max_iter) {
    __shared__ typename PairStack<D>::Entry lds[D * 256];
    const Pixel p = image_pixel(image);
    // a lane reads back only the ray that it wrote itself
    if (p.i >= 0) store_ray(rays + p.i, primary_ray(cam, image.width, image.height, p.x, p.y, uint32_t(p.i)));
    typename PairStack<D>::Entry spill[spill_entries<D>()];
    PairStack<D> st{lds + threadIdx.x, 256, spill};
    PairWave<false, D, I, LB> w;
    w.run_together(s, rays, hits, p.i, flags, max_iter, st);
}

}  // namespace pair

// LDS stack entries, node steps per round, parked lanes that end the node
// phase.  10 entries (20 KB a workgroup) leave the 7 waves per SIMD that the
// registers allow: with 12 (6 waves) 1920 x 1080 primary rays over 640,000 triangles
// take 7% longer.  Bounce rays take as long with (4, 8), 2% longer with (8, 8), 7%
// with (2, 8).
#define CRT_PAIR_SHAPE 10, 4, 16

// Waves of fewer than 64 rays, and images, go from entity to entity together
// (run_together); full waves, whose rays may meet any of them, each at its own
// pace.
hipError_t launch_pair_grid(const PairScene& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                            uint32_t flags, int32_t max_iter, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const int32_t log2 = rays_per_wave_log2(n);
    const int32_t blocks = int32_t((n + (4 << log2) - 1) >> (log2 + 2));
    const unsigned padded = unsigned((blocks + 7) / 8 * 8);
    const bool any = query == CRT_QUERY_ANY, together = log2 < 6;
    const auto fn = any ? (together ? pair::pair_grid<true, true, CRT_PAIR_SHAPE> : pair::pair_grid<true, false, CRT_PAIR_SHAPE>)
                        : (together ? pair::pair_grid<false, true, CRT_PAIR_SHAPE> : pair::pair_grid<false, false, CRT_PAIR_SHAPE>);
    hipLaunchKernelGGL(fn, dim3(padded), dim3(256), 0, stream, s, rays, hits, n, flags, max_iter, log2, blocks);
    return hipGetLastError();
}

hipError_t launch_pair_primary(const PairScene& s, const Camera& cam, crt_ray* rays, crt_hit* hits, int width,
                               int height, uint32_t flags, int32_t max_iter, hipStream_t stream) {
    const dm::ImageTiles image = dm::image_tiles(width, height);
    hipLaunchKernelGGL((pair::pair_primary<CRT_PAIR_SHAPE>),
                       dim3(dm::image_grid(image)), dim3(256), 0, stream, s, cam, rays, hits, image, flags, max_iter);
    return hipGetLastError();
}

}  // namespace crt
