// Kernel arguments and launchers shared by the host runtime and trace.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"

namespace crt {

// Device scene passed by value to every kernel (SSBO bindings 16..19 plus
// u_EntityCount / u_TotalNodes of the reference's traversal include).
struct SceneArgs {
    int32_t format;
    int32_t entity_count;
    int64_t total_nodes;
    const void* nodes;
    const crt_triangle* tris;
    const crt_vertex* verts;
    const crt_entity* entities;
    const crt_tri_record* tri_records;  // wide formats only
};

// SceneArgs of a scene view.
inline SceneArgs scene_args(const crt_scene_view& v) {
    return SceneArgs{v.format, v.entity_count, v.total_nodes, v.nodes, v.triangles, v.vertices, v.entities,
                     v.tri_records};
}

struct Camera {
    float inv_view[16];
    float inv_proj[16];
    float tmax;
};

// A context's stackless scene with the derived arrays of pair_layout.hip: the
// child pairs of every inner node (an object's first pair is that of its root,
// at pair_base of its first node) and one record per triangle.
struct PairScene {
    int32_t entity_count;
    const crt_entity* entities;
    const float4* nodes;     // crt_stackless_node[]
    const float4* pairs;     // crt_stack_node[]; min.w holds the child (pair_walk.h), max.w nothing
    const float4* records;   // crt_tri_record[] by triangle index
};

// Objects are full binary trees one behind the other, so (start + 1) / 2
// leaves every object room for its (nodes - 1) / 2 pairs.
__host__ __device__ constexpr int32_t pair_base(int32_t start) { return (start + 1) >> 1; }
constexpr int32_t kPairStack = 64;   // pending right children that a pair walk can hold

// One object's nodes.
struct NodeRange {
    int32_t start, count;
    bool operator<(const NodeRange& o) const { return start != o.start ? start < o.start : count < o.count; }
};

// A record per triangle; *bad = 1 when one names a vertex outside [0, nverts).
hipError_t launch_gather_records(const crt_triangle* tris, const crt_vertex* verts, int64_t nverts, int64_t n,
                                 crt_tri_record* out, uint32_t* bad, hipStream_t stream);
// The child pairs of the objects (in the order of their nodes, none overlapping,
// below 2^31 nodes) into pairs[(nnodes + 1) / 2]; bad[k] = 1 when object k's
// nodes are no pre-order tree with leaves inside [0, ntris) whose walk holds at
// most kPairStack pending children.  scratch: pairs_scratch bytes.
size_t pairs_scratch(int64_t nnodes, int64_t nobjects);
hipError_t launch_build_pairs(const crt_stackless_node* nodes, int64_t nnodes, const NodeRange* objects,
                              int64_t nobjects, int64_t ntris, crt_stack_node* pairs, void* scratch, uint32_t* bad,
                              hipStream_t stream);
hipError_t launch_pair_grid(const PairScene& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                            uint32_t flags, int32_t max_iter, hipStream_t stream);
hipError_t launch_pair_primary(const PairScene& s, const Camera& cam, crt_ray* rays, crt_hit* hits, int width,
                               int height, uint32_t flags, int32_t max_iter, hipStream_t stream);

constexpr int32_t kMaxIterations = 1024;  // TraverseBVHStackless.glsl:184

// The wave-scheduled walks (wave_walk.h, stack_walk.h, wide_walk.h,
// spec_walk.h) run the walk-end code (the next entity's transform, or the
// ray's hit record) once this many lanes have finished their walks, or once
// no lane can step: that code costs the whole wave however few lanes it
// serves.  Finished lanes only wait; a ray's record does not depend on when
// its end runs (the speculative twin replays the rule for its schedule).
// Measured on config 2: 4-8% off the sequential BVH4 walks, 3% off the BVH2
// wave walks, 6% off the speculative GI launch (16 and 48 gain less).
constexpr int32_t kWalkEndBatch = 32;

hipError_t launch_trace(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                        uint32_t flags, int32_t max_iter, int block, int lds_depth, uint32_t* tri_tests,
                        hipStream_t stream);

hipError_t launch_primary(const SceneArgs& s, const Camera& cam, crt_ray* rays, crt_hit* hits, int width, int height,
                          uint32_t flags, int32_t max_iter, int block, hipStream_t stream);

// Tuning of the persistent kernel.
struct PersistentShape {
    int variant;  // refill / inner / leaf-batch preset
    int grid;     // workgroups launched
};

hipError_t launch_persistent(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                             uint32_t flags, int32_t max_iter, unsigned long long* counter, uint32_t* tri_tests,
                             const PersistentShape& shape, hipStream_t stream);

hipError_t launch_grid(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n, uint32_t flags,
                       int32_t max_iter, uint32_t* tri_tests, int variant, hipStream_t stream);

// Refilling persistent walk of the wide layouts (variant 0..5; grid 0 = fill
// every CU); `counters` is a queue block (queue_acquire) the launch resets itself.
hipError_t launch_wide_persistent(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                                  uint32_t flags, int32_t max_iter, unsigned long long* counters, uint32_t* tri_tests,
                                  int variant, int grid, hipStream_t stream);

// Wave-scheduled walk of the wide layouts (variant 0..5).
hipError_t launch_wide_grid(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                            uint32_t flags, int32_t max_iter, uint32_t* tri_tests, int variant, hipStream_t stream);

// Wave-scheduled walk of the stack layout (variant 0..7).
hipError_t launch_stack_grid(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                             uint32_t flags, int32_t max_iter, uint32_t* tri_tests, int variant, hipStream_t stream);

// Refilling persistent walk of the stack layout (variant 0..7; grid 0 = fill
// every CU); `counters` is a queue block the launch resets itself.
hipError_t launch_stack_persistent(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                                   uint32_t flags, int32_t max_iter, unsigned long long* counters,
                                   uint32_t* tri_tests, int variant, int grid, hipStream_t stream);

// log2 of the rays a wave takes.  A wave costs what its rays cost together, so
// a launch of few rays spreads them over about all the waves that the device holds
// at once (6 or 7 of these walks on each of 1,024 SIMDs): 300 rays over 3,074 triangles take 28 us with
// one ray a wave, 31 with 4 and 40 with 64; 5,976 primary rays 102, 123 and 153;
// 41,736 bounce rays, with 8, 78 against 90.  More waves than fit only add up:
// 59,000 rays take 66 us with 16 a wave, 83 with 4 and 166 with one.
inline int32_t rays_per_wave_log2(int64_t n, int64_t waves = 6144) {
    int32_t k = 0;
    while (k < 6 && (n >> k) > waves) ++k;
    return k;
}
// The speculative walks want fewer waves: they test the leaves of all their rays
// together.  Occlusion and bounce rays of an 86 x 85 image 141 us with 64 rays a
// wave, 122 over 1,024 waves, 114 over 2,048, 108 over 3,072; of 423 x 384
// pixels 144, 126, 124 and 133.  Half waves gain little (40,000 rays over one
// entity of 77,000 triangles 59 us, 59 with 64 a wave) and cost up to 1.28 times as
// much where a ray meets several entities (8 of 3,074 triangles: 117 and 92 us), so a
// wave takes 16 rays or fewer, or 64.  What is left to lose are a few hundred
// rays over many instances that they pass by, where more waves wait for each
// other's instruction fetches: 500 rays over 64 of 20 triangles 131 us in one-ray
// waves, 123 with 64 a wave, in BVH8 218 and 167; overlapping instances gain (8
// of 3,074 triangles: 42 and 76 us, BVH8 50 and 91).
constexpr int64_t kSpecWaves = 2048;
inline int32_t spec_rays_per_wave_log2(int64_t n) {
    const int32_t k = rays_per_wave_log2(n, kSpecWaves);
    return k == 5 ? 6 : k;
}
// Workgroups of four waves that n rays then take.
inline int32_t wave_blocks(int64_t n, int32_t log2) { return int32_t((n + (4 << log2) - 1) >> (log2 + 2)); }

// Ray of a grid launch's lane (workgroups of four waves, dealt to the XCDs so
// that consecutive ones share an L2; the grid is padded to a multiple of 8), or
// -1.  `blocks` = ceil(n / (4 << log2)).
#ifdef __HIPCC__
__device__ __forceinline__ int64_t grid_ray(int64_t n, int32_t log2, int32_t blocks) {
    const int32_t per = (blocks + 7) / 8;
    const int32_t logical = int32_t(blockIdx.x % 8u) * per + int32_t(blockIdx.x / 8u);
    const uint32_t lane = threadIdx.x & 63u;
    if (logical >= blocks || lane >> log2) return -1;
    const int64_t i = ((int64_t(logical) * 4 + (threadIdx.x >> 6)) << log2) + lane;
    return i < n ? i : -1;
}
#endif

// The stack walk over a context's triangle records (s.tri_records, by triangle index).
hipError_t launch_stack_records(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                                uint32_t flags, int32_t max_iter, hipStream_t stream);
hipError_t launch_stack_primary(const SceneArgs& s, const Camera& cam, crt_ray* rays, crt_hit* hits, int width,
                                int height, uint32_t flags, int32_t max_iter, hipStream_t stream);

// Speculative wave walk of the wide layouts (spec.hip; variant 0..5): grid
// launch, and device-filling waves that refill from a queue block.
hipError_t launch_spec_grid(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                            uint32_t flags, int32_t max_iter, uint32_t* tri_tests, int variant, hipStream_t stream);
hipError_t launch_spec_persistent(const SceneArgs& s, int query, const crt_ray* rays, crt_hit* hits, int64_t n,
                                  uint32_t flags, int32_t max_iter, unsigned long long* counters,
                                  uint32_t* tri_tests, int variant, int grid, hipStream_t stream);

// Speculative walks of the BVH2 layouts (spec_bvh2.hip; variant 0..3):
// stack = true for CRT_FORMAT_STACK, false for CRT_FORMAT_STACKLESS.
hipError_t launch_spec_bvh2_grid(const SceneArgs& s, bool stack, int query, const crt_ray* rays, crt_hit* hits,
                                 int64_t n, uint32_t flags, int32_t max_iter, uint32_t* tri_tests, int variant,
                                 hipStream_t stream);
hipError_t launch_spec_bvh2_persistent(const SceneArgs& s, bool stack, int query, const crt_ray* rays, crt_hit* hits,
                                       int64_t n, uint32_t flags, int32_t max_iter, unsigned long long* counters,
                                       uint32_t* tri_tests, int variant, int grid, hipStream_t stream);

// Workgroups of 256 threads that fill every CU with the persistent kernel.
int persistent_fill_grid(int query);

hipError_t launch_copy16(void* dst, const void* src, int64_t n16, hipStream_t stream);

}  // namespace crt
