// What a context derives from the data it buffers (crt_buffer_data) for the
// walks of pair_walk.h and stack_walk.h: one record per triangle, and the child
// pairs of a stackless tree.
//
// Pairs are numbered in the order of their inner nodes, object by object.  An
// inner node's rank is the number of inner nodes before it, from counts per
// workgroup and their scan.  Whether an object's nodes are the pre-order array of
// a plain tree, which the walk of the pairs relies on, is found node by node: an
// inner node i has the children i + 1 and link(i + 1), the right one inherits its
// link, and a leaf's link is the node behind it.  These conditions nest, so
// together they make every node's subtree [i, link(i)); its size then gives the
// right child's rank as well.
//
// Bound: the copies of the data from host memory that come before.  Buffering
// 2.56M triangles with a stackless tree takes 7.5 ms (6.5 without the derived
// arrays); with pairs formed on the host and uploaded it took 40.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "device_math.h"
#include "scan.h"
#include "trace_launch.h"

namespace crt {
namespace pair {

using namespace ::crt::dm;
using scan::kBlock;

// Triangle i's record.  A vertex index outside [0, nverts) sets *bad.
__global__ void __launch_bounds__(kBlock) gather_records(const crt_triangle* __restrict__ tris,
                                                         const crt_vertex* __restrict__ verts, int64_t nverts,
                                                         int64_t n, float4* __restrict__ out,
                                                         uint32_t* __restrict__ bad) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int4 t = *reinterpret_cast<const int4*>(tris[i].packed);
    if (uint32_t(t.x) >= nverts || uint32_t(t.y) >= nverts || uint32_t(t.z) >= nverts) {
        *bad = 1u;
        return;
    }
    const f3 a = vertex_pos(verts, t.x), b = vertex_pos(verts, t.y), c = vertex_pos(verts, t.z);
    out[3 * i] = make_float4(a.x, a.y, a.z, __int_as_float(int32_t(i)));
    out[3 * i + 1] = make_float4(b.x, b.y, b.z, __int_as_float(t.w));
    out[3 * i + 2] = make_float4(c.x, c.y, c.z, 0.0f);
}

__device__ __forceinline__ bool inner(const float4* __restrict__ nodes, int64_t i, int64_t n) {
    return i < n && __float_as_int(nodes[2 * i].w) == -1;
}

__global__ void __launch_bounds__(kBlock) count_inner(const float4* __restrict__ nodes, int64_t n,
                                                      uint32_t* __restrict__ counts) {
    __shared__ uint32_t waves[kBlock / 64];
    uint32_t total;
    (void)scan::block_rank(inner(nodes, int64_t(blockIdx.x) * kBlock + threadIdx.x, n), waves, total);
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// Inner nodes before each object's first node, a wave per object.
__global__ void __launch_bounds__(64) object_ranks(const float4* __restrict__ nodes,
                                                   const NodeRange* __restrict__ objects,
                                                   const int64_t* __restrict__ offsets, int64_t* __restrict__ ranks) {
    const int64_t start = objects[blockIdx.x].start, block = start / kBlock;
    int64_t rank = offsets[block];
    for (int64_t i = block * kBlock; i < start; i += 64)
        rank += __popcll(__ballot(inner(nodes, i + threadIdx.x, start)));
    if (threadIdx.x == 0) ranks[blockIdx.x] = rank;
}

// The pair of inner node i, and the checks of every node (bad[object] = 1).
__global__ void __launch_bounds__(kBlock) write_pairs(const float4* __restrict__ nodes, int64_t n,
                                                      const NodeRange* __restrict__ objects, int64_t nobjects,
                                                      const int64_t* __restrict__ offsets,
                                                      const int64_t* __restrict__ ranks, int64_t ntris,
                                                      float4* __restrict__ pairs, uint32_t* __restrict__ bad) {
    __shared__ uint32_t waves[kBlock / 64];
    const int64_t g = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    uint32_t total;
    const uint32_t below = scan::block_rank(inner(nodes, g, n), waves, total);
    if (g >= n) return;
    // the last object that starts at g or before it
    int64_t lo = 0, hi = nobjects;
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) / 2;
        (objects[mid].start <= g ? lo : hi) = mid;
    }
    const int64_t start = objects[lo].start, count = objects[lo].count;
    const int64_t i = g - start;
    if (i < 0 || i >= count) return;
    const float4* o = nodes + 2 * start;   // the object's nodes
    const auto link_of = [&](int64_t k) { return __float_as_int(o[2 * k + 1].w); };
    const int64_t link = link_of(i), end = link < 0 ? count : link;
    const int32_t packed = __float_as_int(o[2 * i].w);
    bool ok = link >= -1 && link < count && (i > 0 || link == -1);
    if (packed != -1) {
        ok = ok && packed >= 0 && end == i + 1 && int64_t(packed >> 4) + (packed & 0xF) <= ntris;
    } else if (ok && i + 1 < count) {
        const int64_t r = link_of(i + 1);
        // in a plain tree the left subtree's i + 1 .. r - 1 are one node more than twice its inner nodes
        const int64_t left = r - (i + 1), rank = offsets[blockIdx.x] + below - ranks[lo];
        ok = r > i + 1 && r < end && link_of(r) == link && left % 2 == 1 && rank < (count - 1) / 2 &&
             2 * rank - i + 1 <= kPairStack;   // right children pending below i, its own among them
        if (ok) {
            const int32_t first = pair_base(int32_t(start));
            const int32_t lref = int32_t(first + rank + 1), rref = lref + int32_t((left - 1) / 2);
            const float4 lmin = o[2 * i + 2], lmax = o[2 * i + 3], rmin = o[2 * r], rmax = o[2 * r + 1];
            const int32_t lp = __float_as_int(lmin.w), rp = __float_as_int(rmin.w);
            float4* p = pairs + 4 * (first + rank);
            p[0] = make_float4(lmin.x, lmin.y, lmin.z, __int_as_float(lp == -1 ? ~lref : lp));
            p[1] = make_float4(lmax.x, lmax.y, lmax.z, 0.0f);
            p[2] = make_float4(rmin.x, rmin.y, rmin.z, __int_as_float(rp == -1 ? ~rref : rp));
            p[3] = make_float4(rmax.x, rmax.y, rmax.z, 0.0f);
        }
    } else {
        ok = false;
    }
    if (!ok) bad[lo] = 1u;
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

struct Scratch {
    size_t counts, offsets, ranks, total, bytes;
};

inline Scratch scratch(int64_t n, int64_t nobjects) {
    const size_t blocks = size_t((n + kBlock - 1) / kBlock);
    Scratch s{};
    s.offsets = align256(blocks * 4);
    s.ranks = s.offsets + align256(blocks * 8);
    s.total = s.ranks + align256(size_t(nobjects) * 8);
    s.bytes = s.total + 256;
    return s;
}

}  // namespace pair

hipError_t launch_gather_records(const crt_triangle* tris, const crt_vertex* verts, int64_t nverts, int64_t n,
                                 crt_tri_record* out, uint32_t* bad, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(pair::gather_records, dim3(unsigned((n + scan::kBlock - 1) / scan::kBlock)), dim3(scan::kBlock),
                       0, stream, tris, verts, nverts, n, reinterpret_cast<float4*>(out), bad);
    return hipGetLastError();
}

size_t pairs_scratch(int64_t nnodes, int64_t nobjects) { return pair::scratch(nnodes, nobjects).bytes; }

hipError_t launch_build_pairs(const crt_stackless_node* nodes, int64_t nnodes, const NodeRange* objects,
                              int64_t nobjects, int64_t ntris, crt_stack_node* pairs, void* scratch, uint32_t* bad,
                              hipStream_t stream) {
    if (nnodes <= 0 || nobjects <= 0) return hipSuccess;
    const pair::Scratch at = pair::scratch(nnodes, nobjects);
    char* s = static_cast<char*>(scratch);
    auto* counts = reinterpret_cast<uint32_t*>(s);
    auto* offsets = reinterpret_cast<int64_t*>(s + at.offsets);
    auto* ranks = reinterpret_cast<int64_t*>(s + at.ranks);
    const auto* nd = reinterpret_cast<const float4*>(nodes);
    const int64_t blocks = (nnodes + scan::kBlock - 1) / scan::kBlock;
    const dim3 grid{unsigned(blocks)}, block{unsigned(scan::kBlock)};
    hipLaunchKernelGGL(pair::count_inner, grid, block, 0, stream, nd, nnodes, counts);
    hipLaunchKernelGGL(scan::exclusive_scan, dim3(1), dim3(scan::kScanBlock), 0, stream, counts, blocks, offsets,
                       reinterpret_cast<int64_t*>(s + at.total));
    hipLaunchKernelGGL(pair::object_ranks, dim3(unsigned(nobjects)), dim3(64), 0, stream, nd, objects, offsets, ranks);
    hipLaunchKernelGGL(pair::write_pairs, grid, block, 0, stream, nd, nnodes, objects, nobjects, offsets, ranks, ntris,
                       reinterpret_cast<float4*>(pairs), bad);
    return hipGetLastError();
}

}  // namespace crt
