// Device collapse of one object's stack-layout BVH2 into the wide layout
// (crt_wide_build_gpu), for trees built on the device every frame
// (crt_build_bvh_gpu) that the wide walks should trace without a host round
// trip.
//
// It is crt_wide_build's collapse (wide_build.cpp) with 2-triangle leaves,
// level by level.  Each wide node of a level expands its BVH2 node as the host
// does: starting from the node's two children, the inner child of largest
// half surface area (the first one on a tie) is replaced by its own two
// children until the node holds `width` of them; a leaf, or an inner node of
// two adjacent 1-triangle leaves, stays one slot.  So every wide node has the
// host's slots, boxes, leaf ranges and slot order.  Nodes are numbered
// breadth-first, where the host numbers them depth-first as it allocates;
// walks visit the same boxes in the same order, so hit records, visit and
// test counts are identical.
//
// Nothing is read back between levels: the host launches a fixed number of
// level passes (one launch each), the level sizes live on the device, and a
// launch past the tree's depth returns at once (crt_wide_build_gpu_async).
// crt_wide_build_gpu runs the same launches and reads the node count and status
// back once.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>

#include "candela_rt.h"
#include "crt_internal.h"
#include "wide_collapse.h"

namespace crt {
namespace wg {

// ---- level passes --------------------------------------------------------
//
// The host launches a fixed number of passes and reads nothing back, so the
// whole collapse can be captured into a graph.  Level state lives on the
// device, two int64 per level l: lvl[2l] is the number of wide nodes numbered
// through level l (the first index of level l + 1) and lvl[2l + 1] the size of
// level l.  An expanded level leaves its inner children's stack entries in
// kids (W slots a node, -1 for the others) and, per kParents nodes, their
// number (sums).
//
// Pass k takes level p = first[k], numbers its children and expands them, a
// workgroup per kParents nodes: the children before it are the sums before its
// own, so a workgroup adds those up (at most a few thousand words) instead of
// waiting for another launch, and the numbering stays the host's.  Its
// children, at most kBlock, are packed in LDS and expanded by one thread each.
// A level of at most kParents nodes is one workgroup's work: it then goes on
// to the next level by itself while that is as small, so the narrow levels at
// the root and at the end of the tree share a launch.
//
// Bound: the chain of an expansion's dependent loads (its entry, then twice
// the opened child's and its children's), 5 to 10 us a level, and on the wide
// levels the gathered entries.  With two launches a level (expand, then assign
// numbers) and the children in scratch memory, the levels of 2.56M triangles
// took 703 us and those of 11,520 took 223; now 367 and 110 (width 4, 31 passes:
// the first, with the narrow levels at the root, 30 and 22, the widest 52 and 10,
// 4 and 25 past the end at 2 us each).

// Bit of *err: the tree has more levels than were launched.
constexpr unsigned kErrDepth = 8u;
static_assert(kErrLink == CRT_WIDE_GPU_BAD_LINK && kErrCap == CRT_WIDE_GPU_NOT_TREE &&
                  kErrVertex == CRT_WIDE_GPU_BAD_VERTEX && kErrDepth == CRT_WIDE_GPU_TOO_DEEP &&
                  kErrLeaf == CRT_WIDE_GPU_BAD_LEAF,
              "status bits are the header's");
// As many workgroups as the chip holds: a launch past the tree's depth costs
// 2 us with these, 4.6 us with 4,096.
constexpr int kGridMax = 1024;

// Level state and lists in the workspace (kids and sums: wide_collapse.h).
struct Lists {
    int64_t* lvl;
    int32_t* first;
    int32_t* kids;
    uint32_t* sums;
    int64_t sum_stride;
    int64_t cap;
    unsigned* err;

    template <int W>
    __device__ __forceinline__ int32_t* kids_of(int32_t level, int64_t item) const {
        return kids + kids_item(level, item, cap) * W;
    }
    __device__ __forceinline__ uint32_t* sums_of(int32_t level) const { return sums + sums_array(level) * sum_stride; }
};

// Sums of a and b over the workgroup (kBlock threads); every thread gets them.
__device__ __forceinline__ void block_sum2(uint64_t& a, uint64_t& b, uint64_t (*sh)[kBlock / 64]) {
    for (int d = 32; d > 0; d >>= 1) {
        a += __shfl_xor(a, d, 64);
        b += __shfl_xor(b, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = a;
        sh[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    a = b = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        a += sh[0][w];
        b += sh[1][w];
    }
    __syncthreads();
}

template <int W>
struct LevelLds {
    uint64_t sums[2][kBlock / 64];
    uint32_t wave_count[kBlock / 64];
    int32_t list[kBlock];
    uint32_t children[W + 1];   // per kParents items of the next level that this workgroup's touch
};

// Nodes [chunk * kParents, ...) of level p (np nodes, the last numbered
// next_base - 1): numbers their inner children next_base + before, ... and
// expands them.  Adds the children's own numbers of inner children to level
// p + 1's sums, with an atomic unless the workgroup has the level to itself.
template <int W>
__device__ __forceinline__ void expand_chunk(const crt_stack_node* __restrict__ nodes, int64_t node_count,
                                             int64_t ntris, const Lists& L, int32_t p, int64_t np, int64_t next_base,
                                             int64_t chunk, int64_t before, bool alone,
                                             crt_wide_group* __restrict__ groups, LevelLds<W>& lds) {
    const int tid = int(threadIdx.x), wave = tid >> 6;
    const int64_t parent = chunk * kParents<W> + tid / W;
    const int s = tid % W;
    const int32_t entry = parent < np ? L.kids_of<W>(p, parent)[s] : -1;
    const uint64_t ballot = __ballot(entry >= 0);
    const uint32_t below =
        __builtin_amdgcn_mbcnt_hi(uint32_t(ballot >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(ballot), 0u));
    if ((tid & 63) == 0) lds.wave_count[wave] = uint32_t(__popcll(ballot));
    if (tid <= W) lds.children[tid] = 0u;
    __syncthreads();
    uint32_t rank = below, count = 0u;
    for (int w = 0; w < kBlock / 64; ++w) {
        rank += w < wave ? lds.wave_count[w] : 0u;
        count += lds.wave_count[w];
    }
    if (entry >= 0) {
        assign_slot<W>(next_base - np + parent, s, next_base + before + rank, groups);
        lds.list[rank] = entry;
    }
    __syncthreads();
    const int64_t seg0 = sum_of<W>(before);
    if (tid < int(count)) {
        const int64_t item = before + tid;
        const uint32_t m = expand_one<W>(nodes, node_count, ntris, lds.list[tid], next_base + item, groups,
                                         L.kids_of<W>(p + 1, item), L.err);
        if (m) atomicAdd(&lds.children[sum_of<W>(item) - seg0], m);
    }
    __syncthreads();
    if (tid <= W && count > 0u && seg0 + tid <= sum_of<W>(before + count - 1)) {
        uint32_t* out = L.sums_of(p + 1) + seg0 + tid;
        if (alone)
            *out = lds.children[tid];
        else if (lds.children[tid])
            atomicAdd(out, lds.children[tid]);
    }
}

// Clears the sums that level p + 2 will need, when level p + 1 has `count` nodes.
template <int W>
__device__ __forceinline__ void clear_sums(const Lists& L, int32_t p, int64_t count, int64_t first, int64_t stride) {
    const int64_t need = sums_for<W>(count * W);
    uint32_t* out = L.sums_of(p + 2);
    for (int64_t k = first; k < need && k < L.sum_stride; k += stride) out[k] = 0u;
}

// Level 0 and the error word.  A root entry that holds two adjacent
// 1-triangle leaves is one 2-triangle leaf under a root of one slot
// (crt_wide_build's rule): this kernel writes that root, and level 0 is then
// empty.  Otherwise level 0 is the root entry, expanded here.
template <int W>
__global__ void __launch_bounds__(64) root_async(const crt_stack_node* __restrict__ nodes, int64_t node_count,
                                                 int64_t ntris, Lists L, crt_wide_group* __restrict__ groups) {
    if (threadIdx.x != 0) return;
    *L.err = 0u;
    Kid k;
    const bool one = root_one_slot(nodes[0], k);
    if (one) {
        const bool ok = leaf_ok(k.start, k.count, ntris);
        if (!ok) *L.err = kErrLeaf;   // finish_async leaves the root empty
        write_one_slot_root<W>(groups, k, ok);
    } else {
        L.sums_of(0)[0] = expand_one<W>(nodes, node_count, ntris, 0, 0, groups, L.kids_of<W>(0, 0), L.err);
        L.sums_of(1)[0] = 0u;   // level 1 has at most W nodes, within one sum
    }
    L.first[0] = 0;
    L.lvl[0] = 1;
    L.lvl[1] = one ? 0 : 1;
}

// Pass k of `levels` - 1.  A tree whose next level would pass cap stops there (kErrCap).
template <int W>
__global__ void __launch_bounds__(kBlock) level_async(const crt_stack_node* __restrict__ nodes, int64_t node_count,
                                                      int64_t ntris, Lists L, int32_t k, int32_t levels,
                                                      crt_wide_group* __restrict__ groups) {
    __shared__ LevelLds<W> lds;
    int32_t p = L.first[k];
    int64_t np = L.lvl[2 * p + 1];
    if (np == 0 || p >= levels - 1) {
        if (blockIdx.x == 0 && threadIdx.x == 0) L.first[k + 1] = p;
        return;
    }
    int64_t next_base = L.lvl[2 * p];
    if (np <= kParents<W>) {
        if (blockIdx.x != 0) return;
        do {
            __syncthreads();   // the last level's lists and sums are written
            const int64_t all = L.sums_of(p)[0];
            const bool over = next_base + all > L.cap;
            const int64_t size = over ? 0 : all;
            clear_sums<W>(L, p, size, threadIdx.x, kBlock);
            if (size > 0)
                expand_chunk<W>(nodes, node_count, ntris, L, p, np, next_base, 0, 0, true, groups, lds);
            if (threadIdx.x == 0) {
                if (over) atomicOr(L.err, kErrCap);
                L.lvl[2 * p + 2] = next_base + size;
                L.lvl[2 * p + 3] = size;
            }
            next_base += size;
            np = size;
            ++p;
        } while (np > 0 && np <= kParents<W> && p < levels - 1);
        if (threadIdx.x == 0) L.first[k + 1] = p;
        return;
    }
    const int64_t chunks = sums_for<W>(np);
    const uint32_t* sums = L.sums_of(p);
    if (blockIdx.x >= chunks) return;
    uint64_t before = 0, all = 0;
#pragma unroll 8
    for (int64_t j = threadIdx.x; j < chunks; j += kBlock) {
        const uint32_t v = sums[j];
        all += v;
        before += j < blockIdx.x ? v : 0u;
    }
    block_sum2(before, all, lds.sums);
    const bool over = next_base + int64_t(all) > L.cap;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (over) atomicOr(L.err, kErrCap);
        L.lvl[2 * p + 2] = next_base + (over ? 0 : int64_t(all));
        L.lvl[2 * p + 3] = over ? 0 : int64_t(all);
        L.first[k + 1] = p + 1;
    }
    if (over) return;
    // the workgroups that run here, min(grid, chunks) of them, clear together
    const int64_t groups_run = chunks < int64_t(gridDim.x) ? chunks : int64_t(gridDim.x);
    clear_sums<W>(L, p, int64_t(all), int64_t(blockIdx.x) * kBlock + threadIdx.x, groups_run * kBlock);
    for (int64_t c = blockIdx.x;;) {
        expand_chunk<W>(nodes, node_count, ntris, L, p, np, next_base, c, int64_t(before), false, groups, lds);
        const int64_t next = c + gridDim.x;
        if (next >= chunks) break;
        uint64_t more = 0, unused = 0;
        for (int64_t j = c + threadIdx.x; j < next; j += kBlock) more += sums[j];
        block_sum2(more, unused, lds.sums);   // its barriers also end the use of the lists
        before += more;
        c = next;
    }
}

// The node count, the number of levels the tree needs (the first empty
// level; max_levels when none was) and the status word for the caller.  A
// layout with any status bit is incomplete (levels never expanded hold stale
// memory, a failed slot reads as empty): its root is rewritten with every
// slot empty, so a trace that runs after it, in the same graph say, ends at
// the root with no hit.
template <int W>
__global__ void __launch_bounds__(kBlock) finish_async(Lists L, int32_t levels, int64_t* __restrict__ wide_nodes,
                                                       uint32_t* __restrict__ status,
                                                       crt_wide_group* __restrict__ groups) {
    __shared__ uint64_t sh[2][kBlock / 64];
    const int32_t p = L.first[levels - 1];   // the first empty level, or the last one expanded
    const int64_t np = L.lvl[2 * p + 1];
    uint64_t all = 0, unused = 0;            // children of the last level, which nothing numbered
    for (int64_t j = threadIdx.x; j < sums_for<W>(np); j += kBlock) all += L.sums_of(p)[j];
    block_sum2(all, unused, sh);
    const int64_t count = L.lvl[2 * p];
    const bool over = count + int64_t(all) > L.cap;
    const uint32_t st = *L.err | (all == 0 ? 0u : over ? kErrCap : kErrDepth);
    if (st != 0u) {
        // W / 4 groups of 8 fields of 4 words (32 words each)
        for (int k = int(threadIdx.x); k < (W / 4) * 32; k += kBlock) {
            int32_t* g = reinterpret_cast<int32_t*>(groups + k / 32);
            const int word = k % 32;
            g[word] = word >= 28 ? -1 : 0;   // count[4] is the last field
        }
    }
    if (threadIdx.x != 0) return;
    wide_nodes[0] = count + (over ? 0 : int64_t(all));
    wide_nodes[1] = np == 0 ? p : levels;
    *status = st;
}

// Triangle records in leaf order (crt_wide_build's).
__global__ void __launch_bounds__(kBlock) records(const crt_triangle* __restrict__ tris,
                                                  const crt_vertex* __restrict__ verts, int64_t nverts, int64_t n,
                                                  crt_tri_record* __restrict__ out, unsigned* __restrict__ err) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    crt_triangle t = tris[i];
    for (int k = 0; k < 3; ++k) {
        if (t.packed[k] < 0 || int64_t(t.packed[k]) >= nverts) {
            atomicOr(err, kErrVertex);
            t.packed[k] = 0;
        }
    }
    const float4 a = *reinterpret_cast<const float4*>(verts[t.packed[0]].position);
    const float4 b = *reinterpret_cast<const float4*>(verts[t.packed[1]].position);
    const float4 c = *reinterpret_cast<const float4*>(verts[t.packed[2]].position);
    float4* o = reinterpret_cast<float4*>(out + i);
    o[0] = make_float4(a.x, a.y, a.z, __int_as_float(int32_t(i)));
    o[1] = make_float4(b.x, b.y, b.z, __int_as_float(t.packed[3]));
    o[2] = make_float4(c.x, c.y, c.z, __int_as_float(0));
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

struct Layout {
    size_t kids, sums, err, lvl, first, out, bytes;
    int64_t sum_stride;
};

// Levels hold at most `cap` wide nodes (a valid tree has fewer wide nodes
// than triangles); the level state has room for `levels` levels.
inline Layout layout(int64_t cap, int32_t width, int32_t levels) {
    const size_t n = size_t(cap), nb = size_t((cap + kBlock - 1) / kBlock);
    Layout L{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align256(off + bytes);
        return at;
    };
    L.sum_stride = (width == 8 ? sums_for<8>(cap) : sums_for<4>(cap)) + 1;
    L.kids = take(n * size_t(width) * 4);
    L.sums = take(size_t(L.sum_stride) * 3 * 4);
    L.err = take(4);
    L.lvl = take(size_t(2) * size_t(levels + 1) * 8);
    L.first = take(size_t(levels) * 4);
    L.out = take(3 * 8);   // crt_wide_build_gpu's node count, level count and status
    // no less than callers have been told to reserve: the width's child slots
    // and five more words a triangle
    L.bytes = std::max(off, align256(n * (size_t(width) + 5) * 4) + align256(nb * 4) +
                                align256(size_t(levels + 1) * 16));
    return L;
}

template <int W>
void collapse_async(const crt_stack_node* nodes, int64_t node_count, const crt_triangle* tris,
                    const crt_vertex* verts, int64_t nverts, int64_t cap, int32_t levels, crt_wide_group* groups,
                    crt_tri_record* recs, int64_t* wide_nodes, uint32_t* status, char* ws, const Layout& L,
                    hipStream_t st) {
    const Lists lists{reinterpret_cast<int64_t*>(ws + L.lvl),   reinterpret_cast<int32_t*>(ws + L.first),
                      reinterpret_cast<int32_t*>(ws + L.kids),  reinterpret_cast<uint32_t*>(ws + L.sums),
                      L.sum_stride,                              cap,
                      reinterpret_cast<unsigned*>(ws + L.err)};
    const int32_t grid = int32_t(std::min<int64_t>(kGridMax, sums_for<W>(cap)));
    hipLaunchKernelGGL(root_async<W>, dim3(1), dim3(64), 0, st, nodes, node_count, cap, lists, groups);
    hipLaunchKernelGGL(records, dim3(unsigned((cap + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, tris, verts, nverts,
                       cap, recs, lists.err);
    for (int32_t k = 0; k < levels - 1; ++k)
        hipLaunchKernelGGL(level_async<W>, dim3(unsigned(grid)), dim3(kBlock), 0, st, nodes, node_count, cap, lists, k,
                           levels, groups);
    hipLaunchKernelGGL(finish_async<W>, dim3(1), dim3(kBlock), 0, st, lists, levels, wide_nodes, status, groups);
}

}  // namespace wg
}  // namespace crt

extern "C" {

size_t crt_wide_build_gpu_workspace(int64_t ntris, int32_t width) {
    if (ntris < 2 || (width != 4 && width != 8)) return 0;
    return crt::wg::layout(ntris, width, CRT_WIDE_GPU_MAX_LEVELS).bytes;
}

// The asynchronous collapse with kFirstLevels levels, and again with every
// level CRT_WIDE_GPU_MAX_LEVELS allows when the tree is deeper; one readback
// of the node count and status per run.
int crt_wide_build_gpu(const crt_stack_node* nodes, int64_t node_count, const crt_triangle* triangles, int64_t ntris,
                       const crt_vertex* vertices, int64_t nverts, int32_t width, crt_wide_group* groups,
                       crt_tri_record* records, int64_t* wide_nodes, void* workspace, size_t workspace_bytes,
                       void* stream) {
    using namespace crt::wg;
    constexpr int32_t kFirstLevels = 32;
    if (!nodes || !triangles || !vertices || !groups || !records || !wide_nodes || !workspace)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: null argument");
    if (width != 4 && width != 8) return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: width must be 4 or 8");
    if (ntris < 2 || node_count < 1 || nverts < 1 || ntris > 0x7FFFFFFFll)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: needs 2 to 2^31 - 1 triangles and a root entry");
    const Layout L = layout(ntris, width, CRT_WIDE_GPU_MAX_LEVELS);
    if (workspace_bytes < L.bytes || reinterpret_cast<uintptr_t>(workspace) % 256 != 0)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: workspace must be 256-byte aligned and hold "
                                             "crt_wide_build_gpu_workspace(ntris, width) = " +
                                                 std::to_string(L.bytes) + " bytes");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    auto* out = reinterpret_cast<int64_t*>(ws + L.out);
    auto* status = reinterpret_cast<uint32_t*>(out + 2);
    int64_t host_out[3] = {0, 0, 0};
    for (const int32_t levels : {kFirstLevels, int32_t(CRT_WIDE_GPU_MAX_LEVELS)}) {
        if (width == 4)
            collapse_async<4>(nodes, node_count, triangles, vertices, nverts, ntris, levels, groups, records, out,
                              status, ws, L, st);
        else
            collapse_async<8>(nodes, node_count, triangles, vertices, nverts, ntris, levels, groups, records, out,
                              status, ws, L, st);
        if (hipMemcpyAsync(host_out, out, sizeof(host_out), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return crt::set_error(CRT_E_HIP, std::string("crt_wide_build_gpu: ") + hipGetErrorString(hipGetLastError()));
        if (!(uint32_t(host_out[2]) & kErrDepth)) break;
    }
    const uint32_t bad = uint32_t(host_out[2]);
    if (bad & kErrVertex)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: a vertex index leaves the vertex array");
    if (bad & kErrLink) return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: a stack link leaves the node array");
    if (bad & kErrLeaf)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: a leaf range is empty or leaves [0, ntris) (the "
                                             "tree must be built with triangle offset 0)");
    if (bad & kErrCap)
        return crt::set_error(CRT_E_INVALID,
                              "crt_wide_build_gpu: more wide nodes than triangles (the links do not form a tree)");
    if (bad & kErrDepth)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu: the tree has more than " +
                                                 std::to_string(CRT_WIDE_GPU_MAX_LEVELS) + " wide levels");
    *wide_nodes = host_out[0];
    return CRT_OK;
}

size_t crt_wide_build_gpu_async_workspace(int64_t ntris, int32_t width, int32_t max_levels) {
    if (ntris < 2 || (width != 4 && width != 8) || max_levels < 1 || max_levels > CRT_WIDE_GPU_MAX_LEVELS) return 0;
    return crt::wg::layout(ntris, width, max_levels).bytes;
}

int crt_wide_build_gpu_async(const crt_stack_node* nodes, int64_t node_count, const crt_triangle* triangles,
                             int64_t ntris, const crt_vertex* vertices, int64_t nverts, int32_t width,
                             int32_t max_levels, crt_wide_group* groups, crt_tri_record* records,
                             int64_t* wide_nodes, uint32_t* status, void* workspace, size_t workspace_bytes,
                             void* stream) {
    using namespace crt::wg;
    if (!nodes || !triangles || !vertices || !groups || !records || !wide_nodes || !status || !workspace)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu_async: null argument");
    if (width != 4 && width != 8)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu_async: width must be 4 or 8");
    if (max_levels < 1 || max_levels > CRT_WIDE_GPU_MAX_LEVELS)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu_async: max_levels must be 1 to " +
                                                 std::to_string(CRT_WIDE_GPU_MAX_LEVELS));
    if (ntris < 2 || node_count < 1 || nverts < 1 || ntris > 0x7FFFFFFFll)
        return crt::set_error(CRT_E_INVALID,
                              "crt_wide_build_gpu_async: needs 2 to 2^31 - 1 triangles and a root entry");
    const Layout L = layout(ntris, width, max_levels);
    if (workspace_bytes < L.bytes || reinterpret_cast<uintptr_t>(workspace) % 256 != 0)
        return crt::set_error(CRT_E_INVALID, "crt_wide_build_gpu_async: workspace must be 256-byte aligned and hold "
                                             "crt_wide_build_gpu_async_workspace(ntris, width, max_levels) = " +
                                                 std::to_string(L.bytes) + " bytes");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    if (width == 4)
        collapse_async<4>(nodes, node_count, triangles, vertices, nverts, ntris, max_levels, groups, records,
                          wide_nodes, status, ws, L, st);
    else
        collapse_async<8>(nodes, node_count, triangles, vertices, nverts, ntris, max_levels, groups, records,
                          wide_nodes, status, ws, L, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return crt::set_error(CRT_E_HIP, std::string("crt_wide_build_gpu_async: ") + hipGetErrorString(e));
    return CRT_OK;
}

}  // extern "C"
