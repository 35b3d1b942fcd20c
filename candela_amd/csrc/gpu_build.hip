// Device BVH builder: a linear BVH over Morton codes (Karras, "Maximizing
// Parallelism in the Construction of BVHs, Octrees, and k-d Trees", HPG
// 2012), written into the reference's stack layout.
//
// The reference builds on the CPU (BuildBVH, BVHConstructor.cpp:951-1108)
// with binned SAH; that tree is not what this builder produces, so its
// buffers are not byte-identical to BuildBVH's (traversal results are: every
// walk reports the nearest hit).  It exists for scenes rebuilt every frame:
// 15.6M triangles take seconds on the host and milliseconds here.
//
// Steps, all on one stream, none allocating (the caller passes a workspace):
//   1. per triangle its box centroid ((min + max) * 0.5, as ConstructTree
//      caches it, BVHConstructor.cpp:404-427); bounds of the centroids by a
//      grid-stride min/max reduction;
//   2. a 30-bit Morton code of the centroid quantized to 1024 cells per axis
//      (each workgroup folds the partial bounds itself), and the first digit's
//      count per tile;
//   3. a stable LSD radix sort of (code, triangle) by 8-bit digits, 4 passes of
//      two launches: count the digits per tile, then scatter each tile's codes
//      in digit order (a tile finds its place from the counts before it);
//   4. the tree (Karras's radix tree; ties broken by the sorted index, so every
//      code is distinct), the boxes and the stack layout in one pass over
//      chunks of 512 leaves: a node whose leaf range lies in one chunk, all but
//      about one in 60, is found by binary searches in LDS, takes its
//      children's boxes from the chunk's power-of-two box windows and is
//      written at once;
//   5. the remaining nodes, whose range crosses chunks: 16 lanes each find the
//      range and the split 16 codes at a time and forms the boxes from leaf
//      boxes at both ends and the boxes of 64 and 4,096 leaves between them.
//   Entry i holds internal node i's two children; a child covering two
//   triangles is written as a 2-triangle leaf.
//
// Measured on 2.56M triangles (2,000 spheres): 301 us, of them bounds and codes
// 38, sort 109, tree with boxes and entries 104 + 5 + 45; with 4-bit digits,
// three launches a pass and separate tree, box and entry passes it was 743 us.
// 11,520 triangles: 82 us instead of 145, nearly all launches and latency.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>

#include "candela_rt.h"
#include "crt_internal.h"
#include "scan.h"

namespace crt {
namespace gb {

using scan::kBlock;

constexpr int kMortonBits = 30;

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box tri_box(const crt_vertex* __restrict__ v, const uint32_t* __restrict__ idx, int64_t t) {
    Box b;
    const float4 p0 = *reinterpret_cast<const float4*>(v[idx[3 * t + 0]].position);
    const float4 p1 = *reinterpret_cast<const float4*>(v[idx[3 * t + 1]].position);
    const float4 p2 = *reinterpret_cast<const float4*>(v[idx[3 * t + 2]].position);
    b.lo[0] = fminf(fminf(p0.x, p1.x), p2.x);
    b.lo[1] = fminf(fminf(p0.y, p1.y), p2.y);
    b.lo[2] = fminf(fminf(p0.z, p1.z), p2.z);
    b.hi[0] = fmaxf(fmaxf(p0.x, p1.x), p2.x);
    b.hi[1] = fmaxf(fmaxf(p0.y, p1.y), p2.y);
    b.hi[2] = fmaxf(fmaxf(p0.z, p1.z), p2.z);
    return b;
}

__device__ __forceinline__ void centroid(const Box& b, float c[3]) {
    for (int k = 0; k < 3; ++k) c[k] = (b.lo[k] + b.hi[k]) * 0.5f;
}

// Per-workgroup min / max of the centroids over a grid-stride loop:
// partial[k * gridDim.x + block], k = 0..2 lo, 3..5 hi.  Also clears what later
// launches add to, the super-tile counts of every sort pass (kernel stores, no
// memset node, so the chain stays capturable).
constexpr int kBoundsGrid = 1024;   // at most this many workgroups (and partials)

__device__ __forceinline__ float wave_min(float v) {
    for (int d = 32; d > 0; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
    for (int d = 32; d > 0; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

// Min (lo) and max (hi) over the workgroup's threads; every thread gets them.
__device__ __forceinline__ void block_bounds(float lo[3], float hi[3], float (&sh)[6][kBlock / 64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < 3; ++k) {
        lo[k] = wave_min(lo[k]);
        hi[k] = wave_max(hi[k]);
        if (lane == 0) {
            sh[k][wave] = lo[k];
            sh[3 + k][wave] = hi[k];
        }
    }
    __syncthreads();
    for (int k = 0; k < 3; ++k)
        for (int w = 0; w < kBlock / 64; ++w) {
            lo[k] = fminf(lo[k], sh[k][w]);
            hi[k] = fmaxf(hi[k], sh[3 + k][w]);
        }
}

__global__ void __launch_bounds__(kBlock) centroid_bounds(const crt_vertex* __restrict__ v,
                                                          const uint32_t* __restrict__ idx, int64_t n,
                                                          float* __restrict__ partial, uint32_t* __restrict__ supers,
                                                          int64_t super_words) {
    __shared__ float sh[6][kBlock / 64];
    const int64_t stride = int64_t(gridDim.x) * kBlock, first = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    for (int64_t w = first; w < super_words; w += stride) supers[w] = 0u;
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
    float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
#pragma unroll 2
    for (int64_t t = first; t < n; t += stride) {
        float c[3];
        centroid(tri_box(v, idx, t), c);
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(lo[k], c[k]);
            hi[k] = fmaxf(hi[k], c[k]);
        }
    }
    block_bounds(lo, hi, sh);
    if (threadIdx.x < 3) {
        const int k = int(threadIdx.x);
        partial[k * int64_t(gridDim.x) + blockIdx.x] = k == 0 ? lo[0] : k == 1 ? lo[1] : lo[2];
        partial[(3 + k) * int64_t(gridDim.x) + blockIdx.x] = k == 0 ? hi[0] : k == 1 ? hi[1] : hi[2];
    }
}

// 10 bits spread to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ __forceinline__ uint32_t quantize(float c, float lo, float scale) {
    const float x = ((c - lo) * scale) * 1024.0f;
    return uint32_t(fminf(fmaxf(x, 0.0f), 1023.0f));
}

// Radix sort of the codes by 8-bit digits (LSD, stable; the codes' 30 bits take
// 4 passes).  A tile is kTile codes of one workgroup, kItems per thread.  Pass
// p counts each tile's digits (counts[tile * kRadix + digit], and the sums over
// super-tiles of 2^super_log tiles), then scatters: the place of a tile's first
// code of digit d is the number of codes of smaller digits plus the number of
// d's in the tiles before it, which the tile adds up itself from the super-tile
// sums and the counts of its own super-tile (about 70 loads a thread, all
// independent).  That replaces the launch that scanned the counts; a decoupled
// look-back would replace the count as well, but every tile is resident at
// once here, so its chain over 1,250 tiles would cross the XCDs' caches link
// by link.
//
// Bound: launches and latency at a few thousand triangles, memory (16 bytes
// read, 8 written per code and pass) at millions.  2.56M codes: 110 us (20 a
// scatter, 7.5 a count); 8 passes of 4-bit digits with three launches each took
// 252 us.
constexpr int kDigitBits = 8;
constexpr int kRadix = 1 << kDigitBits;
constexpr int kItems = 8;
constexpr int kTile = kBlock * kItems;
constexpr int kWaves = kBlock / 64;
constexpr int kPasses = (kMortonBits + kDigitBits - 1) / kDigitBits;
static_assert(kRadix == kBlock, "a thread per digit");

// Writes a tile's digit counts (hist in LDS) and adds them to its super-tile's.
__device__ __forceinline__ void put_counts(const uint32_t* hist, int super_log, uint32_t* __restrict__ counts,
                                           uint32_t* __restrict__ supers) {
    const uint32_t c = hist[threadIdx.x];
    counts[int64_t(blockIdx.x) * kRadix + threadIdx.x] = c;
    if (c) atomicAdd(supers + int64_t(blockIdx.x >> super_log) * kRadix + threadIdx.x, c);
}

// Morton codes of one tile, and its digit counts for the first pass.
__global__ void __launch_bounds__(kBlock) morton(const crt_vertex* __restrict__ v, const uint32_t* __restrict__ idx,
                                                 int64_t n, const float* __restrict__ partial, int32_t nparts,
                                                 uint32_t* __restrict__ keys, int super_log,
                                                 uint32_t* __restrict__ counts, uint32_t* __restrict__ supers) {
    __shared__ float sh[6][kBlock / 64];
    __shared__ uint32_t hist[kRadix];
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
    float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    hist[threadIdx.x] = 0u;
    for (int32_t b = int32_t(threadIdx.x); b < nparts; b += kBlock)
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(lo[k], partial[k * nparts + b]);
            hi[k] = fmaxf(hi[k], partial[(3 + k) * nparts + b]);
        }
    block_bounds(lo, hi, sh);   // ends after a barrier, so hist is clear as well
    float scale[3];
    for (int k = 0; k < 3; ++k) {
        const float ext = hi[k] - lo[k];
        scale[k] = ext > 0.0f ? 1.0f / ext : 0.0f;   // 0 for a flat axis
    }
#pragma unroll 4
    for (int r = 0; r < kItems; ++r) {
        const int64_t t = int64_t(blockIdx.x) * kTile + r * kBlock + threadIdx.x;
        if (t >= n) break;
        float c[3];
        centroid(tri_box(v, idx, t), c);
        const uint32_t x = quantize(c[0], lo[0], scale[0]);
        const uint32_t y = quantize(c[1], lo[1], scale[1]);
        const uint32_t z = quantize(c[2], lo[2], scale[2]);
        const uint32_t key = (spread3(x) << 2) | (spread3(y) << 1) | spread3(z);
        keys[t] = key;
        atomicAdd(&hist[key & (kRadix - 1)], 1u);
    }
    __syncthreads();
    put_counts(hist, super_log, counts, supers);
}

__global__ void __launch_bounds__(kBlock) count_digits(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                       int super_log, uint32_t* __restrict__ counts,
                                                       uint32_t* __restrict__ supers) {
    __shared__ uint32_t hist[kRadix];
    hist[threadIdx.x] = 0u;
    __syncthreads();
    uint32_t key[kItems];
    const int64_t base = int64_t(blockIdx.x) * kTile + threadIdx.x;
#pragma unroll
    for (int r = 0; r < kItems; ++r) key[r] = base + r * kBlock < n ? keys[base + r * kBlock] : 0u;
#pragma unroll
    for (int r = 0; r < kItems; ++r)
        if (base + r * kBlock < n) atomicAdd(&hist[(key[r] >> shift) & (kRadix - 1)], 1u);
    __syncthreads();
    put_counts(hist, super_log, counts, supers);
}

// Exclusive prefixes of a and b over the workgroup's threads.
__device__ __forceinline__ void block_prefix2(uint32_t& a, uint32_t& b, uint32_t (&sh)[2][kWaves]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t ia = a, ib = b;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t oa = __shfl_up(ia, d, 64), ob = __shfl_up(ib, d, 64);
        if (lane >= d) {
            ia += oa;
            ib += ob;
        }
    }
    if (lane == 63) {
        sh[0][wave] = ia;
        sh[1][wave] = ib;
    }
    __syncthreads();
    uint32_t ba = 0u, bb = 0u;
    for (int w = 0; w < kWaves; ++w) {
        ba += w < wave ? sh[0][w] : 0u;
        bb += w < wave ? sh[1][w] : 0u;
    }
    a = ba + ia - a;
    b = bb + ib - b;
}

// Scatters one tile.  Wave w of the workgroup holds codes [w * 64 * kItems, ...)
// of the tile, 64 at a time in order; a code's rank among its digit's codes is
// the number that earlier rounds of its wave counted (wc), plus its lower lanes
// of the same digit (one ballot per digit bit), plus the earlier waves' totals.
// The tile is put into digit order in LDS first, so that codes of one digit
// leave as runs.  FIRST: the values are the codes' own indices.
template <bool FIRST>
__global__ void __launch_bounds__(kBlock) scatter_digits(const uint32_t* __restrict__ kin,
                                                         const uint32_t* __restrict__ vin, int64_t n, int shift,
                                                         int super_log, int32_t nsupers,
                                                         const uint32_t* __restrict__ counts,
                                                         const uint32_t* __restrict__ supers,
                                                         uint32_t* __restrict__ kout, uint32_t* __restrict__ vout) {
    __shared__ uint32_t wc[kWaves][kRadix];
    __shared__ uint32_t gofs[kRadix];
    __shared__ uint32_t lkey[kTile], lval[kTile];
    __shared__ uint32_t sh[2][kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t tile0 = int64_t(blockIdx.x) * kTile;
    const int64_t base = tile0 + wave * (64 * kItems) + lane;
    uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const int64_t i = base + r * 64;
        key[r] = i < n ? kin[i] : 0u;
        val[r] = FIRST ? uint32_t(i) : (i < n ? vin[i] : 0u);
    }
    // thread d: digit d's codes in all tiles, and in the tiles before this one
    uint32_t total = 0u, before = 0u;
    const int32_t mine = int32_t(blockIdx.x) >> super_log;
#pragma unroll 8
    for (int32_t k = 0; k < nsupers; ++k) {
        const uint32_t c = supers[int64_t(k) * kRadix + threadIdx.x];
        total += c;
        before += k < mine ? c : 0u;
    }
#pragma unroll 8
    for (int32_t t = mine << super_log; t < int32_t(blockIdx.x); ++t) before += counts[int64_t(t) * kRadix + threadIdx.x];
    for (int w = 0; w < kWaves; ++w) wc[w][threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = base + r * 64 < n;
        const uint32_t d = (key[r] >> shift) & (kRadix - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        // one wave's LDS accesses run in order, so every lane reads the count
        // before its digit's first lane adds this round's
        uint32_t old = 0u;
        if (valid) old = wc[wave][d];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers & below) == 0ull) wc[wave][d] = old + uint32_t(__popcll(peers));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        rank[r] = old + uint32_t(__popcll(peers & below));
    }
    __syncthreads();
    // thread d: digit d's start in the tile (local) and in the output (global)
    uint32_t in_tile = 0u;
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = wc[w][threadIdx.x];
        wc[w][threadIdx.x] = in_tile;
        in_tile += c;
    }
    uint32_t global = total, local = in_tile;
    block_prefix2(global, local, sh);
    for (int w = 0; w < kWaves; ++w) wc[w][threadIdx.x] += local;
    gofs[threadIdx.x] = global + before - local;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        if (base + r * 64 < n) {
            const uint32_t p = wc[wave][(key[r] >> shift) & (kRadix - 1)] + rank[r];
            lkey[p] = key[r];
            lval[p] = val[r];
        }
    }
    __syncthreads();
    const int32_t here = int32_t(n - tile0 < kTile ? n - tile0 : kTile);
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const int32_t p = r * kBlock + int32_t(threadIdx.x);
        if (p < here) {
            const uint32_t k = lkey[p];
            const uint32_t pos = gofs[(k >> shift) & (kRadix - 1)] + uint32_t(p);
            kout[pos] = k;
            vout[pos] = lval[p];
        }
    }
}

// Longest common prefix of the codes a at sorted index i and b at j (Karras's
// delta; equal codes are told apart by their indices).
__device__ __forceinline__ int prefix_len(uint32_t a, uint32_t b, int64_t i, int64_t j) {
    return a == b ? 32 + __clz(uint32_t(i ^ j)) : __clz(a ^ b);
}

// delta over the sorted codes in memory; -1 outside [0, n).
__device__ __forceinline__ int delta(const uint32_t* __restrict__ keys, int64_t n, int64_t i, uint32_t key_i,
                                     int64_t j) {
    if (j < 0 || j >= n) return -1;
    return prefix_len(key_i, keys[j], i, j);
}

// A node's box is the min / max over the triangle boxes of its leaf range,
// which min / max give exactly in any order and from overlapping parts, so the
// boxes equal a bottom-up union's bit for bit.
__device__ __forceinline__ Box unite(const Box& a, const Box& b) {
    Box u;
    for (int q = 0; q < 3; ++q) {
        u.lo[q] = fminf(a.lo[q], b.lo[q]);
        u.hi[q] = fmaxf(a.hi[q], b.hi[q]);
    }
    return u;
}

__device__ __forceinline__ Box empty_box() {
    Box b;
    for (int q = 0; q < 3; ++q) {
        b.lo[q] = __builtin_inff();
        b.hi[q] = -__builtin_inff();
    }
    return b;
}

// Union over the wave's lanes; every lane gets it.
__device__ __forceinline__ Box wave_unite(Box b) {
    for (int q = 0; q < 3; ++q) {
        b.lo[q] = wave_min(b.lo[q]);
        b.hi[q] = wave_max(b.hi[q]);
    }
    return b;
}

// Packed leaf word (start << 4 | count) as the stack layout stores it.
__device__ __forceinline__ int32_t leaf_word(int64_t start, int32_t count) {
    return int32_t((uint32_t(start) << 4) | uint32_t(count));
}

// Stack entry of an internal node whose children cover leaves [first, gamma]
// and [gamma + 1, last]: internal child c has index gamma or gamma + 1.
__device__ __forceinline__ void put_entry(crt_stack_node* __restrict__ out, int32_t t_offset, int64_t first,
                                          int64_t gamma, int64_t last, const Box& l, const Box& r) {
    const int64_t nl = gamma - first + 1, nr = last - gamma;
    const int32_t wl = nl <= 2 ? leaf_word(int64_t(t_offset) + first, int32_t(nl)) : -1;
    const int32_t wr = nr <= 2 ? leaf_word(int64_t(t_offset) + gamma + 1, int32_t(nr)) : -1;
    float4* o = reinterpret_cast<float4*>(out);
    o[0] = make_float4(l.lo[0], l.lo[1], l.lo[2], __int_as_float(wl));
    o[1] = make_float4(l.hi[0], l.hi[1], l.hi[2], __int_as_float(nl <= 2 ? 0 : int32_t(gamma)));
    o[2] = make_float4(r.lo[0], r.lo[1], r.lo[2], __int_as_float(wr));
    o[3] = make_float4(r.hi[0], r.hi[1], r.hi[2], __int_as_float(nr <= 2 ? 0 : int32_t(gamma + 1)));
}

// The tree, its boxes and its entries, a chunk of kChunk leaves per workgroup
// and a thread per leaf and internal node.  Karras's tree gives internal node
// i a leaf range with one end at i, so the code just outside the chunk on the
// range's side tells whether the range ends inside (delta falls with the
// distance).  Such a node finds its range and split by binary searches over
// the chunk's codes in LDS.  Its children's boxes are two windows each of a
// table of boxes over 2^k leaves, which is built level by level in two LDS
// buffers, a level's queries answered while it is there: 24 KB in all, so the
// CU keeps its 32 waves.  Nodes whose range leaves the chunk are marked in a
// bit mask for span_nodes (no list: its one counter took 300 us), which also
// reads the leaf boxes and 64-leaf boxes written here.
//
// Bound: the gathers of the sorted triangles' indices and vertices and the
// 64-byte entries (about 190 bytes a triangle).  2.56M triangles: 104 us, 4.7
// TB/s; one launch each for the tree, a bottom-up climb for the boxes and the
// entries took 71 + 230 + 110 us, with child, range, parent and four box arrays
// between.
constexpr int kChunkBits = 9;
constexpr int kChunk = 1 << kChunkBits;
static_assert(kChunk % 64 == 0 && kChunk / 64 <= 16, "a chunk is whole 64-leaf groups");

__global__ void __launch_bounds__(kChunk) chunk_nodes(const crt_vertex* __restrict__ v,
                                                      const uint32_t* __restrict__ idx,
                                                      const int32_t* __restrict__ mesh, int32_t mesh_all,
                                                      const uint32_t* __restrict__ keys,
                                                      const uint32_t* __restrict__ order, int64_t n, int32_t t_offset,
                                                      Box* __restrict__ leaf_box, Box* __restrict__ group_box,
                                                      uint64_t* __restrict__ span,
                                                      crt_stack_node* __restrict__ nodes,
                                                      crt_triangle* __restrict__ tris) {
    __shared__ uint32_t code[kChunk + 2];   // code[1 + k]: leaf base + k; one more at each end
    __shared__ float win[2][6][kChunk];     // boxes over 2^k leaves from each leaf, two levels
    const int64_t base = int64_t(blockIdx.x) * kChunk;
    const int li = int(threadIdx.x), lane = li & 63;
    const int64_t i = base + li;
    code[1 + li] = i < n ? keys[i] : 0u;
    if (li == 0) code[0] = base > 0 ? keys[base - 1] : 0u;
    if (li == kChunk - 1) code[kChunk + 1] = i + 1 < n ? keys[i + 1] : 0u;
    Box cur = empty_box();
    if (i < n) {
        const int64_t t = int64_t(order[i]);
        const uint32_t i0 = idx[3 * t + 0], i1 = idx[3 * t + 1], i2 = idx[3 * t + 2];
        const float4 p0 = *reinterpret_cast<const float4*>(v[i0].position);
        const float4 p1 = *reinterpret_cast<const float4*>(v[i1].position);
        const float4 p2 = *reinterpret_cast<const float4*>(v[i2].position);
        *reinterpret_cast<int4*>(tris + i) = make_int4(int32_t(i0), int32_t(i1), int32_t(i2), mesh ? mesh[t] : mesh_all);
        cur.lo[0] = fminf(fminf(p0.x, p1.x), p2.x);
        cur.lo[1] = fminf(fminf(p0.y, p1.y), p2.y);
        cur.lo[2] = fminf(fminf(p0.z, p1.z), p2.z);
        cur.hi[0] = fmaxf(fmaxf(p0.x, p1.x), p2.x);
        cur.hi[1] = fmaxf(fmaxf(p0.y, p1.y), p2.y);
        cur.hi[2] = fmaxf(fmaxf(p0.z, p1.z), p2.z);
        leaf_box[i] = cur;
    }
    for (int q = 0; q < 3; ++q) {
        win[0][q][li] = cur.lo[q];
        win[0][3 + q][li] = cur.hi[q];
    }
    __syncthreads();

    // node i's range and split, all in chunk positions (position p = leaf base + p)
    const uint32_t own = code[1 + li];
    auto dl = [&](int p) {   // delta(i, base + p), p in [-1, kChunk]
        const int64_t j = base + p;
        return j < 0 || j >= n ? -1 : prefix_len(own, code[1 + p], i, j);
    };
    bool here = false, spans = false;
    int first = 0, gamma = 0, last = 0;
    if (i < n - 1) {
        const int up = dl(li + 1), down = dl(li - 1);
        const int d = up - down >= 0 ? 1 : -1;
        const int dmin = d > 0 ? down : up;
        here = dl(d > 0 ? kChunk : -1) <= dmin;
        spans = !here;
        if (here) {
            int l = 0;
            for (int t = kChunk / 2; t >= 1; t /= 2) {
                const int p = li + (l + t) * d;
                if (p >= 0 && p < kChunk && dl(p) > dmin) l += t;
            }
            const int dnode = dl(li + l * d);
            int s = 0;
            for (int t = kChunk / 2; t >= 1; t /= 2) {
                const int p = li + (s + t) * d;
                if (s + t < l && dl(p) > dnode) s += t;
            }
            gamma = li + s * d + (d < 0 ? -1 : 0);
            first = d > 0 ? li : li - l;
            last = d > 0 ? li + l : li;
        }
    }
    const uint64_t ballot = __ballot(spans);
    if (lane == 0 && i < n) span[i >> 6] = ballot;

    // a range of m leaves is covered by two windows of 2^k, k = floor(log2 m)
    // (at most 2^(kChunkBits - 1), whose two windows cover a whole chunk)
    const int kl = here ? min(31 - __clz(gamma - first + 1), kChunkBits - 1) : -1;
    const int kr = here ? min(31 - __clz(last - gamma), kChunkBits - 1) : -1;
    Box bl = empty_box(), br = empty_box();
#pragma unroll 1
    for (int k = 0; k < kChunkBits; ++k) {
        const float(*w)[kChunk] = win[k & 1];
        auto window = [&](int p) {
            Box b;
            for (int q = 0; q < 3; ++q) {
                b.lo[q] = w[q][p];
                b.hi[q] = w[3 + q][p];
            }
            return b;
        };
        if (k == kl) bl = unite(window(first), window(gamma + 1 - (1 << k)));
        if (k == kr) br = unite(window(gamma + 1), window(last + 1 - (1 << k)));
        if (k == 6 && lane == 0 && i < n) group_box[i >> 6] = cur;
        if (k + 1 < kChunkBits) {
            if (li + (1 << k) < kChunk) cur = unite(cur, window(li + (1 << k)));
            float(*o)[kChunk] = win[(k + 1) & 1];
            for (int q = 0; q < 3; ++q) {
                o[q][li] = cur.lo[q];
                o[3 + q][li] = cur.hi[q];
            }
            __syncthreads();
        }
    }
    if (here) put_entry(nodes + i, t_offset, base + first, base + gamma, base + last, bl, br);
}

// Boxes of 64 groups (4,096 leaves), a wave each.
__global__ void __launch_bounds__(kBlock) super_boxes(const Box* __restrict__ group_box, int64_t groups,
                                                      Box* __restrict__ super_box) {
    const int lane = threadIdx.x & 63;
    const int64_t s = int64_t(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6);
    const int64_t g = s * 64 + lane;
    if (s * 64 >= groups) return;
    const Box b = wave_unite(g < groups ? group_box[g] : empty_box());
    if (lane == 0) super_box[s] = b;
}

// The span pass gives a node kTeam lanes, a DPP row: its searches probe kTeam
// places a round, and its reductions are row rotations without LDS.
constexpr int kTeam = 16;

template <int ROR>
__device__ __forceinline__ float row_ror(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + ROR, 0xF, 0xF, false));
}

// Union over the team's lanes (all active); every lane gets it.
__device__ __forceinline__ Box team_unite(Box b) {
    for (int q = 0; q < 3; ++q) {
        b.lo[q] = fminf(b.lo[q], row_ror<8>(b.lo[q]));
        b.lo[q] = fminf(b.lo[q], row_ror<4>(b.lo[q]));
        b.lo[q] = fminf(b.lo[q], row_ror<2>(b.lo[q]));
        b.lo[q] = fminf(b.lo[q], row_ror<1>(b.lo[q]));
        b.hi[q] = fmaxf(b.hi[q], row_ror<8>(b.hi[q]));
        b.hi[q] = fmaxf(b.hi[q], row_ror<4>(b.hi[q]));
        b.hi[q] = fmaxf(b.hi[q], row_ror<2>(b.hi[q]));
        b.hi[q] = fmaxf(b.hi[q], row_ror<1>(b.hi[q]));
    }
    return b;
}

// Team-wide count of a flag.
__device__ __forceinline__ int team_count(bool flag) {
    return __popc(uint32_t(__ballot(flag) >> (threadIdx.x & 48)) & 0xFFFFu);
}

// Box of leaves [a, b], formed by one team: the leaves of the two end groups,
// the groups of the two end super-groups and the super-groups between.
__device__ __forceinline__ Box range_box(const Box* __restrict__ leaf_box, const Box* __restrict__ group_box,
                                         const Box* __restrict__ super_box, int64_t a, int64_t b, int rank) {
    Box acc = empty_box();
    const int64_t ga = a >> 6, gb = b >> 6;
    for (int64_t k = a + rank; k <= min(b, (ga << 6) + 63); k += kTeam) acc = unite(acc, leaf_box[k]);
    if (gb > ga) {
        for (int64_t k = (gb << 6) + rank; k <= b; k += kTeam) acc = unite(acc, leaf_box[k]);
        // whole groups (ga, gb): by super-group where one lies whole between
        const int64_t g0 = ga + 1, g1 = gb - 1, sa = g0 >> 6, sb = g1 >> 6;
        for (int64_t k = g0 + rank; k <= min(g1, (sa << 6) + 63); k += kTeam) acc = unite(acc, group_box[k]);
        if (g0 <= g1 && sb > sa) {
            for (int64_t k = (sb << 6) + rank; k <= g1; k += kTeam) acc = unite(acc, group_box[k]);
            for (int64_t k = sa + 1 + rank; k < sb; k += kTeam) acc = unite(acc, super_box[k]);
        }
    }
    return team_unite(acc);
}

// Largest l in [lo, hi) with delta(i, i + l * d) > dmin, given that it holds at
// lo and fails at hi: the team's lanes probe kTeam distances per round.
__device__ __forceinline__ int64_t last_above(const uint32_t* __restrict__ keys, int64_t n, int64_t i, uint32_t key_i,
                                              int d, int dmin, int64_t lo, int64_t hi, int rank) {
    while (hi - lo > 1) {
        const int64_t step = (hi - lo + kTeam) / (kTeam + 1);   // probes lo + step, lo + 2 step, ..., below hi
        const int64_t l = lo + (rank + 1) * step;
        // delta falls with l, so the first c probes hold
        const int64_t c = team_count(l < hi && delta(keys, n, i, key_i, i + l * d) > dmin);
        lo += c * step;
        hi = min(hi, lo + step);
    }
    return lo;
}

// A workgroup per chunk, a team per listed node of the chunk: the node's range
// and split as chunk_nodes finds them, its children's boxes and its entry.  A
// chain of about ten dependent loads per node bounds it, so nodes have to be
// many at once: 45 us for 2.56M triangles, where a wave per node and chunks of
// 256 (twice the nodes) took 96.
__global__ void __launch_bounds__(kBlock) span_nodes(const uint32_t* __restrict__ keys, int64_t n, int32_t t_offset,
                                                     const uint64_t* __restrict__ span,
                                                     const Box* __restrict__ leaf_box,
                                                     const Box* __restrict__ group_box,
                                                     const Box* __restrict__ super_box,
                                                     crt_stack_node* __restrict__ nodes) {
    const int rank = int(threadIdx.x) % kTeam, team = int(threadIdx.x) / kTeam;
    // lane r of a team holds group r's mask and the listed nodes in the groups before it
    const int64_t g = int64_t(blockIdx.x) * (kChunk / 64) + rank;
    const uint64_t mask = rank < kChunk / 64 && g * 64 < n ? span[g] : 0ull;
    const int count = __popcll(mask);
    int incl = count;
    for (int k = 1; k < kTeam; k <<= 1) {
        const int o = __shfl_up(incl, k, kTeam);
        if (rank >= k) incl += o;
    }
    const int listed = __shfl(incl, kTeam - 1, kTeam);
    for (int e = team; e < listed; e += kBlock / kTeam) {
        // the group that holds the e-th listed node, and its bit
        const int group = team_count(incl <= e);
        int skip = e - __shfl(incl - count, group, kTeam);
        uint64_t m = uint64_t(uint32_t(__shfl(int(mask), group, kTeam))) |
                     uint64_t(uint32_t(__shfl(int(mask >> 32), group, kTeam))) << 32;
        for (; skip > 0; --skip) m &= m - 1;
        const int64_t i = (int64_t(blockIdx.x) * (kChunk / 64) + group) * 64 + __ffsll((long long)m) - 1;
        const uint32_t key_i = keys[i];
        const int up = delta(keys, n, i, key_i, i + 1), down = delta(keys, n, i, key_i, i - 1);
        const int d = up - down >= 0 ? 1 : -1;
        const int dmin = d > 0 ? down : up;
        // powers of two first: lane r probes distances 2^r and 2^(r + 16), below 2^30
        const bool near = delta(keys, n, i, key_i, i + (int64_t(1) << rank) * d) > dmin;
        const bool far = rank < 14 && delta(keys, n, i, key_i, i + (int64_t(65536) << rank) * d) > dmin;
        const int c = team_count(near) + team_count(far);   // >= 1: the neighbour on this side shares a longer prefix
        const int64_t l = last_above(keys, n, i, key_i, d, dmin, int64_t(1) << (c - 1), int64_t(1) << c, rank);
        const int64_t j = i + l * d;
        const int dnode = delta(keys, n, i, key_i, j);
        const int64_t s = last_above(keys, n, i, key_i, d, dnode, 0, l, rank);
        const int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
        const int64_t first = i < j ? i : j, last = i < j ? j : i;
        const Box bl = range_box(leaf_box, group_box, super_box, first, gamma, rank);
        const Box br = range_box(leaf_box, group_box, super_box, gamma + 1, last, rank);
        if (rank == 0) put_entry(nodes + i, t_offset, first, gamma, last, bl, br);
    }
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

struct Layout {
    size_t keys[2], vals[2], counts, supers, partial, leaf_box, group_box, super_box, span, bytes;
    int64_t tiles, nsupers, groups;
    int super_log;
    int32_t parts;   // workgroups of the bounds reduction
};

inline Layout layout(int64_t n) {
    const size_t un = size_t(n);
    Layout L{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align256(off + bytes);
        return at;
    };
    L.tiles = (n + kTile - 1) / kTile;
    // a tile adds up nsupers sums and up to 2^super_log counts: about the square root of the tiles each
    L.super_log = 4;
    while ((L.tiles >> (2 * L.super_log)) > 1) ++L.super_log;
    L.nsupers = ((L.tiles - 1) >> L.super_log) + 1;
    L.groups = (n + 63) / 64;
    L.parts = int32_t(std::min<int64_t>(kBoundsGrid, (n + kBlock - 1) / kBlock));
    L.keys[0] = take(un * 4);
    L.keys[1] = take(un * 4);
    L.vals[0] = take(un * 4);
    L.vals[1] = take(un * 4);
    L.counts = take(size_t(L.tiles) * kRadix * 4);
    L.supers = take(size_t(kPasses) * size_t(L.nsupers) * kRadix * 4);
    L.partial = take(size_t(L.parts) * 6 * 4);
    L.leaf_box = take(un * sizeof(Box));
    L.group_box = take(size_t(L.groups) * sizeof(Box));
    L.super_box = take(size_t((L.groups + 63) / 64) * sizeof(Box));
    L.span = take(size_t(L.groups) * 8);
    // at least 140 bytes a triangle, what callers have been told to reserve
    // (the arrays above take about 42)
    L.bytes = align256(std::max(off, un * 140));
    return L;
}

}  // namespace gb
}  // namespace crt

extern "C" {

size_t crt_build_bvh_gpu_workspace(int64_t ntris) {
    if (ntris < 2) return 0;
    return crt::gb::layout(ntris).bytes;
}

int crt_build_bvh_gpu(const crt_vertex* vertices, int64_t nverts, const uint32_t* indices, int64_t ntris,
                      const int32_t* mesh_ids, int32_t mesh_id, int32_t t_offset, crt_stack_node* nodes,
                      crt_triangle* triangles, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace crt::gb;
    if (!vertices || !indices || !nodes || !triangles || !workspace)
        return crt::set_error(CRT_E_INVALID, "crt_build_bvh_gpu: null argument");
    if (ntris < 2) return crt::set_error(CRT_E_INVALID, "crt_build_bvh_gpu: the stack layout needs >= 2 triangles");
    if (nverts <= 0 || nverts > 0xFFFFFFFFll) return crt::set_error(CRT_E_INVALID, "crt_build_bvh_gpu: bad vertex count");
    if (t_offset < 0 || uint64_t(ntris) + uint64_t(t_offset) >= (1ull << 28))
        return crt::set_error(CRT_E_INVALID, "crt_build_bvh_gpu: t_offset + triangles exceeds the 28-bit leaf start");
    const Layout L = layout(ntris);
    if (workspace_bytes < L.bytes || reinterpret_cast<uintptr_t>(workspace) % 256 != 0)
        return crt::set_error(CRT_E_INVALID, "crt_build_bvh_gpu: workspace must be 256-byte aligned and hold "
                                             "crt_build_bvh_gpu_workspace(ntris) = " + std::to_string(L.bytes) +
                                             " bytes");
    char* ws = static_cast<char*>(workspace);
    auto at = [&](size_t off) { return static_cast<void*>(ws + off); };
    uint32_t* keys[2] = {static_cast<uint32_t*>(at(L.keys[0])), static_cast<uint32_t*>(at(L.keys[1]))};
    uint32_t* vals[2] = {static_cast<uint32_t*>(at(L.vals[0])), static_cast<uint32_t*>(at(L.vals[1]))};
    auto* counts = static_cast<uint32_t*>(at(L.counts));
    auto* supers = static_cast<uint32_t*>(at(L.supers));
    auto* partial = static_cast<float*>(at(L.partial));
    auto* leaf_box = static_cast<Box*>(at(L.leaf_box));
    auto* group_box = static_cast<Box*>(at(L.group_box));
    auto* super_box = static_cast<Box*>(at(L.super_box));
    auto* span = static_cast<uint64_t*>(at(L.span));
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t n = ntris;
    const int64_t super_words = L.nsupers * kRadix;   // per pass

    hipLaunchKernelGGL(centroid_bounds, dim3(unsigned(L.parts)), dim3(kBlock), 0, st, vertices, indices, n, partial,
                       supers, kPasses * super_words);
    const dim3 nt(unsigned(L.tiles));
    hipLaunchKernelGGL(morton, nt, dim3(kBlock), 0, st, vertices, indices, n, partial, L.parts, keys[0], L.super_log,
                       counts, supers);
    int cur = 0;
    for (int pass = 0; pass < kPasses; ++pass) {
        const int shift = pass * kDigitBits;
        uint32_t* sums = supers + pass * super_words;
        if (pass > 0)
            hipLaunchKernelGGL(count_digits, nt, dim3(kBlock), 0, st, keys[cur], n, shift, L.super_log, counts, sums);
        if (pass == 0)
            hipLaunchKernelGGL(scatter_digits<true>, nt, dim3(kBlock), 0, st, keys[cur], vals[cur], n, shift,
                               L.super_log, int32_t(L.nsupers), counts, sums, keys[1 - cur], vals[1 - cur]);
        else
            hipLaunchKernelGGL(scatter_digits<false>, nt, dim3(kBlock), 0, st, keys[cur], vals[cur], n, shift,
                               L.super_log, int32_t(L.nsupers), counts, sums, keys[1 - cur], vals[1 - cur]);
        cur = 1 - cur;
    }
    const int64_t chunks = (n + kChunk - 1) / kChunk;
    hipLaunchKernelGGL(chunk_nodes, dim3(unsigned(chunks)), dim3(kChunk), 0, st, vertices, indices, mesh_ids, mesh_id,
                       keys[cur], vals[cur], n, t_offset, leaf_box, group_box, span, nodes, triangles);
    if (chunks > 1) {   // one chunk holds every node
        const int64_t super_groups = (L.groups + 63) / 64;
        hipLaunchKernelGGL(super_boxes, dim3(unsigned((super_groups + 3) / 4)), dim3(kBlock), 0, st, group_box,
                           L.groups, super_box);
        hipLaunchKernelGGL(span_nodes, dim3(unsigned(chunks)), dim3(kBlock), 0, st, keys[cur], n, t_offset, span,
                           leaf_box, group_box, super_box, nodes);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return crt::set_error(CRT_E_HIP, std::string("crt_build_bvh_gpu: kernel launch: ") + hipGetErrorString(e));
    return CRT_OK;
}

}  // extern "C"
