// Differentiable shading on top of the traversal: Cook-Torrance direct light
// from point lights plus one diffuse bounce, and its hand-written adjoint.
//
// Forward, per pixel with a primary hit p (triangle t0):
//   C = sum_l CT(p, l; albedo[t0], roughness[t0]) * vis_p(l)
//     + albedo[t0] * sum_l Lambert(q, l; albedo[t1]) * vis_q(l)
// where
//   CT       CookTorranceBRDF (Source/Core/Shaders/Include/CookTorranceBRDF.glsl:37-79)
//            with metalness 0: Lo = normalize(eye - p), Li = -normalize(p - L),
//            F = 0.04 + 0.96 (1 - max(0, Lh.Lo))^5, D = NDF, G = Smith-Schlick
//            with k = (r + 1)^2 / 8, kd = 1 - F,
//            (kd * albedo + F D G / max(1e-5, 4 NL NV)) * radiance * NL;
//   Lambert  GetDirect (Source/Core/Shaders/DiffuseTrace.glsl:368-372):
//            albedo * radiance * clamp(dot(N, Li), 0, 1);
//   radiance = I_l / |L - x|^2 (white point lights);
//   q        the closest hit of one cosine-weighted bounce ray from p
//            (CosWeightedHemisphere, Source/Core/Shaders/Include/Sampling.glsl:1-12,
//            per-pixel PCG uniforms), triangle t1;
//   vis      any-hit shadow rays from x + N * 1e-4 toward L with tmax = |L - x'|.
//
// Backward, loss = sum (C - T)^2: geometry (p, q, normals) comes from the
// forward records; visibility is re-traced, not stored.  Gradients of
// albedo[t0], roughness[t0], albedo[t1] and every intensity are summed over the
// lanes of a wave that share them, then in the workgroup's LDS, and reach memory
// by atomics: the two ground-plane triangles that cover half the image cost one
// per workgroup, not one per pixel.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "crt_internal.h"
#include "device_math.h"
#include "trace_launch.h"
#include "walker.h"

namespace crt {
namespace shade {

using namespace ::crt::dm;

constexpr int kMaxLights = 16;

// A workgroup of kWaves waves works on tiles of 64 pixels, one per lane, and
// deals a tile's rays (one bounce, a shadow ray from p and one from q to every
// light) to its waves one kind of ray at a time: a wave traces the same ray of
// all 64 pixels, which neighbours share most of.  The launch fills the device
// once, and workgroup b takes the tiles b, b + grid, ...
// Bound: VALU issue (80% of the forward pass; the boxes' tree stays in the
// caches).  One forward and backward pass over 1024 x 1024 pixels with 8 lights:
// 1,661 us with a wave per tile, each with its 17 rays in turn (waves of 135 to
// 560 us in two rounds, the chip half empty); 1,160 us as here, 1,295 when a
// lane's leaf is tested as soon as it is reached; 805 us with gradients met in
// LDS and one loop condition per node.  3 waves a tile take 6% more, 4 take 9%.
// An image of so few tiles that all fit the device at once with kWide waves each
// takes those: 64 x 64 pixels 204 -> 133 us, 192 x 192 224 -> 180 (launch_backward
// has the adjoint's).
constexpr int kWaves = 2, kWide = 8;
constexpr float kPi = 3.14159265359f;      // CookTorranceBRDF.glsl:7
constexpr float kOffset = 1e-4f;           // surface offset of secondary rays
constexpr float kTwoPi = 2.0f * 3.14159265359f;  // Sampling.glsl:3

struct Params {
    const float* albedo;
    const float* rough;
    const float* lpos;
    const float* inten;
    int32_t ntri;
    int32_t nl;
};

__device__ __forceinline__ f3 add(f3 a, f3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ f3 scale(f3 a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ f3 normalize(f3 a) { return scale(a, 1.0f / sqrtf(dot(a, a))); }

__device__ __forceinline__ f3 load3(const float* p, int32_t i) { return mk(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }

__device__ __forceinline__ uint32_t pcg(uint32_t v) {
    const uint32_t state = v * 747796405u + 2891336453u;
    const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}

// Face normal of triangle `tri`, turned to face against `dir`.
__device__ __forceinline__ f3 face_normal(const SceneArgs& s, int32_t tri, f3 dir) {
    const int4 tr = *reinterpret_cast<const int4*>(s.tris[tri].packed);
    const f3 a = vertex_pos(s.verts, tr.x), b = vertex_pos(s.verts, tr.y), c = vertex_pos(s.verts, tr.z);
    f3 n = normalize(cross(sub(b, a), sub(c, a)));
    if (dot(n, dir) > 0.0f) n = neg(n);
    return n;
}

constexpr int kStackLds = 16;   // stack layout: entries a lane keeps in LDS

template <int FORMAT, int BLOCK>
constexpr int stack_ints() {
    return FORMAT == CRT_FORMAT_STACK ? kStackLds * BLOCK : 1;
}

// The scene loop for one ray per lane (IntersectScene / its occlusion form,
// TraverseBVHStackless.glsl:280-366, :558-579): the hit triangle or -1, its
// distance in tmax.
template <int FORMAT, bool ANY, int BLOCK>
__device__ __forceinline__ int32_t trace(const SceneArgs& s, f3 org, f3 dir, float& tmax, int32_t* lds) {
    constexpr int kSpill = FORMAT == CRT_FORMAT_STACK ? sdev::spill_entries<kStackLds>() : 1;
    int32_t spill[kSpill];
    walker::Walker<FORMAT, kStackLds> w;
    w.init(lds, BLOCK, spill);
    w.tmax = tmax;
    int32_t hit = -1;
    for (int32_t i = 0; i < s.entity_count; ++i) {
        const crt_entity& e = s.entities[i];
        w.ro = xform(e.inverse, org, 1.0f);
        w.rd = xform(e.inverse, dir, 0.0f);
        w.inv = mk(1.0f / w.rd.x, 1.0f / w.rd.y, 1.0f / w.rd.z);
        w.begin(e.node_offset, e.node_count, s.total_nodes);
        while (w.leaves(s)) {
            int32_t leaf = w.leaf;
            while (true) {
                const int32_t first = leaf >> 4, end = first + (leaf & 0xF);
                for (int32_t k = first; k < end; ++k) {
                    const int4 tr = *reinterpret_cast<const int4*>(s.tris[k].packed);
                    const float t = tri_t(w.ro, w.rd, vertex_pos(s.verts, tr.x), vertex_pos(s.verts, tr.y),
                                          vertex_pos(s.verts, tr.z));
                    if (t > 0.0f && t < w.tmax) {
                        w.tmax = t;
                        hit = k;
                        if (ANY) break;
                    }
                }
                if ((ANY && hit >= 0) || leaf == w.leaf2 || w.leaf2 < 0) break;
                leaf = w.leaf2;
            }
            if (ANY && hit >= 0) break;
        }
        if (ANY && hit >= 0) break;
    }
    tmax = w.tmax;
    return hit;
}

template <int FORMAT, int BLOCK>
__device__ __forceinline__ bool visible(const SceneArgs& s, f3 x, f3 n, f3 light, int32_t* lds) {
    const f3 o = add(x, scale(n, kOffset));
    const f3 d = sub(light, o);
    float dist = sqrtf(dot(d, d));
    return trace<FORMAT, true, BLOCK>(s, o, scale(d, 1.0f / dist), dist, lds) < 0;
}

// Cook-Torrance terms of one light at x: f_c = A * (kd * albedo_c + spec),
// A = radiance * NL; also d(spec)/d(roughness).
struct CT {
    float A, kd, spec, dspec;
};

__device__ __forceinline__ CT cook_torrance(f3 x, f3 n, f3 eye, f3 light, float intensity, float r) {
    const f3 Lo = normalize(sub(eye, x));
    const f3 Li = neg(normalize(sub(x, light)));
    const f3 dl = sub(light, x);
    const float radiance = intensity / dot(dl, dl);
    const f3 Lh = normalize(add(Li, Lo));
    const float cosLo = fmaxf(0.0f, dot(n, Lo));
    const float cosLi = fmaxf(0.0f, dot(n, Li));
    const float dh = dot(n, Lh);
    const float cosLh = fmaxf(0.0f, dh);
    const float c = 1.0f - fmaxf(0.0f, dot(Lh, Lo));
    const float c5 = c * c * c * c * c;
    const float F = 0.04f + (1.0f - 0.04f) * c5;
    const float alpha = r * r;
    const float a2 = alpha * alpha;
    const float cl2 = cosLh * cosLh;
    // The NDF denominator cos^2 (a2 - 1) + 1 equals a2 cos^2 + sin^2.  Near a
    // highlight 1 - cos^2 cancels in FP32 (relative error ~1e-7 / sin^2, i.e.
    // 1e-3 at roughness 0.05), while |n x Lh|^2 gives sin^2 to rounding.  With
    // the half vector below the surface cos is clamped to 0 and den is 1.
    const f3 nh = cross(n, Lh);
    const float s2 = dh > 0.0f ? dot(nh, nh) : 1.0f;
    const float den = a2 * cl2 + s2;
    const float D = a2 / (kPi * den * den);
    const float dD_da2 = (s2 - a2 * cl2) / (kPi * den * den * den);   // (den - 2 a2 cos^2) / (pi den^3)
    const float dD = dD_da2 * 4.0f * r * r * r;
    const float k = (r + 1.0f) * (r + 1.0f) / 8.0f;
    const float dk = (r + 1.0f) / 4.0f;
    const float di = cosLi * (1.0f - k) + k;
    const float dv = cosLo * (1.0f - k) + k;
    const float Si = cosLi / di;
    const float So = cosLo / dv;
    const float dSi = -cosLi * (1.0f - cosLi) / (di * di);
    const float dSo = -cosLo * (1.0f - cosLo) / (dv * dv);
    const float G = Si * So;
    const float dG = (dSi * So + Si * dSo) * dk;
    const float q = fmaxf(1e-5f, 4.0f * cosLi * cosLo);
    CT t;
    t.A = radiance * cosLi;
    t.kd = 1.0f - F;
    t.spec = F * D * G / q;
    t.dspec = F * (dD * G + D * dG) / q;
    return t;
}

// Lambert term of one light at x: albedo * B, B = radiance * clamp(dot(n, Li), 0, 1).
__device__ __forceinline__ float lambert(f3 x, f3 n, f3 light, float intensity) {
    const f3 dl = sub(light, x);
    const float radiance = intensity / dot(dl, dl);
    const f3 Li = neg(normalize(sub(x, light)));
    return radiance * fminf(fmaxf(dot(n, Li), 0.0f), 1.0f);
}


// What the waves of a workgroup share of one tile.  Two of them take turns, so
// that one wave can finish a tile while the others trace the next.
struct Tile {
    unsigned long long vis_p[kMaxLights], vis_q[kMaxLights];   // per light, a bit per pixel
    int32_t next[2];                                           // rays claimed, per phase
    float q[3][64], nq[3][64];
    int32_t tri1[64];
};

// The next ray of a phase for the calling wave.
__device__ __forceinline__ int32_t claim(int32_t* counter) {
    int32_t k = 0;
    if (__lane_id() == 0) k = atomicAdd(counter, 1);
    return __builtin_amdgcn_readfirstlane(k);
}

__device__ __forceinline__ int32_t wave_id() { return __builtin_amdgcn_readfirstlane(int32_t(threadIdx.x >> 6)); }

template <int FORMAT, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) forward_kernel(SceneArgs s, const crt_ray* __restrict__ rays,
                                                             const crt_hit* __restrict__ hits, int64_t npix, Params P,
                                                             uint32_t seed, float* __restrict__ color,
                                                             crt_shade_record* __restrict__ rec) {
    constexpr int BLOCK = 64 * WAVES;
    __shared__ int32_t stack[stack_ints<FORMAT, BLOCK>()];
    __shared__ Tile tiles[2];
    int32_t* my = stack + (FORMAT == CRT_FORMAT_STACK ? threadIdx.x : 0);
    if (threadIdx.x < 4) tiles[threadIdx.x >> 1].next[threadIdx.x & 1] = 0;
    __syncthreads();
    const uint32_t lane = __lane_id();
    const int64_t ntiles = (npix + 63) / 64;
    int32_t turn = 0;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x, ++turn) {
        Tile& T = tiles[turn & 1];
        const int64_t i = tile * 64 + lane;
        int32_t t0 = -1;
        f3 eye = mk(0.0f, 0.0f, 0.0f), p = eye, n = eye;
        if (i < npix) {
            const crt_ray r = rays[i];
            const crt_hit h = hits[i];
            eye = mk(r.org[0], r.org[1], r.org[2]);
            if (h.t > 0.0f && h.tri >= 0) {
                const f3 dir = mk(r.dir[0], r.dir[1], r.dir[2]);
                t0 = h.tri;
                p = add(eye, scale(dir, h.t));
                n = face_normal(s, t0, dir);
            }
        }
        const bool any = __any(t0 >= 0);
        // the bounce, then p to every light
        for (int32_t k = any ? claim(&T.next[0]) : P.nl + 1; k <= P.nl; k = claim(&T.next[0])) {
            if (k == 0) {
                f3 q = mk(0.0f, 0.0f, 0.0f), nq = q;
                int32_t t1 = -1;
                if (t0 >= 0) {
                    // cosine-weighted bounce (Sampling.glsl:1-12) from per-pixel PCG uniforms
                    const uint32_t h1 = pcg(uint32_t(i) ^ (seed * 0x9E3779B9u));
                    const uint32_t h2 = pcg(h1);
                    const float u1 = float(h1 >> 8) * (1.0f / 16777216.0f);
                    const float u2 = float(h2 >> 8) * (1.0f / 16777216.0f);
                    f3 uu = cross(n, mk(0.0f, 1.0f, 1.0f));
                    if (dot(uu, uu) < 1e-12f) uu = cross(n, mk(1.0f, 0.0f, 0.0f));
                    uu = normalize(uu);
                    const f3 vv = cross(uu, n);
                    const float ra = sqrtf(u2);
                    const float rx = ra * cosf(kTwoPi * u1), ry = ra * sinf(kTwoPi * u1), rz = sqrtf(1.0f - u2);
                    const f3 bd = normalize(add(add(scale(uu, rx), scale(vv, ry)), scale(n, rz)));
                    const f3 bo = add(p, scale(n, kOffset));
                    float t = 1000000.0f;
                    t1 = trace<FORMAT, false, BLOCK>(s, bo, bd, t, my);
                    if (t1 >= 0) {
                        q = add(bo, scale(bd, t));
                        nq = face_normal(s, t1, bd);
                    }
                }
                T.tri1[lane] = t1;
                T.q[0][lane] = q.x;
                T.q[1][lane] = q.y;
                T.q[2][lane] = q.z;
                T.nq[0][lane] = nq.x;
                T.nq[1][lane] = nq.y;
                T.nq[2][lane] = nq.z;
            } else {
                const bool seen = t0 >= 0 && visible<FORMAT, BLOCK>(s, p, n, load3(P.lpos, k - 1), my);
                const unsigned long long m = __ballot(seen);
                if (lane == 0) T.vis_p[k - 1] = m;
            }
        }
        __syncthreads();
        int32_t t1 = -1;
        f3 q = mk(0.0f, 0.0f, 0.0f), nq = q;
        if (t0 >= 0) {
            t1 = T.tri1[lane];
            q = mk(T.q[0][lane], T.q[1][lane], T.q[2][lane]);
            nq = mk(T.nq[0][lane], T.nq[1][lane], T.nq[2][lane]);
        }
        // q to every light
        for (int32_t l = any ? claim(&T.next[1]) : P.nl; l < P.nl; l = claim(&T.next[1])) {
            const bool seen = t1 >= 0 && visible<FORMAT, BLOCK>(s, q, nq, load3(P.lpos, l), my);
            const unsigned long long m = __ballot(seen);
            if (lane == 0) T.vis_q[l] = m;
        }
        __syncthreads();
        // one wave, another each time, writes the tile's records and colors; the others go on
        if (wave_id() != turn % WAVES) continue;
        if (lane < 2) T.next[lane] = 0;
        if (i >= npix) continue;
        crt_shade_record out;
        uint32_t vis = 0;
        f3 c = mk(0.0f, 0.0f, 0.0f);
        if (t0 >= 0) {
            const f3 alb0 = load3(P.albedo, t0);
            const float r0 = P.rough[t0];
            const f3 alb1 = t1 >= 0 ? load3(P.albedo, t1) : mk(0.0f, 0.0f, 0.0f);
            float B1 = 0.0f;
            for (int32_t l = 0; l < P.nl; ++l) {
                const f3 L = load3(P.lpos, l);
                const float I = P.inten[l];
                if (T.vis_p[l] >> lane & 1ull) {
                    vis |= 1u << l;
                    const CT t = cook_torrance(p, n, eye, L, I, r0);
                    c = add(c, mk(t.A * (t.kd * alb0.x + t.spec), t.A * (t.kd * alb0.y + t.spec),
                                  t.A * (t.kd * alb0.z + t.spec)));
                }
                if (T.vis_q[l] >> lane & 1ull) {
                    vis |= 1u << (16 + l);
                    B1 += lambert(q, nq, L, I);
                }
            }
            c = add(c, mk(alb0.x * alb1.x * B1, alb0.y * alb1.y * B1, alb0.z * alb1.z * B1));
        }
        color[3 * i] = c.x;
        color[3 * i + 1] = c.y;
        color[3 * i + 2] = c.z;
        out.pad0 = out.pad1 = 0.0f;
        out.tri0 = t0;
        out.tri1 = t1;
        out.vis = vis;
        out.eye[0] = eye.x;
        out.eye[1] = eye.y;
        out.eye[2] = eye.z;
        out.p[0] = p.x;
        out.p[1] = p.y;
        out.p[2] = p.z;
        out.n[0] = n.x;
        out.n[1] = n.y;
        out.n[2] = n.z;
        out.q[0] = q.x;
        out.q[1] = q.y;
        out.q[2] = q.z;
        out.nq[0] = nq.x;
        out.nq[1] = nq.y;
        out.nq[2] = nq.z;
        rec[i] = out;
    }
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Gradients that several pixels of a wave add to one triangle meet in the
// workgroup's LDS first: a few triangles cover most of an image, and their
// global atomics queue up behind each other.  One entry per set; an entry that
// another triangle needs, and every entry at the end, goes to memory.
struct Gradients {
    static constexpr int kSets = 128;
    float v[kSets][4];   // albedo, roughness
    int32_t tri[kSets];

    __device__ __forceinline__ void flush(int k, float* __restrict__ g_albedo, float* __restrict__ g_rough) const {
        if (tri[k] < 0) return;
        for (int c = 0; c < 3; ++c) atomicAdd(g_albedo + 3 * int64_t(tri[k]) + c, v[k][c]);
        if (v[k][3] != 0.0f) atomicAdd(g_rough + tri[k], v[k][3]);
    }
    // Takes over entry k of another table.
    __device__ __forceinline__ void merge(int k, const Gradients& o, float* __restrict__ g_albedo,
                                          float* __restrict__ g_rough) {
        if (o.tri[k] < 0) return;
        if (tri[k] >= 0 && tri[k] != o.tri[k]) return o.flush(k, g_albedo, g_rough);
        for (int c = 0; c < 4; ++c) v[k][c] = tri[k] < 0 ? o.v[k][c] : v[k][c] + o.v[k][c];
        tri[k] = o.tri[k];
    }
    // One lane adds for triangle t.
    __device__ __forceinline__ void add(int32_t t, const float (&g)[4], float* __restrict__ g_albedo,
                                        float* __restrict__ g_rough) {
        const int k = t % kSets;
        const bool mine = tri[k] == t;
        if (!mine) flush(k, g_albedo, g_rough);
        tri[k] = t;
        for (int c = 0; c < 4; ++c) v[k][c] = mine ? v[k][c] + g[c] : g[c];
    }
};

// Adds v to the gradients of triangle idx (none below 0) for every lane; lanes
// that share a triangle are summed in-wave first.  Called by all lanes of a
// wave, by one wave at a time for the same table.
__device__ __forceinline__ void wave_scatter_add(Gradients& G, int32_t idx, const float (&v)[4],
                                                 float* __restrict__ g_albedo, float* __restrict__ g_rough) {
    unsigned long long pending = __ballot(idx >= 0);
    const unsigned lane = __lane_id();
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const int32_t lidx = __shfl(idx, leader);
        const bool mine = idx == lidx && idx >= 0;
        const unsigned long long m = __ballot(mine);
        if (m == (1ull << leader)) {
            // the leader alone holds this index: its own values, no reduction
            if (lane == unsigned(leader)) {
                for (int c = 0; c < 3; ++c) atomicAdd(g_albedo + 3 * int64_t(lidx) + c, v[c]);
                if (v[3] != 0.0f) atomicAdd(g_rough + lidx, v[3]);
            }
        } else {
            float sum[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) sum[k] = wave_sum(mine ? v[k] : 0.0f);
            if (lane == unsigned(leader)) G.add(lidx, sum, g_albedo, g_rough);
        }
        pending &= ~m;
    }
}

// The adjoint of a tile's pixels, one per lane of the wave (a lane without one
// has tri0 < 0), with the visibility its workgroup traced: albedo and
// roughness gradients are added to the triangles' entries, each light's
// intensity gradient, summed over the wave, to the workgroup's LDS sum.
__device__ __forceinline__ void adjoint(const Params& P, const crt_shade_record& R, int64_t i, const Tile& T,
                                        const float* __restrict__ color, const float* __restrict__ target,
                                        float* __restrict__ g_albedo, float* __restrict__ g_rough, Gradients& G,
                                        float* inten_sum) {
    const uint32_t lane = __lane_id();
    const bool valid = R.tri0 >= 0;
    const int32_t t0 = R.tri0;
    const int32_t t1 = valid ? R.tri1 : -1;
    const f3 p = mk(R.p[0], R.p[1], R.p[2]), n = mk(R.n[0], R.n[1], R.n[2]);
    const f3 eye = mk(R.eye[0], R.eye[1], R.eye[2]);
    const f3 q = mk(R.q[0], R.q[1], R.q[2]), nq = mk(R.nq[0], R.nq[1], R.nq[2]);
    f3 g = mk(0.0f, 0.0f, 0.0f), alb0 = g, alb1 = g;
    float r0 = 0.0f;
    if (valid) {
        g = mk(2.0f * (color[3 * i] - target[3 * i]), 2.0f * (color[3 * i + 1] - target[3 * i + 1]),
               2.0f * (color[3 * i + 2] - target[3 * i + 2]));
        alb0 = load3(P.albedo, t0);
        r0 = P.rough[t0];
        if (t1 >= 0) alb1 = load3(P.albedo, t1);
    }
    float SAkd0 = 0.0f, Sd0 = 0.0f, B1 = 0.0f;
    for (int32_t l = 0; l < P.nl; ++l) {
        float dI = 0.0f;
        const f3 L = load3(P.lpos, l);
        const float I = P.inten[l];
        if (T.vis_p[l] >> lane & 1ull) {
            const CT t = cook_torrance(p, n, eye, L, I, r0);
            SAkd0 += t.A * t.kd;
            Sd0 += t.A * t.dspec;
            dI += (g.x * t.A * (t.kd * alb0.x + t.spec) + g.y * t.A * (t.kd * alb0.y + t.spec) +
                   g.z * t.A * (t.kd * alb0.z + t.spec)) / I;
        }
        if (T.vis_q[l] >> lane & 1ull) {
            const float b = lambert(q, nq, L, I);
            B1 += b;
            dI += (g.x * alb0.x * alb1.x + g.y * alb0.y * alb1.y + g.z * alb0.z * alb1.z) * b / I;
        }
        const float sum = wave_sum(dI);
        if (lane == 0) atomicAdd(inten_sum + l, sum);
    }
    const float a0[4] = {g.x * (SAkd0 + alb1.x * B1), g.y * (SAkd0 + alb1.y * B1), g.z * (SAkd0 + alb1.z * B1),
                         (g.x + g.y + g.z) * Sd0};
    const float a1[4] = {g.x * alb0.x * B1, g.y * alb0.y * B1, g.z * alb0.z * B1, 0.0f};
    wave_scatter_add(G, valid ? t0 : -1, a0, g_albedo, g_rough);
    wave_scatter_add(G, t1, a1, g_albedo, g_rough);
}

// Waits until every wave of a tile's group has come here `round` times; the
// waves of a workgroup run at the same time, so each of them does.
template <int WAVES>
__device__ __forceinline__ void group_barrier(int32_t* arrived, int32_t round) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (__lane_id() == 0) __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (__hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < round * WAVES)
        __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// GROUPS tiles per workgroup, WAVES waves on each.  The sums that every pixel
// adds to (a light's intensity, the triangles that cover the image) leave a
// workgroup as one atomic each: one after the other at the same address, they
// are the kernel's bottleneck when every wave sends its own, and each rounds
// the growing sum once more, so few large workgroups are also more exact.
template <int FORMAT, int WAVES, int GROUPS>
__global__ void __launch_bounds__(64 * WAVES * GROUPS)
backward_kernel(SceneArgs s, const crt_shade_record* __restrict__ rec, int64_t npix, Params P,
                const float* __restrict__ color, const float* __restrict__ target, float* __restrict__ g_albedo,
                float* __restrict__ g_rough, float* __restrict__ g_inten) {
    constexpr int BLOCK = 64 * WAVES * GROUPS;
    __shared__ int32_t stack[stack_ints<FORMAT, BLOCK>()];
    __shared__ Tile tiles[GROUPS][2];
    __shared__ Gradients G[GROUPS];
    __shared__ float inten_sum[kMaxLights];
    __shared__ int32_t arrived[GROUPS];
    int32_t* my = stack + (FORMAT == CRT_FORMAT_STACK ? threadIdx.x : 0);
    if (threadIdx.x < unsigned(kMaxLights)) inten_sum[threadIdx.x] = 0.0f;
    if (threadIdx.x < 2 * GROUPS) tiles[threadIdx.x >> 1][threadIdx.x & 1].next[0] = 0;
    if (threadIdx.x < GROUPS) arrived[threadIdx.x] = 0;
    for (int k = threadIdx.x; k < GROUPS * Gradients::kSets; k += BLOCK)
        G[k / Gradients::kSets].tri[k % Gradients::kSets] = -1;
    __syncthreads();
    const uint32_t lane = __lane_id();
    const int32_t group = wave_id() / WAVES, wave = wave_id() % WAVES;
    const int64_t ntiles = (npix + 63) / 64;
    int32_t turn = 0;
    for (int64_t tile = int64_t(group) * gridDim.x + blockIdx.x; tile < ntiles; tile += int64_t(gridDim.x) * GROUPS, ++turn) {
        Tile& T = tiles[group][turn & 1];
        const int64_t i = tile * 64 + lane;
        // every field is initialized: with some left undefined for the lanes past
        // the end, the compiler may assume that there are none and drop the bound
        crt_shade_record R{};
        R.tri0 = R.tri1 = -1;
        if (i < npix) R = rec[i];
        const bool valid = R.tri0 >= 0;
        const bool again = valid && R.tri1 >= 0;
        const bool any = __any(valid);
        for (int32_t k = any ? claim(&T.next[0]) : 2 * P.nl; k < 2 * P.nl; k = claim(&T.next[0])) {
            const bool first = k < P.nl;
            const int32_t l = first ? k : k - P.nl;
            const float* x = first ? R.p : R.q;
            const float* xn = first ? R.n : R.nq;
            const bool seen = (first ? valid : again) &&
                              visible<FORMAT, BLOCK>(s, mk(x[0], x[1], x[2]), mk(xn[0], xn[1], xn[2]), load3(P.lpos, l), my);
            const unsigned long long m = __ballot(seen);
            if (lane == 0) (first ? T.vis_p : T.vis_q)[l] = m;
        }
        group_barrier<WAVES>(&arrived[group], turn + 1);
        // one wave, another each time, takes the tile's gradients; the others go on
        if (wave != turn % WAVES) continue;
        if (lane == 0) T.next[0] = 0;
        if (any) adjoint(P, R, i, T, color, target, g_albedo, g_rough, G[group], inten_sum);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < Gradients::kSets; k += BLOCK) {
        for (int g = 1; g < GROUPS; ++g) G[0].merge(k, G[g], g_albedo, g_rough);
        G[0].flush(k, g_albedo, g_rough);
    }
    if (threadIdx.x < unsigned(P.nl)) atomicAdd(g_inten + threadIdx.x, inten_sum[threadIdx.x]);
}

// Workgroups of `block` threads that fill the device once.
template <typename F>
int64_t resident(F kernel, int block) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), block, 0) !=
            hipSuccess || per_cu <= 0)
        per_cu = 1;
    return int64_t(cus) * per_cu;
}

template <int FORMAT>
void launch_forward(const SceneArgs& s, const crt_ray* rays, const crt_hit* hits, int64_t npix, const Params& P,
                    uint32_t seed, float* color, crt_shade_record* rec, hipStream_t st) {
    const int64_t tiles = (npix + 63) / 64;
    const auto wide = forward_kernel<FORMAT, kWide>;
    const auto fn = forward_kernel<FORMAT, kWaves>;
    if (tiles <= resident(wide, 64 * kWide)) {
        hipLaunchKernelGGL(wide, dim3(unsigned(tiles)), dim3(64 * kWide), 0, st, s, rays, hits, npix, P, seed, color, rec);
        return;
    }
    const int64_t grid = resident(fn, 64 * kWaves);
    hipLaunchKernelGGL(fn, dim3(unsigned(tiles < grid ? tiles : grid)), dim3(64 * kWaves), 0, st, s, rays, hits, npix, P,
                       seed, color, rec);
}

// Waves a tile, and tiles a workgroup, of the adjoint.  A workgroup holds at
// least two tiles, so that a light's gradient takes one addition per 128 pixels
// or fewer: with one (64 pixels an addition) the rounding of an image of 128 x
// 128 pixels was 1.4 times as large.  The most waves with which all tiles are
// resident at once; kMid by the registers (six waves per SIMD over the
// stackless layout, five over the stack layout).  64 x 64 pixels take 50 us with
// 8 waves a tile, 54 with 6, 63 with 4; 192 x 192 pixels 57 with 6, 65 with 4, 100
// with 2, where 8 no longer fit; over the stack layout 103 with 4, 175 with 2.
template <int FORMAT>
void launch_backward(const SceneArgs& s, const crt_shade_record* rec, int64_t npix, const Params& P,
                     const float* color, const float* target, float* g_albedo, float* g_rough, float* g_inten,
                     hipStream_t st) {
    constexpr int kMid = FORMAT == CRT_FORMAT_STACKLESS ? 6 : 4, kGroups = 4;
    const int64_t tiles = (npix + 63) / 64;
    const auto launch = [&](auto fn, int waves, int groups, bool all) {
        const int64_t need = (tiles + groups - 1) / groups, grid = resident(fn, 64 * waves * groups);
        if (all && need > grid) return false;
        hipLaunchKernelGGL(fn, dim3(unsigned(need < grid ? need : grid)), dim3(unsigned(64 * waves * groups)), 0, st, s,
                           rec, npix, P, color, target, g_albedo, g_rough, g_inten);
        return true;
    };
    if (launch(backward_kernel<FORMAT, kWide, 2>, kWide, 2, true)) return;
    if (launch(backward_kernel<FORMAT, kMid, 2>, kMid, 2, true)) return;
    launch(backward_kernel<FORMAT, kWaves, kGroups>, kWaves, kGroups, false);
}

}  // namespace shade
}  // namespace crt

namespace {

int shade_args(const crt_scene_view* scene, const crt_shade_params* params, crt::SceneArgs& a, crt::shade::Params& p) {
    if (!scene || !params) return crt::set_error(CRT_E_INVALID, "shade: null scene or params");
    if (scene->format != CRT_FORMAT_STACKLESS && scene->format != CRT_FORMAT_STACK)
        return crt::set_error(CRT_E_INVALID, "shade: unknown node format");
    if (params->nlights < 1 || params->nlights > crt::shade::kMaxLights)
        return crt::set_error(CRT_E_INVALID, "shade: nlights must be 1..16");
    if (!params->albedo || !params->roughness || !params->light_pos || !params->intensity || params->ntri <= 0)
        return crt::set_error(CRT_E_INVALID, "shade: null parameter buffer");
    a = crt::scene_args(*scene);
    p = crt::shade::Params{params->albedo, params->roughness, params->light_pos, params->intensity, params->ntri,
                           params->nlights};
    return CRT_OK;
}

}  // namespace

extern "C" {

int crt_shade_forward(const crt_scene_view* scene, const crt_ray* primary_rays, const crt_hit* primary_hits,
                      int64_t npix, const crt_shade_params* params, uint32_t seed, float* color,
                      crt_shade_record* records, void* stream) {
    crt::SceneArgs a;
    crt::shade::Params p;
    int rc = shade_args(scene, params, a, p);
    if (rc) return rc;
    if (npix < 0 || (npix > 0 && (!primary_rays || !primary_hits || !color || !records)))
        return crt::set_error(CRT_E_INVALID, "crt_shade_forward: bad buffers");
    if (npix == 0) return CRT_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a.format == CRT_FORMAT_STACKLESS)
        crt::shade::launch_forward<CRT_FORMAT_STACKLESS>(a, primary_rays, primary_hits, npix, p, seed, color, records, st);
    else
        crt::shade::launch_forward<CRT_FORMAT_STACK>(a, primary_rays, primary_hits, npix, p, seed, color, records, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return crt::set_error(CRT_E_HIP, std::string("crt_shade_forward: ") + hipGetErrorString(e));
    return CRT_OK;
}

int crt_shade_backward(const crt_scene_view* scene, const crt_shade_record* records, int64_t npix,
                       const crt_shade_params* params, const float* color, const float* target, float* grad_albedo,
                       float* grad_roughness, float* grad_intensity, void* stream) {
    crt::SceneArgs a;
    crt::shade::Params p;
    int rc = shade_args(scene, params, a, p);
    if (rc) return rc;
    if (npix < 0 || (npix > 0 && (!records || !color || !target || !grad_albedo || !grad_roughness ||
                                  !grad_intensity)))
        return crt::set_error(CRT_E_INVALID, "crt_shade_backward: bad buffers");
    if (npix == 0) return CRT_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a.format == CRT_FORMAT_STACKLESS)
        crt::shade::launch_backward<CRT_FORMAT_STACKLESS>(a, records, npix, p, color, target, grad_albedo,
                                                          grad_roughness, grad_intensity, st);
    else
        crt::shade::launch_backward<CRT_FORMAT_STACK>(a, records, npix, p, color, target, grad_albedo, grad_roughness,
                                                      grad_intensity, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return crt::set_error(CRT_E_HIP, std::string("crt_shade_backward: ") + hipGetErrorString(e));
    return CRT_OK;
}

}  // extern "C"
