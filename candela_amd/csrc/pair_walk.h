// One wave traces up to 64 rays (one per lane) through a stackless BVH that a
// context holds a second time as child pairs.
//
// Per ray the visits, tests and results are those of IntersectBVHStackless /
// IntersectBVHStacklessOcclusion inside the IntersectScene entity loop
// (Source/Core/Shaders/Intersectors/Include/TraverseBVHStackless.glsl:175-366,
// :463-579): left child first, and every box against the TMax that holds when
// the reference visits it.  The stackless array gives one box per dependent
// fetch (about 122 of them per bounce ray over 2.56M triangles), and the walk
// is bound by that chain, not by arithmetic or bandwidth.  A pair entry holds
// both children of an inner node, so a walk has one fetch per inner node it
// enters, about half as many; a triangle record (48 B) holds its positions, so
// a leaf is one fetch instead of index, then vertices.
//
// A right child's box is tested together with its left sibling's, before the
// left subtree is walked.  That gives the visit's own result: with tmin and
// far the box's entry and exit distances,
//     RayBounds(TMax) > 0 and < TMax   <=>   !(far < tmin) and tmin < TMax
// (tmin >= 1e-4; a NaN far drops out of min and max on both sides), so the
// pending child keeps tmin, or infinity for far < tmin, and is compared with
// the TMax of the time its turn comes.
//
// A closest-hit walk counts two visits per pair it enters.  A walk that ends
// has visited exactly those nodes, but until its end the count runs ahead of
// the reference's, so a lane that exceeds the iteration cap starts its ray
// again with `exact` set.  Then, and in an any-hit walk, which ends with
// pending children unvisited, a right child is kept hit or not while its left
// sibling's subtree is walked, and counted and checked against the cap when
// its turn comes.  A ray is walked in one of the two ways from its start to its
// end, whatever the other lanes of its wave do: what one has counted and kept,
// the other cannot go on from.
//
// Bound: the chain of a wave's longest ray (511 visits among the bounce rays
// below, 0.3 us a visit when alone), then VALU issue.  Measured against the
// walk of the stackless array: 347,053 bounce rays over 640,000 triangles 422 ->
// 214 us (of another view 541 -> 265), 1920 x 1080 primary rays of the same scene
// 671 -> 343 us (with 8 x 8 pixels a wave), 300 rays over 3,074 triangles 52 -> 25
// us (one ray a wave).  Both loads of a pair have to be in flight at once (pin):
// with the right box loaded behind the left one's branch, where the compiler moves
// it, the walk takes 1.5 to 1.8 times as long.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "device_math.h"
#include "trace_launch.h"

namespace crt {
namespace pair {

using namespace ::crt::dm;

// A pending or current child: ~index of its pair entry when it is an inner
// node, its packed leaf (start << 4 | count) when it is a leaf.
// The other values say what the lane waits for.
constexpr int32_t kDone = INT32_MIN;       // the walk is over: its end
constexpr int32_t kIdle = INT32_MIN + 1;   // no ray
constexpr int32_t kNone = INT32_MIN + 2;   // the next pending child

template <int D>
constexpr int spill_entries() {
    return kPairStack - D > 0 ? kPairStack - D : 1;
}

// One lane's pending children: D entries in LDS, the rest in scratch.
template <int D>
struct PairStack {
    typedef int32_t Entry __attribute__((ext_vector_type(2)));
    using LdsEntry = __attribute__((address_space(3))) Entry;
    Entry* lds;
    int32_t stride;
    Entry* spill;
    __device__ __forceinline__ LdsEntry* col() const { return (LdsEntry*)lds; }   // see LdsInt
    // Entries beyond the LDS part are rare: one uniform test skips the scratch code.
    __device__ __forceinline__ void put(int32_t sp, int32_t ref, float t) {
        const Entry v = {ref, __float_as_int(t)};
        if (!__any(sp >= D)) {
            col()[sp * stride] = v;
        } else if (sp < D) {
            col()[sp * stride] = v;
        } else {
            spill[sp - D] = v;
        }
    }
    __device__ __forceinline__ Entry get(int32_t sp) const {
        if (!__any(sp >= D)) return col()[sp * stride];
        return sp < D ? col()[sp * stride] : spill[sp - D];
    }
};

// Entry distance of a box, infinity when the ray passes it by (see the top).
__device__ __forceinline__ float entry(float4 bmin, float4 bmax, f3 ro, f3 inv) {
    const float t0x = (bmin.x - ro.x) * inv.x, t0y = (bmin.y - ro.y) * inv.y, t0z = (bmin.z - ro.z) * inv.z;
    const float t1x = (bmax.x - ro.x) * inv.x, t1y = (bmax.y - ro.y) * inv.y, t1z = (bmax.z - ro.z) * inv.z;
    const float tmin = mx(mx(mx(mn(t0x, t1x), mn(t0y, t1y)), mn(t0z, t1z)), 0.0001f);
    const float far = mn(mx(t0x, t1x), mn(mx(t0y, t1y), mx(t0z, t1z)));
    return far < tmin ? __builtin_inff() : tmin;
}

template <bool ANY, int D, int INNER, int LEAF_BATCH>
struct PairWave {
    f3 ro, rd, inv;        // ray in the current entity's space
    float tmax;            // walk TMax (closest: shrinks with every hit)
    float ray_tmax;
    int32_t slot, ent, hit_ent;
    int32_t ref, sp, it;
    int32_t tri, mesh;
    uint32_t status, visits;
    bool exact, redo;

    __device__ __forceinline__ bool stepping() const { return uint32_t(ref) - uint32_t(kNone) < 0u - uint32_t(kNone); }
    __device__ __forceinline__ bool leafing() const { return ref >= 0; }

    // Next entity that takes part; false when the entity loop is over.
    __device__ __forceinline__ bool begin_walk(const PairScene& s, const crt_ray* rays, uint32_t flags) {
        int32_t e = ent + 1;
        while (e < s.entity_count && (flags & CRT_FLAG_IGNORE_TRANSPARENT) &&
               __int_as_float(s.entities[e].data[1]) < 0.99f)
            ++e;
        ent = e;
        if (e >= s.entity_count) return false;
        const crt_entity& en = s.entities[e];
        const float4* rp = reinterpret_cast<const float4*>(rays + slot);
        const float4 a = rp[0], b = rp[1];
        ro = xform(en.inverse, mk(a.x, a.y, a.z), 1.0f);
        rd = xform(en.inverse, mk(b.x, b.y, b.z), 0.0f);
        inv = mk(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
        if (ANY) tmax = ray_tmax;
        const int32_t start = en.node_offset;
        const float4 rmin = s.nodes[2 * int64_t(start)], rmax = s.nodes[2 * int64_t(start) + 1];
        const int32_t packed = __float_as_int(rmin.w);
        it = 1;
        sp = 0;
        ref = entry(rmin, rmax, ro, inv) < tmax ? (packed == -1 ? ~pair_base(start) : packed) : kNone;
        return true;
    }

    __device__ __forceinline__ void begin_ray(const PairScene& s, const crt_ray* rays, crt_hit* __restrict__ hits,
                                              int64_t i, uint32_t flags) {
        slot = int32_t(i);
        ray_tmax = rays[i].tmax;
        exact = false;
        redo = false;
        reset();
        if (!begin_walk(s, rays, flags)) {
            finish(s, rays, hits, flags);
            ref = kIdle;
        }
    }

    __device__ __forceinline__ void reset() {
        tmax = ray_tmax;
        ent = hit_ent = -1;
        tri = mesh = -1;
        status = visits = 0;
    }

    __device__ __forceinline__ void finish(const PairScene& s, const crt_ray* rays, crt_hit* __restrict__ hits,
                                           uint32_t flags) {
        float4 tuvw = make_float4(-1.0f, -1.0f, -1.0f, -1.0f);
        // ClosestT > 0 exactly when a triangle was accepted; its t is then tmax
        const float closest = tri >= 0 ? tmax : -1.0f;
        if (ANY) {
            if (tri >= 0) tuvw.x = closest;
        } else {
            const bool ok = closest > 0.0f && ((flags & CRT_FLAG_TRI0_IS_MISS) ? tri > 0 : tri >= 0);
            if (ok) {
                const crt_entity& e = s.entities[hit_ent];
                const float4* rp = reinterpret_cast<const float4*>(rays + slot);
                const float4 a = rp[0], b = rp[1];
                const f3 lro = xform(e.inverse, mk(a.x, a.y, a.z), 1.0f);
                const f3 lrd = xform(e.inverse, mk(b.x, b.y, b.z), 0.0f);
                const float4* r = s.records + 3 * int64_t(tri);
                const float4 va = r[0], vb = r[1], vc = r[2];
                const f3 p = mk(lro.x + lrd.x * closest, lro.y + lrd.y * closest, lro.z + lrd.z * closest);
                const f3 uvw = barycentrics(p, mk(va.x, va.y, va.z), mk(vb.x, vb.y, vb.z), mk(vc.x, vc.y, vc.z));
                tuvw = make_float4(closest, uvw.x, uvw.y, uvw.z);
            }
        }
        float4* o = reinterpret_cast<float4*>(hits + slot);
        o[0] = tuvw;
        o[1] = make_float4(__int_as_float(tri), __int_as_float(mesh), __int_as_float(hit_ent),
                           __uint_as_float(pack_status(visits, status)));
    }

    // One step of a closest-hit walk: the next pending child whose box still
    // lies before TMax, then, when it is an inner node, its pair.
    __device__ __forceinline__ void step(const PairScene& s, int32_t max_iter, PairStack<D>& st) {
        if (ref == kNone) {
            ref = kDone;
            while (sp > 0) {
                const auto e = st.get(--sp);
                if (__int_as_float(e.y) < tmax) {
                    ref = e.x;
                    break;
                }
            }
        }
        if (ref < 0 && ref != kDone) {
            const float4* p = s.pairs + 4 * int64_t(~ref);
            float4 lmin = p[0], lmax = p[1], rmin = p[2], rmax = p[3];
            pin(lmin);
            pin(lmax);
            pin(rmin);
            pin(rmax);
            const float tl = entry(lmin, lmax, ro, inv), tr = entry(rmin, rmax, ro, inv);
            const int32_t rref = __float_as_int(rmin.w);
            const bool lhit = tl < tmax, rhit = tr < tmax;
            if (lhit && rhit) {
                st.put(sp, rref, tr);
                sp++;
            }
            ref = lhit ? __float_as_int(lmin.w) : rhit ? rref : kNone;
            it += 2;
            if (it > max_iter) {   // counted ahead: perhaps not yet, so the ray starts once more
                redo = true;
                ref = kDone;
            }
        }
    }

    // The same with every visit counted in its turn.
    __device__ __forceinline__ void step_in_order(const PairScene& s, int32_t max_iter, PairStack<D>& st) {
        if (ref == kNone) {
            ref = kDone;
            while (sp > 0) {
                if (it >= max_iter) {
                    status |= CRT_STATUS_ITER_CAP;
                    break;
                }
                it++;
                const auto e = st.get(--sp);
                if (__int_as_float(e.y) < tmax) {
                    ref = e.x;
                    break;
                }
            }
        }
        if (ref < 0 && ref != kDone) {
            const float4* p = s.pairs + 4 * int64_t(~ref);
            float4 lmin = p[0], lmax = p[1], rmin = p[2], rmax = p[3];
            pin(lmin);
            pin(lmax);
            pin(rmin);
            pin(rmax);
            const float tl = entry(lmin, lmax, ro, inv), tr = entry(rmin, rmax, ro, inv);
            const int32_t rref = __float_as_int(rmin.w);
            const bool lhit = tl < tmax, rhit = tr < tmax;
            if (lhit) {
                st.put(sp, rref, tr);
                sp++;
            }
            // visited now: the left child, and the right one unless the walk enters the left
            ref = lhit ? __float_as_int(lmin.w) : rhit ? rref : kNone;
            it += lhit ? 1 : 2;
            if (it > max_iter) {
                it = max_iter;
                status |= CRT_STATUS_ITER_CAP;
                ref = kDone;
            }
        }
    }

    // Tests the two records at p and p + second (second 0: the same once more, which changes nothing).
    __device__ __forceinline__ bool test(const float4* p, int32_t idx, int32_t second) {
        const float4* q = p + 3 * second;
        const float4 a0 = p[0], b0 = p[1], c0 = p[2];
        float4 a1 = q[0], b1 = q[1], c1 = q[2];
        pin(a1);
        pin(b1);
        pin(c1);
        const float t0 = tri_t(ro, rd, mk(a0.x, a0.y, a0.z), mk(b0.x, b0.y, b0.z), mk(c0.x, c0.y, c0.z));
        const float t1 = tri_t(ro, rd, mk(a1.x, a1.y, a1.z), mk(b1.x, b1.y, b1.z), mk(c1.x, c1.y, c1.z));
        const bool h0 = t0 > 0.0f && t0 < tmax;
        if (h0) {
            tmax = t0;
            mesh = __float_as_int(b0.w);
            tri = idx;
            hit_ent = ent;
        }
        const bool h1 = t1 > 0.0f && t1 < tmax && !(ANY && h0);
        if (h1) {
            tmax = t1;
            mesh = __float_as_int(b1.w);
            tri = idx + second;
            hit_ent = ent;
        }
        return ANY && (h0 || h1);
    }

    // One round of the wave: node phase, leaf phase.
    __device__ __forceinline__ void round(const PairScene& s, int32_t max_iter, PairStack<D>& st) {
        // every lane by its own `exact`: the two count and keep pending children differently
        const bool some_exact = ANY || __any(exact && ref != kIdle);
        for (int k = 0; k < INNER; ++k) {
            if (!ANY && stepping() && !exact) step(s, max_iter, st);
            if (some_exact && stepping() && (ANY || exact)) step_in_order(s, max_iter, st);
            if (!__any(stepping()) || __popcll(__ballot(leafing())) >= LEAF_BATCH) break;
        }
        if (leafing()) {
            const int32_t first = ref >> 4, end = first + (ref & 0xF);
            ref = kNone;
            for (int32_t i = first; i < end; i += 2) {
                if (test(s.records + 3 * int64_t(i), i, i + 1 < end ? 1 : 0)) {
                    ref = kDone;
                    break;
                }
            }
        }
    }

    // Walk ends: the next entity or the ray's result.
    __device__ __forceinline__ void walk_ends(const PairScene& s, const crt_ray* rays, crt_hit* __restrict__ hits,
                                              uint32_t flags) {
        // the ends run once kWalkEndBatch lanes wait or no lane can step
        const unsigned long long ends = __ballot(ref == kDone);
        if (ends && (__popcll(ends) >= kWalkEndBatch || !__any(stepping()))) {
            if (ref == kDone) {
                visits += uint32_t(it);
                bool fin = ANY && tri >= 0;   // any hit: the first entity with a hit ends the scene loop
                if (redo) {
                    redo = false;
                    exact = true;
                    fin = false;
                    reset();
                }
                if (!fin) fin = !begin_walk(s, rays, flags);
                if (fin) {
                    finish(s, rays, hits, flags);
                    ref = kIdle;
                }
            }
        }
    }

    // Ray i per lane (i < 0: idle) until every lane is done.
    __device__ __forceinline__ void run(const PairScene& s, const crt_ray* rays, crt_hit* __restrict__ hits, int64_t i,
                                        uint32_t flags, int32_t max_iter, PairStack<D> st) {
        ref = kIdle;
        exact = false;
        if (i >= 0) begin_ray(s, rays, hits, i, flags);
        while (__any(ref != kIdle)) {
            round(s, max_iter, st);
            walk_ends(s, rays, hits, flags);
        }
    }

    // The same, the lanes going from entity to entity together: an entity's record and root are read once for the wave, by
    // scalar loads, and lanes that pass it by wait.  At its own pace every lane fetches its own entities, and neighbours
    // that met the same nodes no longer do: 1920 x 1080 primary rays over 64 instances of 20,480 triangles take 916 us so,
    // 443 together (the array walk 676), 5,000 rays 135 and 106.  But a wave then waits for the longest walk of each entity,
    // not of all together: 400,000 bounce rays over 8 overlapping instances of 640,000 triangles take 770 us at their own
    // pace, 981 together (the array walk 1,697).
    __device__ __forceinline__ void run_together(const PairScene& s, const crt_ray* rays, crt_hit* __restrict__ hits,
                                                 int64_t i, uint32_t flags, int32_t max_iter, PairStack<D> st) {
        bool todo = i >= 0;
        exact = redo = false;
        slot = int32_t(i);
        ray_tmax = todo ? rays[i].tmax : 0.0f;
        do {
            reset();
            ref = kIdle;
            for (int32_t e = 0; e < s.entity_count; ++e) {
                const UniformEntity en(s.entities, e);
                if ((flags & CRT_FLAG_IGNORE_TRANSPARENT) && en.alpha() < 0.99f) continue;
                const bool take = todo && !redo && !(ANY && tri >= 0);
                if (!__any(take)) break;
                ent = e;
                if (take) {
                    const float4* rp = reinterpret_cast<const float4*>(rays + slot);
                    const float4 a = rp[0], b = rp[1];
                    ro = en.to_local(mk(a.x, a.y, a.z), 1.0f);
                    rd = en.to_local(mk(b.x, b.y, b.z), 0.0f);
                    inv = mk(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
                    if (ANY) tmax = ray_tmax;
                    const int32_t start = en.start();
                    const UniformFloat4 n(s.nodes + 2 * int64_t(start));
                    const float4 rmin = n[0], rmax = n[1];
                    const int32_t packed = __float_as_int(rmin.w);
                    it = 1;
                    sp = 0;
                    if (entry(rmin, rmax, ro, inv) < tmax)
                        ref = packed == -1 ? ~pair_base(start) : packed;
                    else
                        visits++;
                }
                while (__any(ref != kIdle)) {
                    round(s, max_iter, st);
                    if (ref == kDone) {
                        visits += uint32_t(it);
                        ref = kIdle;
                    }
                }
            }
            if (todo && !redo) finish(s, rays, hits, flags);
            todo = todo && redo;
            exact = todo;
            redo = false;
        } while (__any(todo));
    }
};

}  // namespace pair
}  // namespace crt
