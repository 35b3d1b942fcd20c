// One entity's walk of either BVH2 layout as a step function, for kernels that
// trace rays inline (shade.hip).  Visits, tests and results are those of
// thread_walk.h's walk_stackless / walk_stack (same order, iteration cap and
// index guards), the guards of a stackless node as one comparison.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "candela_rt.h"
#include "device_math.h"
#include "stack_walk.h"
#include "trace_launch.h"

namespace crt {
namespace walker {

using namespace ::crt::dm;

// leaves() goes on until leaves are to be tested (leaf, then leaf2 unless it
// is -1) and returns true, or returns false at the end of the walk.  Lanes that
// have leaves wait in it for the others, so that the wave tests them together.
template <int FORMAT, int D>
struct Walker;

template <int D>
struct Walker<CRT_FORMAT_STACKLESS, D> {
    f3 ro, rd, inv;
    float tmax;
    int32_t start, ptr, it, leaf;
    uint32_t span;   // nodes start .. start + span pass the index guard
    static constexpr int32_t leaf2 = -1;

    __device__ __forceinline__ void init(int32_t*, int32_t, int32_t*) {}
    __device__ __forceinline__ void begin(int32_t first, int32_t count, int64_t total) {
        const int64_t end = int64_t(first) + count;
        const int64_t last = end < total ? end : total - 1;
        const bool any = first >= 0 && last >= first;
        start = first;
        span = any ? uint32_t(last - first) : 0u;
        ptr = any ? first : first - 1;
        it = 0;
    }
    // The loop-top checks of the walk; start - 1 stands for its end.
    __device__ __forceinline__ bool goes_on() const {
        return it < kMaxIterations && uint32_t(ptr) - uint32_t(start) <= span;
    }
    __device__ __forceinline__ bool leaves(const SceneArgs& s) {
        bool found = false, more = goes_on();
        while (more) {
            it++;
            const float4* p = reinterpret_cast<const float4*>(s.nodes) + 2 * int64_t(ptr);
            const float4 nmin = p[0], nmax = p[1];
            const float tb = bounds_stackless(nmin, nmax, ro, inv, tmax);
            const bool hit = tb > 0.0f && tb < tmax;
            leaf = __float_as_int(nmin.w);
            const bool inner = leaf == -1;
            const int32_t link = __float_as_int(nmax.w);
            ptr = hit && inner ? ptr + 1 : (link < 0 ? -1 : link) + start;
            found = hit && !inner;
            more = goes_on() && !found;
        }
        return found;
    }
};

template <int D>
struct Walker<CRT_FORMAT_STACK, D> : sdev::StackWave<false, D, 1, 1> {
    using Base = sdev::StackWave<false, D, 1, 1>;
    sdev::NodeStack<D> st;
    int32_t leaf2;

    __device__ __forceinline__ void init(int32_t* lds, int32_t stride, int32_t* spill) {
        st = sdev::NodeStack<D>{lds, stride, spill};
        Base::status = 0;
    }
    __device__ __forceinline__ void begin(int32_t first, int32_t count, int64_t) {
        Base::start = Base::cur = first;
        Base::count = count;
        Base::sp = Base::it = 0;
        Base::end_bits = 0;
    }
    __device__ __forceinline__ bool leaves(const SceneArgs& s) {
        if (Base::end_bits) return false;
        int32_t r;
        do r = Base::step(s, kMaxIterations, st);
        while (r == sdev::kNext);
        const bool l0 = sdev::leaf_nonempty(Base::leaf0);
        Base::leaf = l0 ? Base::leaf0 : Base::leaf1;
        leaf2 = l0 && sdev::leaf_nonempty(Base::leaf1) ? Base::leaf1 : -1;
        return r == sdev::kLeaves;
    }
};

}  // namespace walker
}  // namespace crt
