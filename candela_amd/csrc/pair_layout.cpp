// Child pairs of a stackless BVH (pair_walk.h), derived on the host when a
// context buffers its data.
#include <cstring>
#include <vector>

#include "candela_rt.h"
#include "trace_launch.h"

namespace crt {

static int32_t bits(float f) {
    int32_t i;
    std::memcpy(&i, &f, 4);
    return i;
}

bool build_pairs(const crt_stackless_node* nodes, int64_t start, int64_t count, int64_t ntris, crt_stack_node* pairs) {
    if (count <= 0 || start < 0 || start + count > INT32_MAX) return false;
    const crt_stackless_node* n = nodes + start;
    // The walk of a valid tree is the pre-order itself: an inner node i has the
    // children i + 1 and link(i + 1), the right one inherits its link, and a
    // leaf's link is the node behind it.  These conditions nest, so together
    // they make every node's subtree [i, link(i)).
    auto link = [n](int64_t i) { return bits(n[i].max[3]); };
    auto end = [&](int64_t i) { return link(i) < 0 ? count : int64_t(link(i)); };
    if (link(0) != -1) return false;
    std::vector<int32_t> ref(static_cast<size_t>(count));
    std::vector<uint8_t> depth(static_cast<size_t>(count));
    int32_t next = pair_base(int32_t(start));
    for (int64_t i = 0; i < count; ++i) {
        const int32_t packed = bits(n[i].min[3]);
        if (link(i) < -1 || link(i) >= count) return false;
        if (packed == -1) {
            if (i + 1 >= count) return false;
            const int64_t r = link(i + 1);
            if (r <= i + 1 || r >= end(i) || link(r) != link(i)) return false;
            const int d = depth[size_t(i)] + 1;
            if (d > kPairStack) return false;
            depth[size_t(i) + 1] = depth[size_t(r)] = uint8_t(d);
            ref[size_t(i)] = ~next++;
        } else {
            if (packed < 0 || end(i) != i + 1 || int64_t(packed >> 4) + (packed & 0xF) > ntris) return false;
            ref[size_t(i)] = packed;
        }
    }
    auto child = [&](crt_bounds& dst, int64_t i) {
        std::memcpy(dst.min, n[i].min, 12);
        std::memcpy(dst.max, n[i].max, 12);
        std::memcpy(&dst.min[3], &ref[size_t(i)], 4);
        dst.max[3] = 0.0f;
    };
    for (int64_t i = 0; i < count; ++i) {
        if (ref[size_t(i)] >= 0) continue;
        crt_stack_node& p = pairs[~ref[size_t(i)]];
        child(p.left, i + 1);
        child(p.right, link(i + 1));
    }
    return true;
}

}  // namespace crt
