// Host build of the device BVH4 / BVH8 collapse (candela_amd/csrc/wide_gpu.hip).
//
// Runs the per-node functions of wide_collapse.h level by level on one thread,
// with the numbering, the two-ended child lists and the rotating sums of the
// device's level passes (the same index functions; every index checked against
// its array), so the layout equals the device's.  tests/test_wide_collapse_host.py builds it with
// clang++ three ways -- under -fsanitize=undefined with every local set to a
// pattern (-ftrivial-auto-var-init=pattern), with every local zeroed, and
// plainly optimized -- and compares the layouts with crt_wide_build's: a value
// read before it is written, on some path only, would make them differ.
//
// stdin:  int64 node_count, int64 ntris, int32 width, then node_count
//         crt_stack_node entries (64 B each)
// stdout: int64 wide_nodes, uint32 status, then wide_nodes * width / 4
//         crt_wide_group (128 B each)
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

// What the HIP headers provide to the device build, for one host thread.
#define __device__
#define __host__
#define __forceinline__ inline
static inline unsigned atomicOr(unsigned* p, unsigned v) {
    const unsigned old = *p;
    *p = old | v;
    return old;
}
static inline int32_t __float_as_int(float f) {
    int32_t i;
    std::memcpy(&i, &f, sizeof(i));
    return i;
}
using std::max;
using std::min;

#include "wide_collapse.h"

using namespace crt::wg;

// Exits when an index leaves its array.
template <typename T>
struct Checked : std::vector<T> {
    using std::vector<T>::vector;
    T& operator[](int64_t i) {
        if (i < 0 || i >= int64_t(this->size())) {
            std::fprintf(stderr, "index %lld of %zu\n", static_cast<long long>(i), this->size());
            std::exit(3);
        }
        return std::vector<T>::operator[](size_t(i));
    }
};

template <int W>
static int run(const std::vector<crt_stack_node>& nodes, int64_t ntris) {
    const int64_t node_count = int64_t(nodes.size());
    const int64_t cap = ntris;   // the device's output capacity: one wide node per triangle
    Checked<crt_wide_group> groups(size_t(cap) * (W / 4));
    unsigned err = 0;
    int64_t total = 1;
    Kid k;
    if (root_one_slot(nodes[0], k)) {
        const bool ok = leaf_ok(k.start, k.count, ntris);
        if (!ok) err = kErrLeaf;
        write_one_slot_root<W>(groups.data(), k, ok);
    } else {
        // the workspace holds anything
        const int64_t stride = sums_for<W>(cap) + 1;
        Checked<int32_t> kids(size_t(cap) * W, 0x5A5A5A5A);
        Checked<uint32_t> sums(size_t(stride) * 3, 0xEEEEEEEEu);
        const auto kid = [&](int32_t level, int64_t item) { return &kids[kids_item(level, item, cap) * W]; };
        const auto sum = [&](int32_t level, int64_t at) -> uint32_t& {
            if (at >= stride) std::exit(4);
            return sums[sums_array(level) * stride + at];
        };
        sum(0, 0) = expand_one<W>(nodes.data(), node_count, ntris, 0, 0, groups.data(), kid(0, 0), &err);
        sum(1, 0) = 0u;
        int64_t np = 1;   // nodes of level p, the last numbered total - 1
        for (int32_t p = 0; np > 0; ++p) {
            const bool alone = np <= kParents<W>;
            int64_t all = 0;
            for (int64_t c = 0; c < sums_for<W>(np); ++c) all += sum(p, c);
            if (total + all > cap) {   // the pass's cap check
                err |= kErrCap;
                break;
            }
            for (int64_t at = 0; at < sums_for<W>(all * W) && at < stride; ++at) sum(p + 2, at) = 0u;
            int64_t before = 0;
            for (int64_t chunk = 0; chunk < sums_for<W>(np) && all > 0; ++chunk) {   // expand_chunk
                int32_t list[kBlock];
                uint32_t children[W + 1] = {};
                int64_t count = 0;
                for (int tid = 0; tid < kBlock; ++tid) {
                    const int64_t parent = chunk * kParents<W> + tid / W;
                    const int32_t entry = parent < np ? kid(p, parent)[tid % W] : -1;
                    if (entry < 0) continue;
                    (void)groups[(total - np + parent) * (W / 4)];
                    assign_slot<W>(total - np + parent, tid % W, total + before + count, groups.data());
                    list[count++] = entry;
                }
                const int64_t first = sum_of<W>(before);
                for (int64_t i = 0; i < count; ++i) {
                    const int64_t item = before + i;
                    (void)groups[(total + item + 1) * (W / 4) - 1];
                    const uint32_t m = expand_one<W>(nodes.data(), node_count, ntris, list[i], total + item,
                                                     groups.data(), kid(p + 1, item), &err);
                    if (sum_of<W>(item) - first > W) std::exit(5);
                    children[sum_of<W>(item) - first] += m;
                }
                for (int64_t at = 0; at <= W && count > 0 && first + at <= sum_of<W>(before + count - 1); ++at) {
                    if (alone)
                        sum(p + 1, first + at) = children[at];
                    else
                        sum(p + 1, first + at) += children[at];
                }
                before += count;
            }
            if (before != all) std::exit(6);   // the sums count the children
            total += all;
            np = all;
        }
    }
    if (err) {   // finish_async: any status bit leaves the root empty
        for (int q = 0; q < W / 4; ++q) {
            int32_t* g = reinterpret_cast<int32_t*>(&groups[size_t(q)]);
            for (int word = 0; word < 32; ++word) g[word] = word >= 28 ? -1 : 0;
        }
    }
    const uint32_t status = err;
    std::fwrite(&total, sizeof(total), 1, stdout);
    std::fwrite(&status, sizeof(status), 1, stdout);
    std::fwrite(groups.data(), sizeof(crt_wide_group), size_t(total) * (W / 4), stdout);
    return 0;
}

int main() {
    int64_t node_count = 0, ntris = 0;
    int32_t width = 0;
    if (std::fread(&node_count, 8, 1, stdin) != 1 || std::fread(&ntris, 8, 1, stdin) != 1 ||
        std::fread(&width, 4, 1, stdin) != 1 || node_count < 1 || ntris < 2 || (width != 4 && width != 8))
        return 2;
    std::vector<crt_stack_node> nodes(static_cast<size_t>(node_count));
    if (std::fread(nodes.data(), sizeof(crt_stack_node), nodes.size(), stdin) != nodes.size()) return 2;
    return width == 4 ? run<4>(nodes, ntris) : run<8>(nodes, ntris);
}
