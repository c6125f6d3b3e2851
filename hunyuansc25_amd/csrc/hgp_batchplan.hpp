// hgp_batchplan.hpp -- how hgp_partition_batch cuts its graphs into groups and
// up to which size it refines the levels of a group in one launch (host only).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace hgp {

struct BatchGroup {
    int32_t g0, g1;   // graphs [g0, g1) of the batch's order
    int32_t fuse;     // levels of at most this many vertices go into the fused launch
};

// The automatic limit.  The fused launch lasts as long as its slowest graph,
// which one CU refines alone: worth it for the larger levels once the group
// keeps the other CUs busy meanwhile.  Graphs/s of the batched workload (1k-64k
// vertices) without fusing and fusing levels of up to 1024 / 4096 / 8192
// vertices: 16 graphs 444, 399 / 352 / 284; 48 graphs 501, 519 / 432 / 379; 96
// graphs 523, 545 / 543 / 516; 128 graphs 527, 557 / 577 / 565; 256 graphs with
// fusing 567 / 610 / 603; 768 graphs 566 / 612 / 668.  Groups of fewer than
// about 40 graphs, which are faster without, are not told apart from those of
// up to 96.
inline int32_t group_fuse_limit(int32_t graphs) { return graphs < 96 ? 1024 : graphs < 512 ? 4096 : 8192; }

// Groups of graphs whose hierarchies (bytes, in the batch's order) take up to
// about `budget`, one graph at least; limit: the caller's, -1 by the group.
inline std::vector<BatchGroup> plan_batch(const std::vector<size_t> &bytes, size_t budget, int32_t limit)
{
    std::vector<BatchGroup> out;
    const int32_t count = (int32_t)bytes.size();
    for (int32_t g0 = 0; g0 < count;) {
        int32_t g1 = g0;
        size_t gb = 0;
        while (g1 < count && (g1 == g0 || gb < budget)) gb += bytes[(size_t)g1++];
        out.push_back({g0, g1, limit < 0 ? group_fuse_limit(g1 - g0) : limit});
        g0 = g1;
    }
    return out;
}

}  // namespace hgp
