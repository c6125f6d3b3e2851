// batch_plan_test.cpp -- the batch's groups and fuse limits on the host alone:
// every graph in one group, in order; groups end at the budget; the automatic
// limit follows the graphs of the group, not of the batch.
#include "hgp_batchplan.hpp"

#include <cstdio>

#define CHECK(x)                                               \
    do {                                                       \
        if (!(x)) {                                            \
            std::fprintf(stderr, "%d: %s\n", __LINE__, #x);    \
            return 1;                                          \
        }                                                      \
    } while (0)

using hgp::plan_batch;

int main()
{
    const size_t mb = 1 << 20, budget = (size_t)8 << 30;
    CHECK(plan_batch({}, budget, -1).empty());
    for (int limit : {-1, 0, 8192})
        for (int count : {1, 95, 96, 511, 512, 3000}) {
            auto g = plan_batch(std::vector<size_t>((size_t)count, mb), budget, limit);
            CHECK(g.size() == 1 && g[0].g0 == 0 && g[0].g1 == count);
            CHECK(g[0].fuse == (limit >= 0 ? limit : count < 96 ? 1024 : count < 512 ? 4096 : 8192));
        }
    // 600 graphs of 100 MB: seven groups of 82 and the rest, none of which fills the chip
    auto g = plan_batch(std::vector<size_t>(600, 100 * mb), budget, -1);
    CHECK(g.size() == 8);
    int32_t at = 0;
    for (auto &x : g) {
        CHECK(x.g0 == at && x.g1 > x.g0 && x.g1 - x.g0 <= 82 && x.fuse == 1024);
        at = x.g1;
    }
    CHECK(at == 600);
    // two graphs beyond the budget, then 700 small ones
    std::vector<size_t> b(702, mb);
    b[0] = b[1] = 2 * budget;
    g = plan_batch(b, budget, -1);
    CHECK(g.size() == 3 && g[0].g1 == 1 && g[1].g1 == 2 && g[0].fuse == 1024 && g[2].g1 == 702 && g[2].fuse == 8192);
    std::puts("ok");
    return 0;
}
