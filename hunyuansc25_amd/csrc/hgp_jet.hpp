// hgp_jet.hpp -- what the kernels of one Jet iteration share: the control
// block, the modes, the packed (where, dest) words, and the rebalancers'
// entry point.
#pragma once

#include "hgp_common.hpp"

namespace hgp {

enum JetMode : int32_t { kModeLP = 0, kModeRW = 1, kModeRS = 2 };

struct JetCtl {
    int64_t cut, best_cut, best_max, maxwgt, opt, maxdest;
    unsigned long long delta2;      // 2 x cut change (two's complement) of the one-block loop
    int32_t count, balance_counter, mode, done, iters, patience;
    int32_t ncand, nunder, copy_best, filt_num;   // ncand: 1 if an LP candidate exists
};

// Where the move accounting's blocks add their part-weight and cut changes:
// `count` copies (a power of two, at most 8) of k part deltas and twice the cut
// change, `stride` words apart; k_jet_next adds them up and clears them.
// Atomics on one cache line complete one after another (measured: 12 ns each,
// 22 ns for a wave's), so 2048 blocks that flush 256 parts into one copy take
// 45 us however little they computed; spread over copies they overlap (rows of
// <= 8 entries of R-MAT 2^22, k = 256: 26.0 -> 15.5 us a launch).
struct MoveSums {
    int64_t *rep = nullptr;
    int32_t count = 0, stride = 0;
    __device__ unsigned long long *mine() const
    {
        return (unsigned long long *)rep + (size_t)(blockIdx.x & (unsigned)(count - 1)) * stride;
    }
};

// Writes the (where, dest) word of v.
__device__ inline void store_pair(uint16_t *p16, uint32_t *p32, int32_t v, int32_t w, int32_t d)
{
    if (p16) p16[v] = (uint16_t)((uint32_t)w | ((uint32_t)d << 8));
    else p32[v] = (uint32_t)w | ((uint32_t)d << 16);
}

// A level's state as the rebalancers see it: the selection has left a key
// (part * kMaxBuckets + gain bucket, or k * kMaxBuckets: no candidate) and a
// destination per vertex.
struct RbView {
    int32_t n, k;
    const uint32_t *key;
    const wgt_t *vwgt;
    const int32_t *where;
    int32_t *dest;
    uint16_t *pd16;
    uint32_t *pd32;
    const int64_t *pwgts;
    const JetCtl *ctl;
};

// Scratch of a level's rebalancing iterations (right end of the arena).
struct RbScratch {
    uint32_t *key[2], *id[2];   // sorted candidates, two buffers
    uint32_t *hist;             // digit counts per tile
    int32_t *ptile;             // tile of each part's first candidate
    int64_t *phead;             // weight in that tile before it
    int32_t *w;                 // weights in sorted order
    int64_t *tsum, *tevw;       // per tile: candidate weight, evicted weight
    int32_t *tevn;              // per tile: evicted vertices
    int64_t *bs;                // prefix weights of the evicted list
    int32_t *elist;             // evicted vertices in order
    int32_t *es, *ee;           // the parts' slices of the evicted list
    int64_t *cnt;               // [0] candidates, [1] evicted
};
RbScratch rebalance_scratch(Ctx &c, int32_t n, int32_t k);

// One RW or RS step (mode, which the control block holds too): evicts from
// each overweight part its candidates in (bucket, id) order until it is within
// the bound; RW leaves the others where they are, RS deals the evicted ones to
// the parts with room.  Reads key; writes dest and the packed words.
void rebalance(Ctx &c, const RbView &v, const RbScratch &s, int32_t mode);

}  // namespace hgp
