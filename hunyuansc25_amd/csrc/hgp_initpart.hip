// hgp_initpart.hip -- recursive-bisection initial partition of the coarsest
// graph (hunyuangraph_gpu_initialpartition / _RecursiveBisection,
// hunyuangraph_GPU_initialpartition.h:3913-4496).
//
// The recursion is run depth by depth.  All bisection nodes of one depth live
// in one "forest": every vertex of the coarsest graph sits in the contiguous
// range of the tree node that owns it, rows hold forest positions, and edges
// never cross nodes.  One launch runs every trial of every node of the depth
// (a block per GGGP + FM trial; a wave for small node graphs and for the FM on
// queues), so k-1 bisections take ceil(log2 k) launches and no host round-trips.  Tree node ids are heap ids (root 1, children 2i
// and 2i+1), which also key the trial random streams.
#include "hgp_graph.hpp"
#include "hgp_prims.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace hgp {

namespace {

// Arrays of a trial.  Scan FM in LDS: (ed, wd) pairs, row offsets (i32), queue
// (u16) and a state byte, 15 bytes a vertex; node graphs of up to kScanLdsN
// vertices run there (two trials per CU at that size).  Larger ones run in
// global scratch with a 32-bit queue and the node's own row offsets, 13 a
// vertex, 14 apart: a thousand trials walk their arrays side by side, and 13
// apart they lose 3 % at 20000 vertices, 23 % at 30000 (1060 against 864 ms a
// call; 17, with row offsets of their own, 860, but 3 B more a vertex and trial
// is 92 MB more of the 440 such a call allocates).  Heap FM: where, moved (u8),
// ed, id, queue, position index (i32) and two heaps of (key, vertex), n + 1
// slots each.
constexpr int32_t kScanLdsN = 4864;
constexpr int kHeapBytesPerVertex = 34;
constexpr int kHeapLdsBudget = 60 * 1024;
// fm_kind -1 keeps the scan: on the dense coarsest graphs this pipeline
// produces (R-MAT 2^22: 995 vertices, average degree ~300) the queues took
// 187 ms against 2 ms, a move's row being ~300 serial queue updates
constexpr int32_t kAutoHeapMinVertices = INT32_MAX;

__host__ __device__ inline int64_t trial_bytes(int64_t n, bool heap, bool in_lds)
{
    if (heap) return ((2 * n + 3) & ~3ll) + 12 * n + 4 * n + 16 * (n + 1);
    const int64_t n4 = (n + 3) & ~3ll;   // the arg-max reads four vertices at a time
    return (in_lds ? 15 : 14) * n4 + 16;
}

struct Node {
    int32_t start, end, k, fpart;
    int64_t tv, onemin, onemax, ideal0;
    int32_t T, trial_off, best, cnt0;
    int64_t woff;       // offset of the node's trial-where block (bytes)
    int64_t soff;       // offset of the node's global scratch block (bytes)
    int64_t doff, boff; // offsets of the node's dense weight and bit matrices (words)
};

// The root node: a wave per vertex sums its row's weight.
__global__ void __launch_bounds__(kRowBS) k_ip_init(int32_t n, const wgt_t *__restrict__ vwgt,
                                                    const eid_t *__restrict__ xadj,
                                                    const wgt_t *__restrict__ adjwgt, int32_t *__restrict__ node_of,
                                                    int32_t *__restrict__ label, wgt_t *__restrict__ fvw,
                                                    int32_t *__restrict__ fwd, Node *nodes)
{
    const int32_t v = (int32_t)gindex<kWave>();
    if (v >= n) return;   // whole waves
    int32_t s = 0;
    const eid_t e = xadj[v + 1];
#pragma unroll 4
    for (eid_t j = xadj[v] + lane_id(); j < e; j += kWave) s += adjwgt[j];
    s = wave_sum(s);
    if (lane_id() != 0) return;
    node_of[v] = 1;
    label[v] = v;
    fvw[v] = vwgt[v];
    fwd[v] = s;
    if (v == 0) {
        nodes[1].start = 0;
        nodes[1].end = n;
    }
}

// Per active node: total weight and the bisection bounds
// (:3986-3987 with tp1 = kr/k, ub = 1.03^(1/ln k) computed on the host).
__global__ void __launch_bounds__(256) k_ip_setup(const int32_t *__restrict__ act, Node *nodes,
                                                  const wgt_t *__restrict__ fvw, double ub, int32_t trials)
{
    __shared__ int64_t sh[4];
    Node &nd = nodes[act[blockIdx.x]];
    int64_t s = 0;
    for (int32_t v = nd.start + threadIdx.x; v < nd.end; v += blockDim.x) s += fvw[v];
    s = wave_sum(s);
    if (lane_id() == 0) sh[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t tv = sh[0] + sh[1] + sh[2] + sh[3];
        int32_t k = nd.k, kl = k >> 1, kr = k - kl;
        double t1 = ((double)tv * (double)kr) / (double)k;
        nd.tv = tv;
        nd.onemax = (int64_t)floor(ub * t1);
        nd.onemin = (int64_t)floor(t1 / ub);
        nd.ideal0 = (tv * kl) / k;
        int32_t nn = nd.end - nd.start;
        nd.T = trials < nn ? trials : nn;
        nd.best = -1;
    }
}

// Exclusive offsets of trials, scratch and dense matrices over the active
// nodes: running sums in one block, 256 nodes a step (one thread walking the nodes
// took 145 us for 500 of them).
__global__ void __launch_bounds__(256) k_ip_offsets(const int32_t *__restrict__ act, int32_t nact, Node *nodes,
                                                    int32_t lds_cap, bool heap, int32_t *total)
{
    __shared__ int64_t sh[256 / kWave];
    int64_t t = 0, w = 0, s = 0, d = 0, b = 0;
    for (int32_t a0 = 0; a0 < nact; a0 += 256) {
        const int32_t a = a0 + threadIdx.x;
        Node *nd = a < nact ? &nodes[act[a]] : nullptr;
        const int64_t nn = nd ? nd->end - nd->start : 0, tr = nd ? nd->T : 0;
        const int64_t sc = nn > lds_cap ? tr * ((trial_bytes(nn, heap, false) + 255) & ~255ll) : 0;
        int64_t at, tot;
        at = block_exclusive_scan<int64_t>(tr, sh, &tot) + t;
        t += tot;
        if (nd) nd->trial_off = (int32_t)at;
        at = block_exclusive_scan<int64_t>(tr * nn, sh, &tot) + w;
        w += tot;
        if (nd) nd->woff = at;
        at = block_exclusive_scan<int64_t>(sc, sh, &tot) + s;
        s += tot;
        if (nd) nd->soff = at;
        at = block_exclusive_scan<int64_t>(nn * ((nn + 3) & ~3ll), sh, &tot) + d;
        d += tot;
        if (nd) nd->doff = at;
        at = block_exclusive_scan<int64_t>(nn * ((nn + 31) / 32), sh, &tot) + b;
        b += tot;
        if (nd) nd->boff = at;
    }
    if (threadIdx.x == 0) *total = (int32_t)t;
}

struct TrialMem {
    uint8_t *where, *moved;
    int32_t *ed, *id, *queue;
    int32_t *loc, *hkey[2], *hval[2];
};

// ---- device priority queue (hunyuangraph_GPU_priorityqueue.h:27-225), run by
// one lane: a max-heap of vertices with a position index.  An element moves
// above another when its key is strictly greater, or, with `ties`, equal with
// a smaller vertex id (the top is then the unique (gain desc, id asc)
// maximum); a removal refills the hole from the last slot.
struct Heap {
    int32_t *key, *val, *loc;
    int32_t cnt;
    bool ties;
    __device__ bool above(int32_t ka, int32_t va, int32_t kb, int32_t vb) const
    {
        return ka > kb || (ties && ka == kb && va < vb);
    }
    __device__ void place(int32_t i, int32_t k, int32_t v)
    {
        key[i] = k;
        val[i] = v;
        loc[v] = i;
    }
    __device__ void up(int32_t i, int32_t k, int32_t v)
    {
        while (i > 0) {
            int32_t j = (i - 1) >> 1;
            int32_t kj = key[j], vj = val[j];
            if (!above(k, v, kj, vj)) break;
            place(i, kj, vj);
            i = j;
        }
        place(i, k, v);
    }
    __device__ void down(int32_t i, int32_t k, int32_t v)
    {
        int32_t j;
        while ((j = 2 * i + 1) < cnt) {
            int32_t kj = key[j], vj = val[j];
            if (j + 1 < cnt) {
                int32_t k1 = key[j + 1], v1 = val[j + 1];
                if (above(kj, vj, k, v)) {
                    if (above(k1, v1, kj, vj)) { j++; kj = k1; vj = v1; }
                } else if (above(k1, v1, k, v)) {
                    j++; kj = k1; vj = v1;
                } else {
                    break;
                }
            } else if (!above(kj, vj, k, v)) {
                break;
            }
            place(i, kj, vj);
            i = j;
        }
        place(i, k, v);
    }
    __device__ void insert(int32_t v, int32_t k) { up(cnt++, k, v); }
    __device__ int32_t top()
    {
        if (cnt == 0) return -1;
        int32_t t = val[0];
        loc[t] = -1;
        if (--cnt > 0) down(0, key[cnt], val[cnt]);
        return t;
    }
    __device__ void remove(int32_t v)
    {
        int32_t i = loc[v];
        loc[v] = -1;
        if (--cnt > 0 && val[cnt] != v) {
            int32_t nk = key[cnt], nv = val[cnt];
            if (above(nk, nv, key[i], v)) up(i, nk, nv);
            else down(i, nk, nv);
        }
    }
    __device__ void update(int32_t v, int32_t k)
    {
        int32_t i = loc[v];
        if (k > key[i]) up(i, k, v);
        else down(i, k, v);
    }
};

__device__ inline void fence_wave()
{
    __threadfence_block();
    __syncthreads();
}

// Trial gw of the depth: its node (the last active node whose trials start at
// or before gw).
__device__ inline int32_t trial_node(const int32_t *__restrict__ act, int32_t nact, const Node *__restrict__ nodes,
                                     int32_t gw)
{
    int32_t lo = 0, hi = nact - 1;
    while (lo < hi) {
        int32_t mid = (lo + hi + 1) >> 1;
        if (nodes[act[mid]].trial_off <= gw) lo = mid; else hi = mid - 1;
    }
    return act[lo];
}

// Start vertex of trial t (sampled when the node has more vertices than trials).
__device__ inline int32_t trial_start(const Node &nd, int32_t nid, int32_t n, int32_t t, uint64_t seed, int32_t &draw)
{
    if (nd.T >= n) return t;
    int32_t len = n / nd.T, rem = n % nd.T, left;
    if (t < rem) { len++; left = t * len; }
    else left = rem * (len + 1) + (t - rem) * len;
    return left + (int32_t)(trial_rng(seed, (uint32_t)nid, t, draw++) % (uint64_t)len);
}

// One GGGP + FM trial per wave (hunyuangraph_gpu_BFS_warp_2wayrefine_noedit[_sampling],
// :2426-3659) with the queue-driven FM.  Every lane runs the serial BFS;
// vertex scans and neighbour updates are spread over the 64 lanes.
// The boundary flag is derived: bnd(v) = deg(v) == 0 || ed[v] > 0, which is
// the invariant the reference's incremental updates maintain.
__global__ void __launch_bounds__(kWave) k_ip_trials_heap(const int32_t *__restrict__ act, int32_t nact,
                                                          const Node *__restrict__ nodes, const int32_t *total,
                                                          const eid_t *__restrict__ fx,
                                                          const vid_t *__restrict__ fadj,
                                                          const wgt_t *__restrict__ fw, const wgt_t *__restrict__ fvw,
                                                          uint64_t seed, int32_t fm_passes, int32_t fm_kind,
                                                          int32_t lds_cap, uint8_t *__restrict__ trial_where,
                                                          char *__restrict__ gscratch, int64_t *__restrict__ tcut)
{
    extern __shared__ char lds[];
    int32_t gw = blockIdx.x;
    if (gw >= *total) return;
    int lane = threadIdx.x;
    const int32_t nid = trial_node(act, nact, nodes, gw);
    const Node nd = nodes[nid];
    const int32_t t = gw - nd.trial_off;
    const int32_t n = nd.end - nd.start, s0 = nd.start;
    char *base;
    if (n <= lds_cap) base = lds;
    else base = gscratch + nd.soff + (int64_t)t * ((trial_bytes(n, true, false) + 255) & ~255ll);
    TrialMem M;
    M.where = (uint8_t *)base;
    M.moved = M.where + n;
    M.ed = (int32_t *)(base + (((int64_t)2 * n + 3) & ~3ll));
    M.id = M.ed + n;
    M.queue = M.id + n;
    M.loc = M.queue + n;
    M.hkey[0] = M.loc + n;
    M.hval[0] = M.hkey[0] + (n + 1);
    M.hkey[1] = M.hval[0] + (n + 1);
    M.hval[1] = M.hkey[1] + (n + 1);
    const int64_t tv = nd.tv, onemin = nd.onemin, onemax = nd.onemax, ideal0 = nd.ideal0;

    for (int32_t i = lane; i < n; i += kWave) { M.where[i] = 1; M.moved[i] = 0; }
    fence_wave();

    // GGGP: BFS from the start vertex, moving vertices to side 0 in BFS order.
    // Every lane runs the same control flow on the same values; the rows of
    // dequeued vertices are scanned 64 entries at a time and the unvisited
    // neighbours appended in row order (ballot ranks), as a serial scan would.
    int64_t pw0 = 0, pw1 = tv;
    {
        int32_t draw = 0;
        const int32_t start = trial_start(nd, nid, n, t, seed, draw);
        int32_t first = 0, last = 1, nleft = n - 1, drain = 0;
        if (lane == 0) {
            M.queue[0] = start;
            M.moved[start] = 1;
        }
        fence_wave();
        for (;;) {
            if (first == last) {
                if (nleft == 0 || drain) break;
                // restart from the r-th unvisited vertex in id order
                int32_t r = (int32_t)(trial_rng(seed, (uint32_t)nid, t, draw++) % (uint64_t)nleft);
                int32_t v = -1;
                for (int32_t b0 = 0; b0 < n; b0 += kWave) {
                    int32_t u = b0 + lane;
                    bool un = u < n && M.moved[u] == 0;
                    uint64_t bal = __ballot(un);
                    int32_t cnt = __popcll(bal);
                    if (r < cnt) {
                        uint64_t pick = __ballot(un && __popcll(bal & lanemask_lt()) == r);
                        v = b0 + (__ffsll((long long)pick) - 1);
                        break;
                    }
                    r -= cnt;
                }
                if (lane == 0) {
                    M.queue[0] = v;
                    M.moved[v] = 1;
                }
                fence_wave();
                first = 0;
                last = 1;
                nleft--;
            }
            int32_t v = M.queue[first++];
            int32_t wv = fvw[s0 + v];
            if (pw0 > 0 && pw1 - wv < onemin) { drain = 1; continue; }
            if (lane == 0) M.where[v] = 0;
            pw0 += wv;
            pw1 -= wv;
            if (pw1 <= onemax) break;
            drain = 0;
            // once every vertex is queued a row has nothing fresh to append
            eid_t rb = fx[s0 + v], re = nleft > 0 ? fx[s0 + v + 1] : rb;
            for (eid_t j0 = rb; j0 < re; j0 += kWave) {
                eid_t j = j0 + lane;
                int32_t x = j < re ? fadj[j] - s0 : -1;
                bool fresh = x >= 0 && M.moved[x] == 0;
                uint64_t bal = __ballot(fresh);
                if (fresh) {
                    M.queue[last + __popcll(bal & lanemask_lt())] = x;
                    M.moved[x] = 1;
                }
                last += __popcll(bal);
                nleft -= __popcll(bal);
            }
            fence_wave();
        }
    }
    fence_wave();

    // ed / id and the cut (compute_v_ed_id_bnd, :23-62).  From here on
    // moved[v] holds bit 0 = moved in this pass, bit 1 = v has no edges.
    int64_t cutacc = 0;
    for (int32_t v = lane; v < n; v += kWave) {
        int32_t e = 0, in = 0;
        uint8_t me = M.where[v];
        eid_t rb = fx[s0 + v], re = fx[s0 + v + 1];
        eid_t j = rb;
        for (; j + 8 <= re; j += 8) {   // eight entries' loads in flight
            int32_t x[8], w[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                x[t] = fadj[j + t];
                w[t] = fw[j + t];
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                if (M.where[x[t] - s0] != me) e += w[t]; else in += w[t];
            }
        }
        for (; j < re; j++) {
            if (M.where[fadj[j] - s0] != me) e += fw[j]; else in += fw[j];
        }
        M.ed[v] = e;
        M.id[v] = in;
        M.moved[v] = rb == re ? 2 : 0;
        cutacc += e;
    }
    int64_t cut = wave_sum(cutacc) / 2;
    fence_wave();

    int64_t pw[2] = {pw0, pw1};
    const int64_t ideal[2] = {ideal0, tv - ideal0};
    int64_t limit = n / 100;
    if (limit < 15) limit = 15;
    if (limit > 100) limit = 100;
    int32_t *swaps = M.queue;

    // FM driven by two priority queues (FM_2way_cut_refinement,
    // hunyuangraph_GPU_initialpartition.h:160-300).  Lane 0 runs every
    // queue operation in the serial order; the lanes share the gain
    // updates of a move's row.  fm_kind 1: (gain desc, id asc) keys and
    // the part bounds of the scan FM, so the moves are the same;
    // fm_kind 2: the reference's queue order and balance rule
    // (|ideal0 - pw0| <= origdiff + avgvwgt, weights applied before the
    // test as hunyuangraph_CPU_2wayrefine.h:133-145 does).
    Heap q[2];
    for (int s = 0; s < 2; s++) {
        q[s].key = M.hkey[s];
        q[s].val = M.hval[s];
        q[s].loc = M.loc;
        q[s].cnt = 0;
        q[s].ties = fm_kind == 1;
    }
    const bool live_rule = fm_kind == 1;
    const int64_t a20 = (pw[0] + pw[1]) / 20, a2n = 2 * (pw[0] + pw[1]) / n;
    const int64_t avgvwgt = a20 < a2n ? a20 : a2n;
    const int64_t origdiff = ideal[0] - pw[0] < 0 ? pw[0] - ideal[0] : ideal[0] - pw[0];
    for (int32_t pass = 0; pass < fm_passes; pass++) {
        int64_t mincutorder = -1;
        int64_t newcut = cut, mincut = cut, initcut = cut;
        int64_t d0 = ideal[0] - pw[0];
        int64_t mindiff = d0 < 0 ? -d0 : d0;
        if (lane == 0) {
            q[0].cnt = q[1].cnt = 0;
            for (int32_t v = 0; v < n; v++) {
                int32_t e = M.ed[v];
                if (e > 0 || (M.moved[v] & 2)) q[M.where[v]].insert(v, e - M.id[v]);
            }
        }
        int32_t nswaps;
        for (nswaps = 0; nswaps < n; nswaps++) {
            int from = (ideal[0] - pw[0] < ideal[1] - pw[1]) ? 0 : 1;
            int to = from ^ 1;
            int32_t bv = -1, bg = 0;
            if (lane == 0) {
                bv = q[from].top();
                if (bv >= 0) bg = M.ed[bv] - M.id[bv];
            }
            bv = __shfl(bv, 0, kWave);
            bg = __shfl(bg, 0, kWave);
            if (bv == -1) break;
            int32_t wv = fvw[s0 + bv];
            newcut -= bg;
            bool accept;
            if (live_rule) {
                int64_t dd = ideal[0] - pw[0];
                dd = dd < 0 ? -dd : dd;
                accept = (newcut < mincut && pw[to] + wv <= onemax && pw[from] - wv <= onemax) ||
                         (newcut == mincut && dd < mindiff);
                if (accept) mindiff = dd;
                pw[to] += wv;
                pw[from] -= wv;
            } else {
                pw[to] += wv;
                pw[from] -= wv;
                int64_t dd = ideal[0] - pw[0];
                dd = dd < 0 ? -dd : dd;
                accept = (newcut < mincut && dd <= origdiff + avgvwgt) || (newcut == mincut && dd < mindiff);
                if (accept) mindiff = dd;
            }
            if (accept) {
                mincut = newcut;
                mincutorder = nswaps;
            } else if (nswaps - mincutorder > limit) {
                newcut += bg;
                pw[from] += wv;
                pw[to] -= wv;
                break;
            }
            if (lane == 0) {
                M.where[bv] = (uint8_t)to;
                M.moved[bv] |= 1;
                swaps[nswaps] = bv;
                int32_t tmp = M.ed[bv];
                M.ed[bv] = M.id[bv];
                M.id[bv] = tmp;
            }
            fence_wave();
            const eid_t rb = fx[s0 + bv], re = fx[s0 + bv + 1];
            for (eid_t j = rb + lane; j < re; j += kWave) {
                int32_t x = fadj[j] - s0;
                int32_t kw = (M.where[x] == from) ? -fw[j] : fw[j];
                M.id[x] += kw;     // rows hold no duplicates: one lane per neighbour
                M.ed[x] -= kw;
            }
            fence_wave();
            if (lane == 0) {
                // queue upkeep in row order: a neighbour that left the
                // boundary is deleted, one that stays is re-keyed, one
                // that joined is inserted (moved vertices stay out)
                for (eid_t j = rb; j < re; j++) {
                    int32_t x = fadj[j] - s0;
                    uint8_t st = M.moved[x];
                    if (st & 1) continue;
                    int32_t e = M.ed[x];
                    int32_t kw = (M.where[x] == from) ? -fw[j] : fw[j];
                    bool was = e + kw > 0;
                    int sx = M.where[x];
                    if (was) {
                        if (e == 0) q[sx].remove(x);
                        else q[sx].update(x, e - M.id[x]);
                    } else if (e > 0) {
                        q[sx].insert(x, e - M.id[x]);
                    }
                }
            }
            fence_wave();
        }
        for (int32_t i = lane; i < nswaps; i += kWave) M.moved[swaps[i]] &= 2;
        fence_wave();
        for (nswaps--; nswaps > mincutorder; nswaps--) {
            int32_t v = swaps[nswaps];
            int from = M.where[v];
            int to = from ^ 1;
            int32_t wv = fvw[s0 + v];
            fence_wave();
            if (lane == 0) {
                M.where[v] = (uint8_t)to;
                int32_t tmp = M.ed[v];
                M.ed[v] = M.id[v];
                M.id[v] = tmp;
            }
            pw[to] += wv;
            pw[from] -= wv;
            fence_wave();
            for (eid_t j = fx[s0 + v] + lane; j < fx[s0 + v + 1]; j += kWave) {
                int32_t x = fadj[j] - s0;
                int32_t kw = (M.where[x] == from) ? -fw[j] : fw[j];
                M.id[x] += kw;
                M.ed[x] -= kw;
            }
            fence_wave();
        }
        cut = mincut;
        if (mincutorder <= 0 || mincut == initcut) break;
    }

    uint8_t *out = trial_where + nd.woff + (int64_t)t * n;
    for (int32_t i = lane; i < n; i += kWave) out[i] = M.where[i];
    if (lane == 0) tcut[gw] = cut;
}

// ---------------------------------------------------------------- scan FM

// One GGGP + FM trial per block of NT threads, the FM choosing each move by
// an arg-max scan.  A trial is a serial chain (a BFS step, then an FM move at
// a time), so its time is the latency of one step times the steps, and each
// step is made of as few round trips as its data allow:
//  * the row offsets sit in LDS with the trial, so a row's entries are one
//    load away, several per lane at once, and the BFS loads the next row while
//    it works through this one;
//  * a vertex keeps its external weight ed and its row's weight wd (summed
//    once per node by k_ip_edges), so its gain is 2 ed - wd and a move changes
//    one word per neighbour; the BFS keeps ed as it goes, so no pass over all
//    rows follows it;
//  * the arg-max reads four vertices per thread and step and reduces on the
//    VALU;
//  * 256 threads for node graphs of kWideTrial vertices and more, one wave
//    below, where a step has no work for more.
// Used where the dense trials below are not: coarsest graphs of more than
// kDenseN vertices, rows that do not ascend, an arena without room for the
// matrices.
constexpr int32_t kWideTrial = 128;
constexpr uint8_t kStSide = 1, kStMoved = 2, kStAlone = 4;   // state byte: side, queued or moved, no edges

// The node's graph in the forest arrays.
struct TrialRows {
    const vid_t *adj;    // the node's entries (forest positions)
    const wgt_t *w, *vw;
    int32_t s0;
    // entries first, first + step, ... of [.., e): neighbour -1 past the end
    template <int P>
    __device__ void load(int32_t first, int32_t e, int step, int32_t (&x)[P], int32_t (&wt)[P]) const
    {
#pragma unroll
        for (int q = 0; q < P; q++) {
            const int32_t j = first + q * step;
            x[q] = j < e ? adj[j] - s0 : -1;
            wt[q] = j < e ? w[j] : 0;
        }
    }
};

// The trial's arrays: (ed, wd) per vertex, row offsets from the node's first
// entry (in LDS only), queue / swap list, state bytes.
template <class Q>
struct ScanMem {
    static constexpr bool kOffsets = sizeof(Q) == 2;   // (a 16-bit queue: in LDS)
    int2 *ew;
    int32_t *off;
    Q *queue;
    uint8_t *st;
    const eid_t *fx;   // the node's rows in the forest
    __device__ ScanMem(char *base, int32_t n, const eid_t *node_rows) : fx(node_rows)
    {
        const int64_t n4 = (n + 3) & ~3;
        ew = (int2 *)base;
        off = (int32_t *)(base + 8 * n4);
        queue = (Q *)(kOffsets ? off + n4 + 4 : off);
        st = (uint8_t *)(queue + n4);
    }
    // first entry of row v, from the node's first one
    __device__ int32_t row(int32_t v) const
    {
        if constexpr (kOffsets) return off[v];
        else return (int32_t)(fx[v] - fx[0]);
    }
    // marks v queued; whether it was not before (one of several lanes that
    // mark the same vertex sees it fresh); old: the state byte before
    __device__ bool mark(int32_t v, uint32_t &old) const
    {
        const int sh = 8 * (v & 3);
        old = (atomicOr((uint32_t *)st + (v >> 2), (uint32_t)kStMoved << sh) >> sh) & 255u;
        return !(old & kStMoved);
    }
};

// GGGP: BFS from a start vertex, moving vertices to side 0 in BFS order, run by
// one wave: every lane follows the same control flow on the same values; rows
// are taken 64 entries at a time and the unvisited neighbours appended in row
// order (ballot ranks), as a serial scan would.  ed is kept current.  Returns
// side 0's weight.
template <class Q>
__device__ inline int64_t trial_grow(const TrialRows &G, const ScanMem<Q> &M, int32_t n, const Node &nd,
                                     int32_t nid, int32_t t, uint64_t seed)
{
    constexpr int P = 4;   // 64-entry pieces of a row in flight
    const int lane = lane_id();
    const int64_t onemin = nd.onemin, onemax = nd.onemax;
    int64_t pw0 = 0, pw1 = nd.tv;
    int32_t draw = 0;
    const int32_t start = trial_start(nd, nid, n, t, seed, draw);
    int32_t first = 0, last = 1, nleft = n - 1, drain = 0;
    if (lane == 0) {
        M.queue[0] = (Q)start;
        M.st[start] |= kStMoved;
    }
    wave_lds_sync();
    // the next vertex in the queue: its position, row and weight, loaded ahead
    int32_t ahead = -1, av = 0, aw = 0, ab = 0, ae = 0, ax[P], at[P];
    for (;;) {
        if (first == last) {
            if (nleft == 0 || drain) break;
            // restart from the r-th unvisited vertex in id order
            int32_t r = (int32_t)(trial_rng(seed, (uint32_t)nid, t, draw++) % (uint64_t)nleft);
            int32_t v = -1;
            for (int32_t b0 = 0; b0 < n; b0 += kWave) {
                int32_t u = b0 + lane;
                bool un = u < n && !(M.st[u] & kStMoved);
                uint64_t bal = __ballot(un);
                int32_t cnt = __popcll(bal);
                if (r < cnt) {
                    uint64_t pick = __ballot(un && __popcll(bal & lanemask_lt()) == r);
                    v = b0 + (__ffsll((long long)pick) - 1);
                    break;
                }
                r -= cnt;
            }
            if (lane == 0) {
                M.queue[0] = (Q)v;
                M.st[v] |= kStMoved;
            }
            wave_lds_sync();
            first = 0;
            last = 1;
            nleft--;
            ahead = -1;
        }
        int32_t v, wv, rb, re, x[P], w[P];
        if (ahead == first) {
            v = av;
            wv = aw;
            rb = ab;
            re = ae;
#pragma unroll
            for (int q = 0; q < P; q++) {
                x[q] = ax[q];
                w[q] = at[q];
            }
        } else {
            v = wave_read((int32_t)M.queue[first], 0);
            rb = wave_read(M.row(v), 0);
            re = wave_read(M.row(v + 1), 0);
            wv = G.vw[v];
            G.load(rb + lane, re, kWave, x, w);
        }
        first++;
        if (first < last) {
            ahead = first;
            av = wave_read((int32_t)M.queue[first], 0);
            ab = wave_read(M.row(av), 0);
            ae = wave_read(M.row(av + 1), 0);
            aw = G.vw[av];
            G.load(ab + lane, ae, kWave, ax, at);
        }
        wv = wave_read(wv, 0);
        if (pw0 > 0 && pw1 - wv < onemin) { drain = 1; continue; }
        pw0 += wv;
        pw1 -= wv;
        const bool stop = pw1 <= onemax;
        if (lane == 0) {
            M.st[v] &= (uint8_t)~kStSide;
            const int2 e = M.ew[v];
            M.ew[v] = make_int2(e.y - e.x, e.y);
        }
        drain = 0;
        // the row: neighbours of side 1 gain an external edge, those of side 0
        // lose one; the unvisited ones join the queue (not after the last vertex)
        for (int32_t j0 = rb; j0 < re; j0 += P * kWave) {
            if (j0 > rb) G.load(j0 + lane, re, kWave, x, w);
            bool fresh[P];
#pragma unroll
            for (int q = 0; q < P; q++) {
                fresh[q] = false;
                if (x[q] < 0) continue;
                uint32_t old;
                fresh[q] = M.mark(x[q], old);
                atomicAdd(&M.ew[x[q]].x, (old & kStSide) ? w[q] : -w[q]);
            }
#pragma unroll
            for (int q = 0; q < P; q++) {
                const uint64_t bal = __ballot(fresh[q]);
                if (fresh[q]) M.queue[last + __popcll(bal & lanemask_lt())] = (Q)x[q];
                last += __popcll(bal);
                nleft -= __popcll(bal);
            }
        }
        wave_lds_sync();
        if (stop) break;
    }
    return pw0;
}

// Moves v (a vertex of side `from`) to the other side: its external and
// internal weight change places and its neighbours' external weight changes
// by each edge.  x, w hold the row's first P*NT entries (x = -1 past the end).
template <int NT, int P, class Q>
__device__ inline void trial_move(const TrialRows &G, const ScanMem<Q> &M, int32_t v, int from, int32_t rb,
                                  int32_t re, int32_t (&x)[P], int32_t (&w)[P])
{
    const int tid = threadIdx.x;
    if (tid == 0) {
        const int2 e = M.ew[v];
        M.ew[v] = make_int2(e.y - e.x, e.y);
    }
    for (int32_t j0 = rb; j0 < re; j0 += P * NT) {
        if (j0 > rb) G.load(j0 + tid, re, NT, x, w);
#pragma unroll
        for (int q = 0; q < P; q++) {
            if (x[q] < 0) continue;
            atomicAdd(&M.ew[x[q]].x, (M.st[x[q]] & kStSide) == from ? w[q] : -w[q]);
        }
    }
}

template <int NT>
struct TrialShared {
    int2 best[2][NT / kWave];   // each wave's (gain, vertex), by parity of the move
    int64_t sum[NT / kWave];
    int64_t pw0;
};

// The trial in arrays at `base`; returns its cut.  Every thread of the block
// calls it and follows the same control flow.
template <int NT, class Q>
__device__ inline int64_t scan_trial(const TrialRows &G, char *base, int32_t n, const Node &nd, int32_t nid, int32_t t,
                                     const eid_t *__restrict__ fx, const int32_t *__restrict__ fwd, uint64_t seed,
                                     int32_t fm_passes, TrialShared<NT> &S)
{
    constexpr int NW = NT / kWave;
    constexpr int P = NT == kWave ? 4 : 2;   // row entries per thread in flight
    const int tid = threadIdx.x, lane = lane_id();
    const ScanMem<Q> M(base, n, fx + G.s0);
    if constexpr (ScanMem<Q>::kOffsets)
        for (int32_t i = tid; i <= n; i += NT) M.off[i] = (int32_t)(M.fx[i] - M.fx[0]);
    for (int32_t i = tid; i < ((n + 3) & ~3); i += NT) {
        M.st[i] = kStSide;
        M.ew[i] = make_int2(0, i < n ? fwd[G.s0 + i] : 0);   // the padding stays out of the arg-max: ed 0, not alone
    }
    __syncthreads();
    if (tid < kWave) {
        const int64_t w0 = trial_grow<Q>(G, M, n, nd, nid, t, seed);
        if (tid == 0) S.pw0 = w0;
    }
    __syncthreads();
    // side weights (an array indexed by the side would go to scratch memory)
    int64_t pw0 = S.pw0, pw1 = nd.tv - S.pw0;
    const int64_t ideal0 = nd.ideal0, ideal1 = nd.tv - nd.ideal0;
    const int64_t onemax = nd.onemax;

    // the cut (compute_v_ed_id_bnd, :23-62); from here on kStMoved means
    // moved in this pass
    int64_t cutacc = 0;
    for (int32_t v = tid; v < n; v += NT) {
        const int2 e = M.ew[v];
        M.st[v] = (uint8_t)((M.st[v] & kStSide) | (M.row(v) == M.row(v + 1) ? kStAlone : 0));
        cutacc += e.x;
    }
    cutacc = wave_sum(cutacc);
    if (lane == 0) S.sum[tid / kWave] = cutacc;
    __syncthreads();
    int64_t cut = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) cut += S.sum[i];
    cut /= 2;

    int64_t limit = n / 100;
    if (limit < 15) limit = 15;
    if (limit > 100) limit = 100;
    Q *swaps = M.queue;
    for (int32_t pass = 0; pass < fm_passes; pass++) {
        int64_t mincutorder = -1;
        int64_t newcut = cut, mincut = cut, initcut = cut;
        int64_t d0 = ideal0 - pw0;
        int64_t mindiff = d0 < 0 ? -d0 : d0;
        int32_t nswaps;
        for (nswaps = 0; nswaps < n; nswaps++) {
            const int from = (ideal0 - pw0 < ideal1 - pw1) ? 0 : 1;
            // the boundary vertex of side `from`, not moved in this pass, of
            // largest gain (2 ed - wd; |gain| < 2^30), the smallest id among equals
            int32_t g = INT32_MIN, bv = INT32_MAX;
            for (int32_t u0 = tid * 4; u0 < n; u0 += NT * 4) {
                const int4 a = *(const int4 *)(M.ew + u0), b = *(const int4 *)(M.ew + u0 + 2);
                const uint32_t s4 = *(const uint32_t *)(M.st + u0);
                const int32_t ed[4] = {a.x, a.z, b.x, b.z}, wd[4] = {a.y, a.w, b.y, b.w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t st = (s4 >> (8 * q)) & 255u;
                    const bool can = ((st & (kStSide | kStMoved)) == (uint32_t)from) & ((ed[q] > 0) | ((st & kStAlone) != 0));
                    const int32_t gq = can ? 2 * ed[q] - wd[q] : INT32_MIN;
                    bv = gq > g ? u0 + q : bv;
                    g = gq > g ? gq : g;
                }
            }
            const int32_t gm = lanes_reduce<kWave>(g, [](int32_t a, int32_t b) { return a > b ? a : b; });
            bv = lanes_reduce<kWave>(g == gm ? bv : INT32_MAX, [](int32_t a, int32_t b) { return a < b ? a : b; });
            g = gm;
            if constexpr (NW > 1) {
                int2 *slot = S.best[nswaps & 1];
                if (lane == 0) slot[tid / kWave] = make_int2(g, bv);
                __syncthreads();
                g = INT32_MIN;
                bv = INT32_MAX;
#pragma unroll
                for (int i = 0; i < NW; i++) {   // waves hold ascending ids only within a step: compare them
                    const int2 o = slot[i];
                    const bool take = (o.x > g) | ((o.x == g) & (o.y < bv));
                    g = take ? o.x : g;
                    bv = take ? o.y : bv;
                }
            }
            // the same in every lane: kept in scalar registers, so that the
            // serial decisions below are scalar branches
            bv = wave_read(bv, 0);
            const int32_t bg = wave_read(g, 0);
            if (bg == INT32_MIN) break;
            const int32_t rb = wave_read(M.row(bv), 0), re = wave_read(M.row(bv + 1), 0);
            const int32_t wv = wave_read(G.vw[bv], 0);
            int32_t x[P], w[P];   // the row, on its way while the move is judged
            G.load(rb + tid, re, NT, x, w);
            newcut -= bg;
            int64_t dd = ideal0 - pw0;
            dd = dd < 0 ? -dd : dd;
            const int64_t into = (from ? pw0 : pw1) + wv, outof = (from ? pw1 : pw0) - wv;
            // selects instead of short-circuit branches: as `if ((a && b) || (c && d))`
            // around the three assignments this is compiled (ROCm 7.2, all operands
            // in scalar registers) into a jump for c && d that lands behind the move
            // of mincutorder and before those of mincut and mindiff
            const bool keep = ((newcut < mincut) & (into <= onemax) & (outof <= onemax)) |
                              ((newcut == mincut) & (dd < mindiff));
            if (!keep && nswaps - mincutorder > limit) break;
            mincut = keep ? newcut : mincut;
            mindiff = keep ? dd : mindiff;
            mincutorder = keep ? nswaps : mincutorder;
            pw0 = from ? into : outof;
            pw1 = from ? outof : into;
            if (tid == 0) {
                M.st[bv] = (uint8_t)((M.st[bv] ^ kStSide) | kStMoved);
                swaps[nswaps] = (Q)bv;
            }
            trial_move<NT, P, Q>(G, M, bv, from, rb, re, x, w);
            __syncthreads();
        }
        __syncthreads();   // the swap list is whole
        for (int32_t i = tid; i < nswaps; i += NT) M.st[swaps[i]] &= (uint8_t)~kStMoved;
        __syncthreads();
        for (nswaps--; nswaps > mincutorder; nswaps--) {
            const int32_t v = wave_read((int32_t)swaps[nswaps], 0);
            const int from = wave_read((int32_t)M.st[v], 0) & kStSide;
            const int32_t rb = wave_read(M.row(v), 0), re = wave_read(M.row(v + 1), 0);
            const int32_t wv = wave_read(G.vw[v], 0);
            int32_t x[P], w[P];
            G.load(rb + tid, re, NT, x, w);
            __syncthreads();   // every thread has read v's side
            if (tid == 0) M.st[v] ^= kStSide;
            pw0 += from ? wv : -wv;
            pw1 += from ? -wv : wv;
            trial_move<NT, P, Q>(G, M, v, from, rb, re, x, w);
            __syncthreads();
        }
        cut = mincut;
        if (mincutorder <= 0 || mincut == initcut) break;
    }
    return cut;
}

template <int NT>
__global__ void __launch_bounds__(NT) k_ip_trials(const int32_t *__restrict__ act, int32_t nact,
                                                  const Node *__restrict__ nodes, const int32_t *total,
                                                  const eid_t *__restrict__ fx, const vid_t *__restrict__ fadj,
                                                  const wgt_t *__restrict__ fw, const wgt_t *__restrict__ fvw,
                                                  const int32_t *__restrict__ fwd, uint64_t seed, int32_t fm_passes,
                                                  int32_t lds_cap,
                                                  uint8_t *__restrict__ trial_where, char *__restrict__ gscratch,
                                                  int64_t *__restrict__ tcut)
{
    extern __shared__ __align__(16) char lds[];
    __shared__ TrialShared<NT> S;
    const int32_t gw = blockIdx.x;
    if (gw >= *total) return;
    const int32_t nid = trial_node(act, nact, nodes, gw);
    const Node nd = nodes[nid];
    const int32_t t = gw - nd.trial_off, n = nd.end - nd.start;
    const eid_t fb = fx[nd.start];
    const TrialRows G{fadj + fb, fw + fb, fvw + nd.start, nd.start};
    const uint8_t *st;
    int64_t cut;
    if (n <= lds_cap) {   // a 16-bit queue: lds_cap < 2^16
        cut = scan_trial<NT, uint16_t>(G, lds, n, nd, nid, t, fx, fwd, seed, fm_passes, S);
        st = ScanMem<uint16_t>(lds, n, fx + nd.start).st;
    } else {
        char *base = gscratch + nd.soff + (int64_t)t * ((trial_bytes(n, false, false) + 255) & ~255ll);
        cut = scan_trial<NT, int32_t>(G, base, n, nd, nid, t, fx, fwd, seed, fm_passes, S);
        st = ScanMem<int32_t>(base, n, fx + nd.start).st;
    }
    uint8_t *out = trial_where + nd.woff + (int64_t)t * n;
    for (int32_t i = threadIdx.x; i < n; i += NT) out[i] = st[i] & kStSide;
    if (threadIdx.x == 0) tcut[gw] = cut;
}

// ---------------------------------------------------------------- dense scan FM

// The same trial on a dense copy of the node's graph, for coarsest graphs of
// up to kDenseN vertices with strictly ascending rows.  A trial is bound by the
// latency of its serial steps; on lists a step was index load, weight load,
// LDS atomics per neighbour, then a scan of LDS.  Here
//  * a thread owns 4 or 8 vertices for the whole trial, their state in
//    registers: S0 (edge weight to side 0), row weight, side, moved;
//  * moving v adds or subtracts row v of the weight matrix W: one 16-byte load
//    per 4 vertices, no indices and no atomics, whatever the row's length; the
//    sums do not depend on the order, so a pass is undone, and the sums after
//    the BFS are made, with many rows in flight;
//  * a BFS step is one word of the adjacency bit matrix per lane, masked with
//    the unvisited ones;
//  * a move takes one barrier (none with one wave).
// The matrices are built once per depth (5-9 us).  All depths of a partition
// (one wave per trial on lists -> this): R-MAT 2^22, k = 256 (999 vertices,
// 297k entries) 5.6 -> 1.6 ms, R-MAT 2^17, k = 1000 (1945 vertices) 17.5 ->
// 3.8 ms, 3-D RGG 2^20, k = 64 (430 vertices) 3.3 -> 1.2 ms.
constexpr int32_t kDenseN = 4096;

struct DenseNode {
    const int32_t *W;      // n rows of `stride` words (a multiple of 4, zero past n)
    const uint32_t *B;     // n rows of `words` words
    const wgt_t *vw;
    const int32_t *wd;
    int32_t n, stride, words;
};

__host__ __device__ inline int64_t dense_stride(int64_t n) { return (n + 3) & ~3ll; }
__host__ __device__ inline int64_t dense_words(int64_t n) { return (n + 31) / 32; }

// Rows of the weight and bit matrices of the depth's active nodes: a block per
// vertex spreads its list row in LDS and writes it out in order.
__global__ void __launch_bounds__(256) k_ip_dense(int32_t n, const int32_t *__restrict__ node_of,
                                                  const Node *__restrict__ nodes, const eid_t *__restrict__ fx,
                                                  const vid_t *__restrict__ fadj, const wgt_t *__restrict__ fw,
                                                  int32_t *__restrict__ W, uint32_t *__restrict__ B)
{
    extern __shared__ int32_t row[];
    const int32_t v = blockIdx.x, tid = threadIdx.x;
    const Node &nd = nodes[node_of[v]];
    if (nd.k < 2) return;
    const int32_t nn = nd.end - nd.start, s0 = nd.start;
    const int32_t stride = (int32_t)dense_stride(nn), words = (int32_t)dense_words(nn);
    for (int32_t i = tid; i < words * 32; i += 256) row[i] = 0;
    __syncthreads();
    const eid_t e = fx[v + 1];
#pragma unroll 4
    for (eid_t j = fx[v] + tid; j < e; j += 256) row[fadj[j] - s0] = fw[j];
    __syncthreads();
    int32_t *wr = W + nd.doff + (int64_t)(v - s0) * stride;
    for (int32_t i = tid; i < stride; i += 256) wr[i] = row[i];
    uint32_t *br = B + nd.boff + (int64_t)(v - s0) * words;
    for (int32_t i0 = tid & ~(kWave - 1); i0 < words * 32; i0 += 256) {   // whole waves, 64 entries each
        const int32_t i = i0 + lane_id();
        const uint64_t m = __ballot(i < words * 32 && row[i] != 0);
        if (lane_id() < 2 && i0 / 32 + lane_id() < words) br[i0 / 32 + lane_id()] = (uint32_t)(m >> (32 * lane_id()));
    }
}

// trial_grow on the bit matrix (WPL words per lane): lists the vertices of side
// 0 in `taken` and sets their side bytes to 0; returns their number and weight.
template <int WPL>
__device__ inline int32_t dense_grow(const DenseNode &D, uint16_t *queue, uint16_t *taken, uint8_t *side,
                                     const Node &nd, int32_t nid, int32_t t, uint64_t seed, int64_t &w0)
{
    const int lane = lane_id();
    const int32_t n = D.n;
    const int64_t onemin = nd.onemin, onemax = nd.onemax;
    int64_t pw0 = 0, pw1 = nd.tv;
    int32_t draw = 0, nt = 0;
    const int32_t start = trial_start(nd, nid, n, t, seed, draw);
    int32_t first = 0, last = 1, nleft = n - 1, drain = 0;
    uint32_t open[WPL];   // unvisited vertices among this lane's 32 * WPL
#pragma unroll
    for (int q = 0; q < WPL; q++) {
        const int32_t left = n - (lane * WPL + q) * 32;
        open[q] = left >= 32 ? ~0u : (left > 0 ? (1u << left) - 1u : 0u);
    }
    auto visit = [&](int32_t v) {
        if (lane == 0) queue[0] = (uint16_t)v;
#pragma unroll
        for (int q = 0; q < WPL; q++)
            if (v / 32 == lane * WPL + q) open[q] &= ~(1u << (v & 31));
    };
    auto load_row = [&](int32_t v, uint32_t (&b)[WPL]) {
#pragma unroll
        for (int q = 0; q < WPL; q++) {
            const int32_t i = lane * WPL + q;
            b[q] = i < D.words ? D.B[(int64_t)v * D.words + i] : 0u;
        }
    };
    visit(start);
    wave_lds_sync();
    int32_t ahead = -1, av = 0, aw = 0;   // the next vertex of the queue, loaded ahead
    uint32_t ab[WPL];
    for (;;) {
        if (first == last) {
            if (nleft == 0 || drain) break;
            // restart from the r-th unvisited vertex in id order
            int32_t r = (int32_t)(trial_rng(seed, (uint32_t)nid, t, draw++) % (uint64_t)nleft);
            int32_t own = 0;
#pragma unroll
            for (int q = 0; q < WPL; q++) own += __popc(open[q]);
            const int32_t before = wave_inclusive_scan(own) - own;
            int32_t v = -1;
            if (r >= before && r < before + own) {
                r -= before;
#pragma unroll
                for (int q = 0; q < WPL; q++) {
                    uint32_t b = open[q];
                    const int32_t c = __popc(b);
                    if (v < 0 && r < c) {
                        for (; r > 0; r--) b &= b - 1;
                        v = (lane * WPL + q) * 32 + (__ffs(b) - 1);
                    }
                    r -= c;
                }
            }
            v = wave_max(v);
            visit(v);
            wave_lds_sync();
            first = 0;
            last = 1;
            nleft--;
            ahead = -1;
        }
        int32_t v, wv;
        uint32_t b[WPL];
        if (ahead == first) {
            v = av;
            wv = aw;
#pragma unroll
            for (int q = 0; q < WPL; q++) b[q] = ab[q];
        } else {
            v = wave_read((int32_t)queue[first], 0);
            wv = D.vw[v];
            load_row(v, b);
        }
        first++;
        if (first < last) {
            ahead = first;
            av = wave_read((int32_t)queue[first], 0);
            aw = D.vw[av];
            load_row(av, ab);
        }
        wv = wave_read(wv, 0);
        if (pw0 > 0 && pw1 - wv < onemin) { drain = 1; continue; }
        pw0 += wv;
        pw1 -= wv;
        if (lane == 0) {
            side[v] = 0;
            taken[nt] = (uint16_t)v;
        }
        nt++;
        if (pw1 <= onemax) break;
        drain = 0;
        // the unvisited neighbours join the queue in id (row) order
        int32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < WPL; q++) {
            b[q] &= open[q];
            open[q] &= ~b[q];
            cnt += __popc(b[q]);
        }
        const int32_t incl = wave_inclusive_scan(cnt), tot = wave_read(incl, kWave - 1);
        int32_t at = last + incl - cnt;
#pragma unroll
        for (int q = 0; q < WPL; q++) {
            uint32_t f = b[q];
            while (f) {
                queue[at++] = (uint16_t)((lane * WPL + q) * 32 + (__ffs(f) - 1));
                f &= f - 1;
            }
        }
        last += tot;
        nleft -= tot;
        wave_lds_sync();
    }
    w0 = pw0;
    return nt;
}

template <int NT>
struct DenseShared {
    int2 best[2][NT / kWave];   // each wave's (gain, vertex), by parity of the move
    int64_t sum[NT / kWave];
    int64_t pw0;
    int32_t ntaken;
};

template <int NT>
__device__ inline void trial_sync()
{
    if constexpr (NT == kWave) wave_lds_sync();   // (the block's other waves have left)
    else __syncthreads();
}

// LDS of a dense trial: queue / swap list and taken list (u16), side bytes.
__host__ __device__ inline int64_t dense_bytes(int64_t n) { return 5 * dense_stride(n) + 16; }

template <int NT, int V, int NTMAX>
__device__ inline int64_t dense_trial(const DenseNode &D, char *lds, const Node &nd, int32_t nid, int32_t t,
                                      uint64_t seed, int32_t fm_passes, DenseShared<NTMAX> &S,
                                      uint8_t *__restrict__ out)
{
    constexpr int NW = NT / kWave, C = V / 4;
    const int tid = threadIdx.x, lane = lane_id();
    const int32_t n = D.n, n4 = D.stride;
    uint16_t *queue = (uint16_t *)lds, *taken = queue + n4;
    uint8_t *sideb = (uint8_t *)(taken + n4);
    for (int32_t i = tid * 4; i < n4; i += NT * 4) *(uint32_t *)(sideb + i) = 0x01010101u;
    trial_sync<NT>();
    if (tid < kWave) {
        int64_t w0;
        const int32_t nt = n <= 2048 ? dense_grow<1>(D, queue, taken, sideb, nd, nid, t, seed, w0)
                                     : dense_grow<2>(D, queue, taken, sideb, nd, nid, t, seed, w0);
        if (tid == 0) {
            S.pw0 = w0;
            S.ntaken = nt;
        }
    }
    trial_sync<NT>();
    int64_t pw0 = S.pw0, pw1 = nd.tv - S.pw0;
    const int64_t ideal0 = nd.ideal0, ideal1 = nd.tv - nd.ideal0;
    const int64_t onemax = nd.onemax;

    // the thread's vertices: chunk c holds u = c*4*NT + 4*tid .. + 3
    int32_t s[V], wd[V];
    uint32_t side = 0, gone = 0, alone = 0;   // bits: side 1; outside the node; no edges
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int32_t u0 = c * 4 * NT + 4 * tid;
        const uint32_t s4 = u0 < n4 ? *(const uint32_t *)(sideb + u0) : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = c * 4 + j;
            const bool in = u0 + j < n;
            s[i] = 0;
            wd[i] = in ? D.wd[u0 + j] : 0;
            side |= (in ? (s4 >> (8 * j)) & 1u : 0u) << i;
            gone |= (in ? 0u : 1u) << i;
            alone |= (in && wd[i] == 0 ? 1u : 0u) << i;
        }
    }
    // s += sign * row v; w[] holds the row's pieces
    auto load = [&](int32_t v, int4 (&w)[C]) {
        const int32_t *r = D.W + (int64_t)v * n4;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int32_t u0 = c * 4 * NT + 4 * tid;
            w[c] = u0 < n4 ? *(const int4 *)(r + u0) : make_int4(0, 0, 0, 0);
        }
    };
    auto add = [&](int sign, const int4 (&w)[C]) {
#pragma unroll
        for (int c = 0; c < C; c++) {
            s[c * 4] += sign * w[c].x;
            s[c * 4 + 1] += sign * w[c].y;
            s[c * 4 + 2] += sign * w[c].z;
            s[c * 4 + 3] += sign * w[c].w;
        }
    };
    // sums over lists of rows: R rows in flight
    constexpr int R = V == 4 ? 4 : 2;
    {
        const int32_t nt = S.ntaken;
        for (int32_t i = 0; i < nt; i += R) {
            int4 w[R][C];
#pragma unroll
            for (int r = 0; r < R; r++)
                load(wave_read((int32_t)taken[i + r < nt ? i + r : i], 0), w[r]);
#pragma unroll
            for (int r = 0; r < R; r++)
                if (i + r < nt) add(1, w[r]);
        }
    }
    // the cut: every cut edge once, from its end in side 1
    int64_t cut = 0;
#pragma unroll
    for (int i = 0; i < V; i++) cut += (side >> i) & 1u ? s[i] : 0;
    cut = wave_sum(cut);
    if constexpr (NW > 1) {
        if (lane == 0) S.sum[tid / kWave] = cut;
        __syncthreads();
        cut = 0;
#pragma unroll
        for (int i = 0; i < NW; i++) cut += S.sum[i];
    }

    int64_t limit = n / 100;
    if (limit < 15) limit = 15;
    if (limit > 100) limit = 100;
    uint16_t *swaps = queue;   // vertex, with the side it left in bit 15
    for (int32_t pass = 0; pass < fm_passes; pass++) {
        int64_t mincutorder = -1;
        int64_t newcut = cut, mincut = cut, initcut = cut;
        int64_t d0 = ideal0 - pw0;
        int64_t mindiff = d0 < 0 ? -d0 : d0;
        uint32_t out_of_play = gone;   // and moved in this pass
        int32_t nswaps;
        for (nswaps = 0; nswaps < n; nswaps++) {
            const int from = (ideal0 - pw0 < ideal1 - pw1) ? 0 : 1;
            // the boundary vertex of side `from`, not moved in this pass, of
            // largest gain (2 ed - wd; |gain| < 2^30), the smallest id among equals
            const uint32_t play = (from ? side : ~side) & ~out_of_play;
            int32_t g = INT32_MIN, bv = INT32_MAX;
#pragma unroll
            for (int i = 0; i < V; i++) {
                const int32_t ed = from ? s[i] : wd[i] - s[i];
                const bool can = ((play >> i) & 1u) != 0 && (ed > 0 || ((alone >> i) & 1u) != 0);
                const int32_t gi = can ? 2 * ed - wd[i] : INT32_MIN;
                bv = gi > g ? (i / 4) * 4 * NT + 4 * tid + (i & 3) : bv;
                g = gi > g ? gi : g;
            }
            const int32_t gm = lanes_reduce<kWave>(g, [](int32_t a, int32_t b) { return a > b ? a : b; });
            bv = lanes_reduce<kWave>(g == gm ? bv : INT32_MAX, [](int32_t a, int32_t b) { return a < b ? a : b; });
            g = gm;
            if constexpr (NW > 1) {
                int2 *slot = S.best[nswaps & 1];
                if (lane == 0) slot[tid / kWave] = make_int2(g, bv);
                __syncthreads();
                g = INT32_MIN;
                bv = INT32_MAX;
#pragma unroll
                for (int i = 0; i < NW; i++) {
                    const int2 o = slot[i];
                    const bool take = (o.x > g) | ((o.x == g) & (o.y < bv));
                    g = take ? o.x : g;
                    bv = take ? o.y : bv;
                }
            }
            // the same in every lane: kept in scalar registers, so that the
            // serial decisions below are scalar branches
            bv = wave_read(bv, 0);
            const int32_t bg = wave_read(g, 0);
            if (bg == INT32_MIN) break;
            int4 w[C];   // the row, on its way while the move is judged
            load(bv, w);
            const int32_t wv = wave_read(D.vw[bv], 0);
            newcut -= bg;
            int64_t dd = ideal0 - pw0;
            dd = dd < 0 ? -dd : dd;
            const int64_t into = (from ? pw0 : pw1) + wv, outof = (from ? pw1 : pw0) - wv;
            // (selects for the reason given in scan_trial)
            const bool keep = ((newcut < mincut) & (into <= onemax) & (outof <= onemax)) |
                              ((newcut == mincut) & (dd < mindiff));
            if (!keep && nswaps - mincutorder > limit) break;
            mincut = keep ? newcut : mincut;
            mindiff = keep ? dd : mindiff;
            mincutorder = keep ? nswaps : mincutorder;
            pw0 = from ? into : outof;
            pw1 = from ? outof : into;
            const uint32_t own = (bv >> 2) % NT == tid ? 1u << ((bv / (4 * NT)) * 4 + (bv & 3)) : 0u;
            side ^= own;
            out_of_play |= own;
            if (tid == 0) swaps[nswaps] = (uint16_t)(bv | (from << 15));
            add(from ? 1 : -1, w);
        }
        trial_sync<NT>();   // the swap list is whole
        for (int32_t i = (int32_t)mincutorder + 1; i < nswaps; i += R) {
            int4 w[R][C];
            int32_t x[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                x[r] = wave_read((int32_t)swaps[i + r < nswaps ? i + r : i], 0);
                load(x[r] & 0x7FFF, w[r]);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (i + r >= nswaps) break;
                const int32_t v = x[r] & 0x7FFF, back = x[r] >> 15;   // back to side `back`
                const int32_t wv = wave_read(D.vw[v], 0);
                pw0 += back ? -wv : wv;
                pw1 += back ? wv : -wv;
                side ^= (v >> 2) % NT == tid ? 1u << ((v / (4 * NT)) * 4 + (v & 3)) : 0u;
                add(back ? -1 : 1, w[r]);
            }
        }
        cut = mincut;
        if (mincutorder <= 0 || mincut == initcut) break;
        trial_sync<NT>();   // every wave has read the swap list
    }
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int32_t u = (i / 4) * 4 * NT + 4 * tid + (i & 3);
        if (u < n) out[u] = (uint8_t)((side >> i) & 1u);
    }
    return cut;
}

// A block of NTMAX threads per trial; node graphs of up to 256 vertices keep
// one wave of it (4 vertices a thread), larger ones 4 or 8 vertices a thread
// (up to 8 * NTMAX vertices).
template <int NTMAX>
__global__ void __launch_bounds__(NTMAX) k_ip_trials_dense(const int32_t *__restrict__ act, int32_t nact,
                                                           const Node *__restrict__ nodes, const int32_t *total,
                                                           const int32_t *__restrict__ W,
                                                           const uint32_t *__restrict__ B,
                                                           const wgt_t *__restrict__ fvw,
                                                           const int32_t *__restrict__ fwd, uint64_t seed,
                                                           int32_t fm_passes, uint8_t *__restrict__ trial_where,
                                                           int64_t *__restrict__ tcut)
{
    extern __shared__ __align__(16) char lds[];
    __shared__ DenseShared<NTMAX> S;
    const int32_t gw = blockIdx.x;
    if (gw >= *total) return;
    const int32_t nid = trial_node(act, nact, nodes, gw);
    const Node nd = nodes[nid];
    const int32_t t = gw - nd.trial_off;
    DenseNode D;
    D.n = nd.end - nd.start;
    D.stride = (int32_t)dense_stride(D.n);
    D.words = (int32_t)dense_words(D.n);
    D.W = W + nd.doff;
    D.B = B + nd.boff;
    D.vw = fvw + nd.start;
    D.wd = fwd + nd.start;
    uint8_t *out = trial_where + nd.woff + (int64_t)t * D.n;
    int64_t cut;
    if (D.n <= 4 * kWave) {
        if (threadIdx.x >= kWave) return;
        cut = dense_trial<kWave, 4, NTMAX>(D, lds, nd, nid, t, seed, fm_passes, S, out);
    } else if (D.n <= 4 * NTMAX) {
        cut = dense_trial<NTMAX, 4, NTMAX>(D, lds, nd, nid, t, seed, fm_passes, S, out);
    } else {
        cut = dense_trial<NTMAX, 8, NTMAX>(D, lds, nd, nid, t, seed, fm_passes, S, out);
    }
    if (threadIdx.x == 0) tcut[gw] = cut;
}

// Arg-min cut over a node's trials, first minimum wins (:3713-3812).
__global__ void __launch_bounds__(256) k_ip_select(const int32_t *__restrict__ act, Node *nodes,
                                                   const int64_t *__restrict__ tcut)
{
    __shared__ int64_t sc[256];
    __shared__ int32_t si[256];
    Node &nd = nodes[act[blockIdx.x]];
    int64_t bc = INT64_MAX;
    int32_t bi = -1;
    for (int32_t t = threadIdx.x; t < nd.T; t += blockDim.x) {
        int64_t c = tcut[nd.trial_off + t];
        if (c < bc) { bc = c; bi = t; }
    }
    sc[threadIdx.x] = bc;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            int64_t oc = sc[threadIdx.x + s];
            int32_t oi = si[threadIdx.x + s];
            if (oi != -1 && (si[threadIdx.x] == -1 || oc < sc[threadIdx.x] ||
                             (oc == sc[threadIdx.x] && oi < si[threadIdx.x]))) {
                sc[threadIdx.x] = oc;
                si[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) nd.best = si[0];
}

// Write the winning bisection through the labels (:3896-3902) and record
// each vertex's side for the split (-1 for vertices of finished nodes).
__global__ void k_ip_side(int32_t n, const int32_t *__restrict__ node_of, const Node *__restrict__ nodes,
                          const uint8_t *__restrict__ trial_where, const int32_t *__restrict__ label,
                          int32_t *__restrict__ part, int8_t *__restrict__ side)
{
    int32_t v = (int32_t)((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (v >= n) return;
    const Node &nd = nodes[node_of[v]];
    if (nd.k < 2 || nd.best < 0) { side[v] = -1; return; }
    int32_t nn = nd.end - nd.start;
    uint8_t w = trial_where[nd.woff + (int64_t)nd.best * nn + (v - nd.start)];
    part[label[v]] = nd.fpart + w;
    side[v] = (int8_t)w;
}

__global__ void __launch_bounds__(256) k_ip_count0(const int32_t *__restrict__ act, Node *nodes, int32_t ntab,
                                                   const int8_t *__restrict__ side)
{
    __shared__ int32_t sh[4];
    int32_t id = act[blockIdx.x];
    Node &nd = nodes[id];
    int32_t s = 0;
    for (int32_t v = nd.start + threadIdx.x; v < nd.end; v += blockDim.x) s += side[v] == 0;
    s = wave_sum(s);
    if (lane_id() == 0) sh[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t c0 = sh[0] + sh[1] + sh[2] + sh[3];
        nd.cnt0 = c0;
        if (2 * id + 1 < ntab) {
            nodes[2 * id].start = nd.start;
            nodes[2 * id].end = nd.start + c0;
            nodes[2 * id + 1].start = nd.start + c0;
            nodes[2 * id + 1].end = nd.end;
        }
    }
}

__global__ void k_ip_f0(int32_t n, const int8_t *__restrict__ side, int32_t *__restrict__ f0)
{
    int32_t v = (int32_t)((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (v < n) f0[v] = side[v] == 0;
}

// Order-preserving split (hunyuangraph_GPU_splitgraph.h:802-944): side-0
// vertices first, then side-1, each in their old order, inside the node's
// range.  Rows keep only same-side entries; finished nodes drop their rows.
// A wave per vertex: the rows of the coarsest graph are long (a thread per
// row took 97 us a launch for 2000 rows of about 200 entries).
__global__ void __launch_bounds__(kRowBS) k_ip_pos(int32_t n, const int32_t *__restrict__ node_of,
                                                   const Node *__restrict__ nodes, const int8_t *__restrict__ side,
                                                   const int32_t *__restrict__ s0, const eid_t *__restrict__ fx,
                                                   const vid_t *__restrict__ fadj, int32_t *__restrict__ pos,
                                                   int32_t *__restrict__ nnode_of, int32_t *__restrict__ nlabel,
                                                   const int32_t *__restrict__ label, wgt_t *__restrict__ nfvw,
                                                   const wgt_t *__restrict__ fvw, int64_t *__restrict__ ndeg)
{
    const int32_t v = (int32_t)gindex<kWave>();
    if (v >= n) return;   // whole waves
    const int lane = lane_id();
    const int32_t id = node_of[v];
    const int8_t sd = side[v];
    int32_t p = v, d = 0, nid = id;
    if (sd >= 0) {
        const Node &nd = nodes[id];
        const int32_t before = nd.start > 0 ? s0[nd.start - 1] : 0;
        const int32_t rank0 = (s0[v] - (sd == 0 ? 1 : 0)) - before;
        const int32_t rank1 = (v - nd.start) - rank0;
        p = sd == 0 ? nd.start + rank0 : nd.start + nd.cnt0 + rank1;
        nid = 2 * id + sd;
        const eid_t je = fx[v + 1];
#pragma unroll 4
        for (eid_t j = fx[v] + lane; j < je; j += kWave) d += side[fadj[j]] == sd;
        d = wave_sum(d);
    }
    if (lane == 0) {
        nnode_of[p] = nid;
        pos[v] = p;
        nlabel[p] = label[v];
        nfvw[p] = fvw[v];
        ndeg[p] = d;
    }
}

// The same-side entries of each row, in row order, at the row's new place, and
// their total weight: a wave per row, ranked by ballots.
__global__ void __launch_bounds__(kRowBS) k_ip_edges(int32_t n, const int8_t *__restrict__ side,
                                                     const int32_t *__restrict__ pos, const eid_t *__restrict__ fx,
                                                     const vid_t *__restrict__ fadj, const wgt_t *__restrict__ fw,
                                                     const eid_t *__restrict__ nfx, vid_t *__restrict__ nfadj,
                                                     wgt_t *__restrict__ nfw, int32_t *__restrict__ nfwd)
{
    constexpr int P = 4;   // 64-entry pieces in flight
    const int32_t v = (int32_t)gindex<kWave>();
    if (v >= n) return;   // whole waves
    const int lane = lane_id();
    const int8_t sd = side[v];
    if (sd < 0) return;
    const int32_t np = pos[v];
    eid_t o = nfx[np];
    int32_t wsum = 0;
    const eid_t je = fx[v + 1];
    for (eid_t j0 = fx[v]; j0 < je; j0 += P * kWave) {
        int32_t x[P], w[P];
#pragma unroll
        for (int q = 0; q < P; q++) {
            const eid_t j = j0 + lane + q * kWave;
            x[q] = j < je ? fadj[j] : -1;
            w[q] = j < je ? fw[j] : 0;
        }
#pragma unroll
        for (int q = 0; q < P; q++) x[q] = x[q] >= 0 && side[x[q]] == sd ? pos[x[q]] : -1;
#pragma unroll
        for (int q = 0; q < P; q++) {
            const uint64_t m = __ballot(x[q] >= 0);
            if (x[q] >= 0) {
                const eid_t at = o + __popcll(m & lanemask_lt());
                nfadj[at] = x[q];
                nfw[at] = w[q];
                wsum += w[q];
            }
            o += __popcll(m);
        }
    }
    wsum = wave_sum(wsum);
    if (lane == 0) nfwd[np] = wsum;
}

struct TreeNode { int32_t id, k, fpart; };

// fm_kind -1 picks the queue-driven FM (the same moves as the scan) once the
// coarsest graph is large enough for O(log n) queue steps to beat an O(n/64)
// scan per move.
bool fm_uses_heap(int32_t fm_kind, int32_t n)
{
    if (fm_kind >= 0) return fm_kind != 0;
    return n >= kAutoHeapMinVertices;
}

}  // namespace

// The matrices and, on top, what the scans after them take.
size_t dense_trial_bytes(int32_t n)
{
    if (n > kDenseN) return 0;
    return sizeof(int32_t) * (size_t)(n * (dense_stride(n) + 3) + n * (dense_words(n) + 1)) + (64 << 10);
}

void initial_partition(Ctx &c, const DevGraph &g, int32_t k, const Params &p, int32_t *where)
{
    int32_t n = g.n;
    if (n <= 0) return;
    fill<int32_t>(c, where, n, 0);
    if (k <= 1) return;

    // tree shape depends on k only
    std::vector<std::vector<TreeNode>> depth_nodes;
    std::vector<TreeNode> cur{{1, k, 0}};
    int32_t maxid = 1;
    while (!cur.empty()) {
        depth_nodes.push_back(cur);
        std::vector<TreeNode> nxt;
        for (auto &t : cur) {
            int32_t kl = t.k >> 1, kr = t.k - kl;
            maxid = std::max(maxid, 2 * t.id + 1);
            if (t.k > 2) {
                if (kl >= 2) nxt.push_back({2 * t.id, kl, t.fpart});
                if (kr >= 2) nxt.push_back({2 * t.id + 1, kr, t.fpart + kl});
            }
        }
        cur.swap(nxt);
    }
    int32_t ntab = maxid + 1;
    std::vector<Node> htab(ntab);
    for (auto &t : htab) { t.start = t.end = 0; t.k = 1; t.fpart = 0; t.best = -1; t.T = 0; }
    {
        // k and fpart of every tree node (leaves included)
        std::vector<TreeNode> stack{{1, k, 0}};
        while (!stack.empty()) {
            TreeNode t = stack.back();
            stack.pop_back();
            if (t.id >= ntab) continue;
            htab[t.id].k = t.k;
            htab[t.id].fpart = t.fpart;
            if (t.k >= 2) {
                stack.push_back({2 * t.id, t.k >> 1, t.fpart});
                stack.push_back({2 * t.id + 1, t.k - (t.k >> 1), t.fpart + (t.k >> 1)});
            }
        }
    }

    double ub = std::pow((double)p.ub_num / (double)p.ub_den, 1.0 / std::log((double)k));
    const bool heap = fm_uses_heap(p.fm_kind, n);
    const int32_t fm_kind = p.fm_kind < 0 ? (heap ? 1 : 0) : p.fm_kind;
    int32_t lds_cap = heap ? (kHeapLdsBudget - 64) / kHeapBytesPerVertex : kScanLdsN;
    int32_t lds_n = std::min(n, lds_cap);
    size_t lds_bytes = (size_t)trial_bytes(lds_n, heap, true) + 16;

    size_t mark = c.arena.right_mark();
    Node *nodes = c.arena.ralloc<Node>((size_t)ntab);
    // active node ids of every depth, back to back
    std::vector<int32_t> hact;
    std::vector<size_t> act_off;
    for (auto &dn : depth_nodes) {
        act_off.push_back(hact.size());
        for (auto &t : dn) hact.push_back(t.id);
    }
    int32_t *act_all = c.arena.ralloc<int32_t>(hact.size());
    upload_staged(c, nodes, htab.data(), sizeof(Node) * (size_t)ntab);
    upload_staged(c, act_all, hact.data(), sizeof(int32_t) * hact.size());
    int32_t *total = c.arena.ralloc<int32_t>(1);
    int64_t maxtrials = (int64_t)std::min(p.trials, n);
    uint8_t *trial_where = c.arena.ralloc<uint8_t>((size_t)(maxtrials * n));
    char *gscratch = nullptr;
    if (n > lds_cap) {
        // sum over nodes of T * round256(trial_bytes(nn)): trial_bytes is affine
        // in nn but for a constant below 80 a node, and at most n / lds_cap + 1
        // nodes use global scratch
        size_t gs = (size_t)maxtrials * ((size_t)trial_bytes(n, heap, false) + 512 * ((size_t)(n / lds_cap) + 1));
        gscratch = c.arena.ralloc<char>(gs);
    }
    // trials of one depth: sum of min(trials, n_node) <= n
    int64_t *tcut = c.arena.ralloc<int64_t>((size_t)n + 1);
    int32_t *node_of[2], *label[2], *fwd[2];
    wgt_t *fvw[2], *fw[2];
    eid_t *fx[2];
    vid_t *fadj[2];
    int64_t mm = g.m > 0 ? g.m : 1;
    for (int b = 0; b < 2; b++) {
        node_of[b] = c.arena.ralloc<int32_t>((size_t)n);
        label[b] = c.arena.ralloc<int32_t>((size_t)n);
        fvw[b] = c.arena.ralloc<wgt_t>((size_t)n);
        fwd[b] = c.arena.ralloc<int32_t>((size_t)n);
        fx[b] = c.arena.ralloc<eid_t>((size_t)n + 1);
        fadj[b] = c.arena.ralloc<vid_t>((size_t)mm);
        fw[b] = c.arena.ralloc<wgt_t>((size_t)mm);
    }
    int8_t *side = c.arena.ralloc<int8_t>((size_t)n);
    int32_t *f0 = c.arena.ralloc<int32_t>((size_t)n);
    int32_t *pos = c.arena.ralloc<int32_t>((size_t)n);
    int64_t *ndeg = c.arena.ralloc<int64_t>((size_t)n);
    // dense trials: the graph as matrices, rebuilt per depth node by node.  They
    // take 69 MB at 4096 vertices, more than the whole estimate of a small graph
    // whose coarsening stops early (pairs, mostly isolated vertices), and the
    // lists a few MB for the same moves: dense only where the arena as it is has
    // room for them, so that no call grows its arena or its claim on a budget
    // for them.
    const bool dense = !heap && g.ascending && n <= kDenseN && c.arena.free_bytes() >= dense_trial_bytes(n);
    int32_t *W = nullptr;
    uint32_t *B = nullptr;
    if (dense) {
        W = c.arena.ralloc<int32_t>((size_t)(n * (dense_stride(n) + 3)));
        B = c.arena.ralloc<uint32_t>((size_t)(n * (dense_words(n) + 1)));
    }

    unsigned gv = grid_for(n, 256);
    k_ip_init<<<grid_groups(n, kWave), kRowBS, 0, c.stream>>>(n, g.vwgt, g.xadj, g.adjwgt, node_of[0], label[0],
                                                             fvw[0], fwd[0], nodes);
    HGP_LAUNCH_CHECK();
    HGP_CHECK_HIP(hipMemcpyAsync(fx[0], g.xadj, sizeof(eid_t) * ((size_t)n + 1), hipMemcpyDeviceToDevice, c.stream));
    if (g.m > 0) {
        HGP_CHECK_HIP(hipMemcpyAsync(fadj[0], g.adjncy, sizeof(vid_t) * (size_t)g.m, hipMemcpyDeviceToDevice, c.stream));
        HGP_CHECK_HIP(hipMemcpyAsync(fw[0], g.adjwgt, sizeof(wgt_t) * (size_t)g.m, hipMemcpyDeviceToDevice, c.stream));
    }

    int cb = 0;
    for (size_t d = 0; d < depth_nodes.size(); d++) {
        const auto &dn = depth_nodes[d];
        int32_t nact = (int32_t)dn.size();
        const int32_t *act = act_all + act_off[d];
        k_ip_setup<<<nact, 256, 0, c.stream>>>(act, nodes, fvw[cb], ub, p.trials);
        HGP_LAUNCH_CHECK();
        k_ip_offsets<<<1, 256, 0, c.stream>>>(act, nact, nodes, lds_cap, heap, total);
        HGP_LAUNCH_CHECK();
        if (dense) {
            KScope ks(c, "k_ip_dense", 0.0);
            k_ip_dense<<<(unsigned)n, 256, 4 * 32 * dense_words(n), c.stream>>>(n, node_of[cb], nodes, fx[cb],
                                                                               fadj[cb], fw[cb], W, B);
            HGP_LAUNCH_CHECK();
        }
        int64_t waves = std::min<int64_t>((int64_t)nact * p.trials, n);
        {
            KScope ks(c, "k_ip_trials", 0.0);
            const unsigned grid = (unsigned)std::max<int64_t>(waves, 1);
            // the average node graph of the depth decides the block size
            const bool wide = n / nact >= kWideTrial;
            if (heap)
                k_ip_trials_heap<<<grid, kWave, lds_bytes, c.stream>>>(act, nact, nodes, total, fx[cb], fadj[cb],
                                                                       fw[cb], fvw[cb], p.seed, p.fm_passes, fm_kind,
                                                                       lds_cap, trial_where, gscratch, tcut);
            else if (dense && n <= 2048)
                k_ip_trials_dense<256><<<grid, 256, dense_bytes(n), c.stream>>>(
                    act, nact, nodes, total, W, B, fvw[cb], fwd[cb], p.seed, p.fm_passes, trial_where, tcut);
            else if (dense)
                k_ip_trials_dense<512><<<grid, 512, dense_bytes(n), c.stream>>>(
                    act, nact, nodes, total, W, B, fvw[cb], fwd[cb], p.seed, p.fm_passes, trial_where, tcut);
            else if (wide)
                k_ip_trials<256><<<grid, 256, lds_bytes, c.stream>>>(act, nact, nodes, total, fx[cb], fadj[cb],
                                                                     fw[cb], fvw[cb], fwd[cb], p.seed, p.fm_passes,
                                                                     lds_cap, trial_where, gscratch, tcut);
            else
                k_ip_trials<kWave><<<grid, kWave, lds_bytes, c.stream>>>(act, nact, nodes, total, fx[cb], fadj[cb],
                                                                         fw[cb], fvw[cb], fwd[cb], p.seed,
                                                                         p.fm_passes, lds_cap, trial_where, gscratch,
                                                                         tcut);
            HGP_LAUNCH_CHECK();
        }
        k_ip_select<<<nact, 256, 0, c.stream>>>(act, nodes, tcut);
        HGP_LAUNCH_CHECK();
        k_ip_side<<<gv, 256, 0, c.stream>>>(n, node_of[cb], nodes, trial_where, label[cb], where, side);
        HGP_LAUNCH_CHECK();
        if (d + 1 == depth_nodes.size()) break;
        k_ip_count0<<<nact, 256, 0, c.stream>>>(act, nodes, ntab, side);
        HGP_LAUNCH_CHECK();
        k_ip_f0<<<gv, 256, 0, c.stream>>>(n, side, f0);
        HGP_LAUNCH_CHECK();
        scan_inclusive(c, f0, f0, n);
        int nb = cb ^ 1;
        k_ip_pos<<<grid_groups(n, kWave), kRowBS, 0, c.stream>>>(n, node_of[cb], nodes, side, f0, fx[cb], fadj[cb], pos, node_of[nb],
                                           label[nb], label[cb], fvw[nb], fvw[cb], ndeg);
        HGP_LAUNCH_CHECK();
        offsets_from_counts(c, ndeg, fx[nb], n);
        k_ip_edges<<<grid_groups(n, kWave), kRowBS, 0, c.stream>>>(n, side, pos, fx[cb], fadj[cb], fw[cb], fx[nb], fadj[nb], fw[nb],
                                                                    fwd[nb]);
        HGP_LAUNCH_CHECK();
        cb = nb;
    }
    c.arena.right_release(mark);
}

}  // namespace hgp
