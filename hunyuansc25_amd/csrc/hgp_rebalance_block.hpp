// hgp_rebalance_block.hpp -- the rebalancing step of one level inside one block
// of kRbBS threads: used by the single-launch step of small levels and by the
// one-block Jet loop.
#pragma once

#include "hgp_group.hpp"
#include "hgp_jet.hpp"

namespace hgp {

constexpr int kRbBS = 1024;                  // threads of the sorting blocks
constexpr int kRbNW = kRbBS / kWave;
// Ranks of a wave's items by digit, in row-major order, on top of the counts
// in my[256] (advanced past the items): row r of the wave is d[r] of its 64
// lanes, live bit r tells whether the lane's item takes part.
template <int R>
__device__ inline void row_ranks(const uint32_t (&d)[R], uint32_t live, int rows, int32_t *my, int32_t (&rk)[R])
{
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;   // the same for the whole wave
        const bool on = (live >> r) & 1u;
        uint64_t m = __ballot(on);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d[r] >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const int32_t base = my[d[r]], low = __popcll(m & lt);
        rk[r] = base + low;
        wave_lds_sync();   // every lane has its base
        if (on && low == 0) my[d[r]] = base + __popcll(m);
        wave_lds_sync();
    }
}

// Turns the counts wc[wave][digit] into the number of items before each
// (digit, wave) in digit order; returns the total.  dsum: 4 ints.
__device__ inline int32_t digit_bases(int32_t (*wc)[256], int32_t *dsum)
{
    const int tid = threadIdx.x, w = tid / kWave;
    int32_t run = 0;
    if (tid < 256) {
#pragma unroll
        for (int x = 0; x < kRbNW; x++) {
            const int32_t c = wc[x][tid];
            wc[x][tid] = run;
            run += c;
        }
        const int32_t incl = wave_inclusive_scan(run);
        if (lane_id() == kWave - 1) dsum[w] = incl;
        run = incl - run;
    }
    __syncthreads();
    const int32_t total = dsum[0] + dsum[1] + dsum[2] + dsum[3];
    if (tid < 256) {
        for (int x = 0; x < w; x++) run += dsum[x];
#pragma unroll
        for (int x = 0; x < kRbNW; x++) wc[x][tid] += run;
    }
    __syncthreads();
    return total;
}

// Cookie cutter (:2710-2745), one wave: slice the evicted list (in sorted
// order, prefix weights bs[0..ne]) into consecutive runs, part by part, each
// filling room[p] = max(0, maxwgt - pwgts[p]).  A slice starts where the last
// one ended, so the parts are a serial chain; what a part costs is the search
// for the first index hi in (start, limit], limit = min(ne, start + room)
// (weights are >= 1), whose prefix reaches bs[start] + room (limit if none).
// The wave walks the prefixes in blocks of 128, the next one always on its way,
// and finds hi in the block at hand with two ballots; the values at hi and
// hi - 1, whose nearer one ends the slice, come from the lanes.  Only a slice
// that reaches more than kCookieFar entries past the block is searched in
// memory.  (64-way searches in memory, two or three dependent loads and two
// more for the ends, took 133 us a call at k = 1000.)
constexpr int32_t kCookieFar = 1024;

__device__ inline void cut_cookies(int32_t k, int32_t ne, const int64_t *bs, const int64_t *room, int32_t *es,
                                   int32_t *ee)
{
    constexpr int32_t B = 2 * kWave;
    const int lane = lane_id();
    auto load = [&](int32_t base, int64_t &x0, int64_t &x1) {
        x0 = base + lane <= ne ? bs[base + lane] : INT64_MAX;
        x1 = base + kWave + lane <= ne ? bs[base + kWave + lane] : INT64_MAX;
    };
    int32_t base = 0, start = 0;
    int64_t c0, c1, n0, n1, prev = 0, bstart = 0;   // this block, the next, the value before this block
    load(0, c0, c1);
    load(B, n0, n1);
    for (int32_t p0 = 0; p0 < k; p0 += kWave) {
        const int32_t p = p0 + lane;
        const int64_t mine = p < k ? room[p] : 0;
        uint64_t todo = start < ne ? __ballot(mine > 0) : 0;   // the other parts' slices are empty
        int32_t s = start, e = start;                          // this lane's slice
        while (todo) {
            const int l = __ffsll((long long)todo) - 1;
            todo &= todo - 1;
            const int64_t cap = wave_read(mine, l), find = bstart + cap;
            const int32_t limit = (int32_t)min((int64_t)ne, (int64_t)start + cap);
            int32_t hi;
            int64_t bh, bl;
            for (;;) {
                const uint64_t m0 = __ballot(base + lane >= limit || c0 >= find);
                const uint64_t m1 = __ballot(base + kWave + lane >= limit || c1 >= find);
                if (m0 | m1) {
                    const int f = m0 ? __ffsll((long long)m0) - 1 : kWave + __ffsll((long long)m1) - 1;
                    hi = base + f;
                    bh = m0 ? wave_read(c0, f) : wave_read(c1, f - kWave);
                    bl = f == 0 ? prev : (f <= kWave ? wave_read(c0, f - 1) : wave_read(c1, f - 1 - kWave));
                    break;
                }
                if (limit - (base + B) > kCookieFar) {
                    int32_t L = base + B, H = limit;   // hi in [L, H]; H stands for "none below H"
                    while (L < H) {
                        const int32_t span = H - L, step = (span + kWave - 1) / kWave;
                        const int32_t pos = L + lane * step;
                        const uint64_t m = __ballot(pos < H && bs[pos] >= find);
                        const int f = m ? __ffsll((long long)m) - 1 : (span + step - 1) / step;   // samples below find
                        if (m) H = L + f * step;
                        if (f == 0) break;   // the first sample reaches it
                        L += (f - 1) * step + 1;
                    }
                    hi = H;
                    bh = bs[hi];
                    bl = bs[hi - 1];
                    base = hi / B * B;
                    prev = bs[base > 0 ? base - 1 : 0];
                    load(base, c0, c1);
                    load(base + B, n0, n1);
                    break;
                }
                prev = wave_read(c1, kWave - 1);
                base += B;
                c0 = n0;
                c1 = n1;
                load(base + B, n0, n1);
            }
            int64_t dh = bh - find, dl = bl - find;
            dh = dh < 0 ? -dh : dh;
            dl = dl < 0 ? -dl : dl;
            const bool up = dh < dl;
            if (lane == l) s = start;
            start = up ? hi : hi - 1;
            bstart = up ? bh : bl;
            if (lane >= l) e = start;
            if (lane > l) s = start;
            if (start >= ne) break;   // the list is used up: the later slices are empty
        }
        if (p < k) {
            es[p] = s;
            ee[p] = e;
        }
    }
}

// select_dest_parts_rs (:2747-2766): entry i of the evicted list, vertex v,
// goes to the part whose slice holds i, or stays.
__device__ inline void assign_evicted(const RbView &A, int32_t i, int32_t v, const int32_t *es, const int32_t *ee)
{
    int32_t lo = 0, hi = A.k - 1;
    while (lo < hi) {
        const int32_t mid = (lo + hi + 1) >> 1;
        if (es[mid] <= i) lo = mid; else hi = mid - 1;
    }
    const int32_t w = A.where[v], d = i < ee[lo] ? lo : w;
    A.dest[v] = d;
    store_pair(A.pd16, A.pd32, v, w, d);
}

// LDS of rb_block.
template <int R>
struct RbLds {
    uint32_t sk[R * kRbBS];          // keys; later the evicted ids and the slices
    uint16_t sv[R * kRbBS];          // ids
    int32_t wc[kRbNW][256];
    int64_t wsum[kRbNW];
    int32_t wcnt[kRbNW], dsum[4];
    static_assert(R * kRbBS <= 65536, "16-bit ids");
};

// The whole step of a level of at most 1024 R vertices in one block.  The
// digit passes rank a wave's items with ballots and per-wave counts (no
// block barrier inside a pass but the three around the counts); the sorted
// keys and ids sit in LDS, then in registers, R per thread.
// part: k words of LDS (prefix weight at the part's first candidate, later its
// room).  k <= 256 R.  Every thread of the block calls it; the caller's barrier
// follows.
template <int R>
__device__ inline void rb_block(const RbView &A, int bits, int64_t *__restrict__ bs, RbLds<R> &L, int64_t *part)
{
    constexpr int N = R * kRbBS;
    const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
    const uint32_t nokey = (uint32_t)A.k * kMaxBuckets;
    const bool rs = A.ctl->mode == kModeRS;
    uint32_t key[R];
    int32_t id[R];
    int32_t nc = A.n;
    for (int shift = 0; shift < bits; shift += 8) {
        const int rows = (nc + kRbBS - 1) / kRbBS;
        uint32_t live = 0, d[R];
        int32_t rk[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r >= rows) break;
            const int32_t i = (w * rows + r) * kWave + lane;
            key[r] = nokey;
            id[r] = 0;
            if (i < nc) {
                key[r] = shift == 0 ? A.key[i] : L.sk[i];
                id[r] = shift == 0 ? i : (int32_t)L.sv[i];
            }
        }
        for (int i = lane; i < 256; i += kWave) L.wc[w][i] = 0;
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r >= rows) break;
            live |= (key[r] < nokey ? 1u : 0u) << r;
            d[r] = (key[r] >> shift) & 255u;
        }
        row_ranks<R>(d, live, rows, L.wc[w], rk);
        __syncthreads();
        nc = digit_bases(L.wc, L.dsum);
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r >= rows) break;
            if ((live >> r) & 1u) {
                const int32_t at = L.wc[w][d[r]] + rk[r];
                L.sk[at] = key[r];
                L.sv[at] = (uint16_t)id[r];
            }
        }
        __syncthreads();
    }
    // the sorted candidates, their weights and prefix weights
    const int rows = (nc + kRbBS - 1) / kRbBS;
    int32_t wt[R];
    int64_t pre[R], run = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        const int32_t i = (w * rows + r) * kWave + lane;
        key[r] = i < nc ? L.sk[i] : nokey;
        id[r] = i < nc ? (int32_t)L.sv[i] : 0;
        wt[r] = i < nc ? A.vwgt[id[r]] : 0;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        pre[r] = wave_inclusive_scan((int64_t)wt[r]) + run;
        run = wave_read(pre[r], kWave - 1);
    }
    if (lane == 0) L.wsum[w] = run;
    __syncthreads();
    int64_t off = 0;
    for (int x = 0; x < w; x++) off += L.wsum[x];
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        const int32_t i = (w * rows + r) * kWave + lane;
        pre[r] += off - wt[r];   // of the candidates before this one
        if (i < nc) {
            const uint32_t p = key[r] / kMaxBuckets;
            if (i == 0 || L.sk[i - 1] / kMaxBuckets != p) part[p] = pre[r];
        }
    }
    __syncthreads();
    // Evict a candidate iff those ahead of it in its part weigh less than the
    // part's excess (filter_scores_below_cutoff :3344-3366 for RW,
    // find_score_cutoffs/filter_below_cutoffs :2641-2691 for RS).
    uint32_t ev = 0;
    const int64_t maxwgt = A.ctl->maxwgt;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        const int32_t i = (w * rows + r) * kWave + lane;
        if (i >= nc) continue;
        const uint32_t p = key[r] / kMaxBuckets;
        if (pre[r] - part[p] < A.pwgts[p] - maxwgt) {
            ev |= 1u << r;
        } else {   // (a candidate's key holds its own part)
            const int32_t v = id[r], x = (int32_t)p;
            A.dest[v] = x;
            store_pair(A.pd16, A.pd32, v, x, x);
        }
    }
    if (!rs) return;
    // the evicted list: ids in LDS (over the keys), prefix weights in memory
    uint16_t *se = (uint16_t *)L.sk;
    int32_t *es = (int32_t *)(L.sk + N / 2), *ee = es + N / 4;   // k <= N / 4 (checked by the host)
    int32_t cnt = 0;
    run = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        const bool on = (ev >> r) & 1u;
        const uint64_t m = __ballot(on);
        key[r] = (uint32_t)(cnt + __popcll(m & lanemask_lt()));   // rank in the wave
        cnt += __popcll(m);
        pre[r] = wave_inclusive_scan((int64_t)(on ? wt[r] : 0)) + run;
        run = wave_read(pre[r], kWave - 1);
    }
    __syncthreads();   // the sums, part and the keys have been read
    if (lane == 0) {
        L.wsum[w] = run;
        L.wcnt[w] = cnt;
    }
    for (int32_t p = tid; p < A.k; p += kRbBS) part[p] = maxwgt > A.pwgts[p] ? maxwgt - A.pwgts[p] : 0;
    __syncthreads();
    off = 0;
    int32_t at = 0, ne = 0;
    for (int x = 0; x < kRbNW; x++) {
        off += x < w ? L.wsum[x] : 0;
        at += x < w ? L.wcnt[x] : 0;
        ne += L.wcnt[x];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= rows) break;
        if ((ev >> r) & 1u) {
            const int32_t j = at + (int32_t)key[r];
            se[j] = (uint16_t)id[r];
            bs[j + 1] = off + pre[r];
        }
    }
    if (tid == 0) bs[0] = 0;
    __syncthreads();
    if (w == 0) cut_cookies(A.k, ne, bs, part, es, ee);
    __syncthreads();
    for (int32_t i = tid; i < ne; i += kRbBS) assign_evicted(A, i, (int32_t)se[i], es, ee);
}

}  // namespace hgp
