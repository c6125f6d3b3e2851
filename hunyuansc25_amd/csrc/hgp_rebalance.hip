// hgp_rebalance.hip -- the rebalancing step of a Jet iteration (RW and RS,
// hunyuangraph_GPU_krefine.h:2515-2766, 3243-3366): order the candidates by
// (part, gain bucket, vertex id), evict from each overweight part the prefix
// that covers its excess, and in RS deal the evicted list to the parts with
// room (the cookie cutter).
//
// The step runs once per iteration on every level, most of them small, so it
// is bound by the latency of its chain of launches and by the barriers inside
// them.  Levels of up to kRbBlockN vertices take one launch: a block sorts the
// candidates in LDS and goes on to the last assignment.  Larger levels sort
// with two or three digit passes over tiles; the first pass drops the vertices
// that are no candidates (half to nine tenths of them), so the later passes,
// the weight scan and the eviction walk the candidates alone.
#include "hgp_jet.hpp"
#include "hgp_group.hpp"
#include "hgp_prims.hpp"
#include "hgp_rebalance_block.hpp"

#include <algorithm>

namespace hgp {

namespace {

constexpr int32_t kRbBlockN = 16 * kRbBS;    // largest level that one block takes
constexpr int kRbR = 8, kRbTBS = 256;        // weight tiles: 8 rows of 64 per wave, 4 waves
constexpr int kRbTile = kRbR * kRbTBS;
constexpr int kRbSR = 4;                     // sort tiles: 4 rows of 64 per wave (16 rows left too few blocks)
constexpr int kRbFuseTiles = 64;             // up to this many sort tiles the scatter sums the counts itself

template <int R>
__global__ void __launch_bounds__(kRbBS) k_rb_block(RbView A, int bits, int64_t *__restrict__ bs)
{
    extern __shared__ int64_t part[];   // k
    __shared__ RbLds<R> L;
    rb_block<R>(A, bits, bs, L, part);
}

// ---------------------------------------------------------------- larger levels

// Items of a sort tile: kRbBS * R, wave w taking rows of 64 from w * R on.
// First pass: the vertices' keys, those without one left out; later passes:
// the *nc sorted keys.
template <int R>
__device__ inline uint32_t load_keys(const uint32_t *__restrict__ kin, int32_t cnt, uint32_t nokey, int64_t tile,
                                     uint32_t (&key)[R])
{
    const int w = threadIdx.x / kWave;
    uint32_t live = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int64_t i = tile * (kRbBS * R) + (w * R + r) * kWave + lane_id();
        key[r] = i < cnt ? kin[i] : nokey;
    }
#pragma unroll
    for (int r = 0; r < R; r++) live |= (key[r] < nokey ? 1u : 0u) << r;
    return live;
}

// Digit counts per tile, hist[tile * 256 + digit].
template <int R>
__global__ void __launch_bounds__(kRbBS) k_rb_hist(const uint32_t *__restrict__ kin, int32_t n,
                                                   const int64_t *__restrict__ nc, uint32_t nokey, int shift,
                                                   uint32_t *__restrict__ hist)
{
    __shared__ int32_t wc[kRbNW][256];
    const int tid = threadIdx.x, w = tid / kWave;
    const int32_t cnt = nc ? (int32_t)*nc : n;
    if ((int64_t)blockIdx.x * (kRbBS * R) >= cnt) {   // (the scatter sums every tile's counts)
        if (tid < 256) hist[(int64_t)blockIdx.x * 256 + tid] = 0;
        return;
    }
    for (int i = lane_id(); i < 256; i += kWave) wc[w][i] = 0;
    uint32_t key[R], d[R];
    const uint32_t live = load_keys<R>(kin, cnt, nokey, blockIdx.x, key);
#pragma unroll
    for (int r = 0; r < R; r++) d[r] = (key[r] >> shift) & 255u;
    wave_lds_sync();
    // one counter update per row and distinct digit (equal digits are common:
    // a few buckets hold most candidates)
#pragma unroll
    for (int r = 0; r < R; r++) {
        const bool on = (live >> r) & 1u;
        uint64_t m = __ballot(on);
        if (!m) continue;
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d[r] >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        if (on && (m & lanemask_lt()) == 0) atomicAdd(&wc[w][d[r]], (int32_t)__popcll(m));
    }
    __syncthreads();
    if (tid < 256) {
        int32_t s = 0;
#pragma unroll
        for (int x = 0; x < kRbNW; x++) s += wc[x][tid];
        hist[(int64_t)blockIdx.x * 256 + tid] = (uint32_t)s;
    }
}

// Past kRbFuseTiles tiles: column d of hist becomes its exclusive prefix, its
// total goes to hist[ntiles * 256 + d].
__global__ void __launch_bounds__(kRowBS) k_rb_columns(int32_t ntiles, uint32_t *__restrict__ hist)
{
    __shared__ uint32_t sh[kRowBS / kWave];
    const int d = blockIdx.x;
    uint32_t carry = 0;
    for (int32_t t0 = 0; t0 < ntiles; t0 += kRowBS) {
        const int32_t t = t0 + threadIdx.x;
        const uint32_t x = t < ntiles ? hist[(int64_t)t * 256 + d] : 0u;
        uint32_t tot;
        const uint32_t ex = block_exclusive_scan(x, sh, &tot);
        if (t < ntiles) hist[(int64_t)t * 256 + d] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) hist[(int64_t)ntiles * 256 + d] = carry;
}

// Stable scatter of a tile by one digit; vin null: the ids are the items'
// indices.  The first pass leaves the number of candidates in *total; the last
// one (wout given) brings the candidates' weights along: their gather runs
// while the items are ranked.
template <int R>
__global__ void __launch_bounds__(kRbBS) k_rb_scatter(const uint32_t *__restrict__ kin,
                                                      const uint32_t *__restrict__ vin, int32_t n,
                                                      const int64_t *__restrict__ nc, uint32_t nokey, int shift,
                                                      int32_t ntiles, const uint32_t *__restrict__ hist, int columns,
                                                      uint32_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                      int64_t *__restrict__ total, const wgt_t *__restrict__ vwgt,
                                                      int32_t *__restrict__ wout)
{
    __shared__ int32_t wc[kRbNW][256];
    __shared__ uint32_t before[kRbBS / 256][256], all[kRbBS / 256][256];
    __shared__ uint32_t dsum[4];
    const int tid = threadIdx.x, w = tid / kWave, dg = tid & 255, g = tid / 256;
    const int32_t cnt = nc ? (int32_t)*nc : n;
    if (blockIdx.x > 0 && (int64_t)blockIdx.x * (kRbBS * R) >= cnt) return;
    uint32_t key[R], d[R], val[R];
    const uint32_t live = load_keys<R>(kin, cnt, nokey, blockIdx.x, key);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int64_t i = (int64_t)blockIdx.x * (kRbBS * R) + (w * R + r) * kWave + lane_id();
        val[r] = vin ? (i < cnt ? vin[i] : 0u) : (uint32_t)i;
        d[r] = (key[r] >> shift) & 255u;
    }
    int32_t wt[R];
    if (wout) {
#pragma unroll
        for (int r = 0; r < R; r++) wt[r] = (live >> r) & 1u ? vwgt[val[r]] : 0;
    }
    // this tile's first slot of each digit: smaller digits of all tiles, then
    // the digit in the tiles before
    uint32_t bf = 0, tot = 0;
    if (columns) {
        if (g == 0) {
            bf = hist[(int64_t)blockIdx.x * 256 + dg];
            tot = hist[(int64_t)ntiles * 256 + dg];
        }
    } else {
#pragma unroll 8
        for (int32_t t = g; t < ntiles; t += kRbBS / 256) {
            const uint32_t x = hist[(int64_t)t * 256 + dg];
            tot += x;
            bf += t < (int32_t)blockIdx.x ? x : 0u;
        }
    }
    before[g][dg] = bf;
    all[g][dg] = tot;
    for (int i = lane_id(); i < 256; i += kWave) wc[w][i] = 0;
    wave_lds_sync();
    int32_t rk[R];
    row_ranks<R>(d, live, R, wc[w], rk);
    __syncthreads();
    uint32_t first = 0, mine = 0;
    if (tid < 256) {
#pragma unroll
        for (int x = 0; x < kRbBS / 256; x++) {
            first += before[x][tid];
            mine += all[x][tid];
        }
        const uint32_t incl = wave_inclusive_scan(mine);
        if (lane_id() == kWave - 1) dsum[w] = incl;
        first += incl - mine;
    }
    __syncthreads();
    if (tid < 256) {
        for (int x = 0; x < w; x++) first += dsum[x];
        int32_t run = (int32_t)first;
#pragma unroll
        for (int x = 0; x < kRbNW; x++) {
            const int32_t c = wc[x][tid];
            wc[x][tid] = run;
            run += c;
        }
    }
    if (total && blockIdx.x == 0 && tid == 0) *total = (int64_t)(dsum[0] + dsum[1] + dsum[2] + dsum[3]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
        if ((live >> r) & 1u) {
            const int32_t at = wc[w][d[r]] + rk[r];
            kout[at] = key[r];
            vout[at] = val[r];
            if (wout) wout[at] = wt[r];
        }
    }
}

// Weight of the sorted candidates per tile, and where each part's candidates
// begin: their tile and the weight in it before them.  (Sums per part by
// atomics took 6 us more: atomics on one cache line complete every 12 ns.)
// The loads go out before the number of candidates is known (the arrays hold n
// items) and are masked after.
__global__ void __launch_bounds__(kRbTBS) k_rb_sums(int32_t n, const int64_t *__restrict__ nc,
                                                    const uint32_t *__restrict__ key, const int32_t *__restrict__ wt,
                                                    int64_t *__restrict__ tsum, int32_t *__restrict__ ptile,
                                                    int64_t *__restrict__ phead)
{
    __shared__ int64_t sh[kRbTBS / kWave];
    const int w = threadIdx.x / kWave, lane = lane_id();
    const int64_t t0 = (int64_t)blockIdx.x * kRbTile, base = t0 + w * (kWave * kRbR) + lane;
    uint32_t p[kRbR], before[kRbR];   // parts of the item and of the one before it
    int32_t x[kRbR];
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        const int64_t i = base + r * kWave;
        x[r] = i < n ? wt[i] : 0;
        p[r] = i < n ? key[i] : 0u;
        before[r] = i < n && i > 0 ? key[i - 1] : ~0u;
    }
    const int64_t cnt = *nc;
    if (t0 >= cnt) return;
    int64_t pre[kRbR], run = 0;
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        x[r] = base + r * kWave < cnt ? x[r] : 0;
        pre[r] = wave_inclusive_scan((int64_t)x[r]) + run;
        run = wave_read(pre[r], kWave - 1);
    }
    if (lane == 0) sh[w] = run;
    __syncthreads();
    int64_t off = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kRbTBS / kWave; i++) {
        off += i < w ? sh[i] : 0;
        all += sh[i];
    }
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        if (base + r * kWave < cnt && before[r] / kMaxBuckets != p[r] / kMaxBuckets) {
            ptile[p[r] / kMaxBuckets] = (int32_t)blockIdx.x;
            phead[p[r] / kMaxBuckets] = off + pre[r] - x[r];
        }
    }
    if (threadIdx.x == 0) tsum[blockIdx.x] = all;
}

// Evict a candidate iff those ahead of it in its part weigh less than the
// part's excess.  RW and RS leave the others where they are; RS marks the
// evicted ones by their weight in wt (0 for the others) and counts them per
// tile.  Only the tile's first part can begin before the tile: the block adds
// the tiles from that part's first one on.
__global__ void __launch_bounds__(kRbTBS) k_rb_evict(RbView A, const int64_t *__restrict__ nc,
                                                     const uint32_t *__restrict__ key,
                                                     const uint32_t *__restrict__ id, int32_t *__restrict__ wt,
                                                     const int64_t *__restrict__ tsum,
                                                     const int32_t *__restrict__ ptile,
                                                     const int64_t *__restrict__ phead, int32_t *__restrict__ tevn,
                                                     int64_t *__restrict__ tevw)
{
    extern __shared__ int64_t part[];   // k: weight in the tile before the part's first candidate
    __shared__ int64_t sh[kRbTBS / kWave], shp[kRbTBS / kWave];
    __shared__ int32_t shn[kRbTBS / kWave];
    const int w = threadIdx.x / kWave, lane = lane_id();
    const int64_t t0 = (int64_t)blockIdx.x * kRbTile, base = t0 + w * (kWave * kRbR) + lane;
    uint32_t p[kRbR], v[kRbR], before[kRbR];
    int32_t x[kRbR];
#pragma unroll
    for (int r = 0; r < kRbR; r++) {   // before the number of candidates is known, masked after
        const int64_t i = base + r * kWave;
        x[r] = i < A.n ? wt[i] : 0;
        p[r] = i < A.n ? key[i] : 0u;
        v[r] = i < A.n ? id[i] : 0u;
        before[r] = i < A.n && i > t0 ? key[i - 1] : ~0u;
    }
    const bool rs = A.ctl->mode == kModeRS;
    const int64_t maxwgt = A.ctl->maxwgt, cnt = *nc;
    if (t0 >= cnt) return;
    const uint32_t p0 = key[t0] / kMaxBuckets;   // the tile's first part
    const int32_t pt = ptile[p0];
    int64_t ahead = 0;   // its candidates in the tiles before this one
#pragma unroll 4
    for (int32_t i = pt + (int32_t)threadIdx.x; i < (int32_t)blockIdx.x; i += kRbTBS) ahead += tsum[i];
    if (threadIdx.x == 0 && pt < (int32_t)blockIdx.x) ahead -= phead[p0];
    int64_t pre[kRbR], run = 0;
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        const bool in = base + r * kWave < cnt;
        x[r] = in ? x[r] : 0;
        p[r] = in ? p[r] / kMaxBuckets : p0;
        pre[r] = wave_inclusive_scan((int64_t)x[r]) + run;
        run = wave_read(pre[r], kWave - 1);
    }
    ahead = wave_sum(ahead);
    if (lane == 0) {
        sh[w] = run;
        shp[w] = ahead;
    }
    __syncthreads();
    int64_t off = 0;
    ahead = 0;
#pragma unroll
    for (int i = 0; i < kRbTBS / kWave; i++) {
        ahead += shp[i];
        off += i < w ? sh[i] : 0;
    }
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        pre[r] += off - x[r];   // of the tile's items before this one
        if (base + r * kWave < cnt && before[r] / kMaxBuckets != p[r]) part[p[r]] = p[r] == p0 ? -ahead : pre[r];
    }
    __syncthreads();
    int32_t en = 0;
    int64_t ew = 0;
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        const int64_t i = base + r * kWave;
        if (i >= cnt) continue;
        const bool evict = pre[r] - part[p[r]] < A.pwgts[p[r]] - maxwgt;
        if (!evict) {
            const int32_t y = (int32_t)p[r];   // a candidate's key holds its own part
            A.dest[v[r]] = y;
            store_pair(A.pd16, A.pd32, (int32_t)v[r], y, y);
            if (rs) wt[i] = 0;
        } else {
            en++;
            ew += x[r];
        }
    }
    if (!rs) return;
    en = wave_sum(en);
    ew = wave_sum(ew);
    if (lane == 0) {
        shn[w] = en;
        sh[w] = ew;   // (read before the last barrier)
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kRbTBS / kWave; i++) {
            en += shn[i];
            ew += sh[i];
        }
        tevn[blockIdx.x] = en;
        tevw[blockIdx.x] = ew;
    }
}

// The evicted list in sorted order with its prefix weights (bs[0] = 0) and its
// length (ne).
__global__ void __launch_bounds__(kRbTBS) k_rb_elist(int32_t n, const int64_t *__restrict__ nc,
                                                     const uint32_t *__restrict__ id, const int32_t *__restrict__ wt,
                                                     const int32_t *__restrict__ tevn,
                                                     const int64_t *__restrict__ tevw, int32_t *__restrict__ elist,
                                                     int64_t *__restrict__ bs, int64_t *__restrict__ ne)
{
    __shared__ int64_t sh[kRbTBS / kWave], shp[kRbTBS / kWave];
    __shared__ int32_t shn[kRbTBS / kWave], shm[kRbTBS / kWave];
    const int w = threadIdx.x / kWave, lane = lane_id();
    const int64_t t0 = (int64_t)blockIdx.x * kRbTile, base = t0 + w * (kWave * kRbR) + lane;
    int32_t x[kRbR], rk[kRbR], n0 = 0, nb = 0;
    uint32_t v[kRbR];
    int64_t pre[kRbR], run = 0, wb = 0;
#pragma unroll
    for (int r = 0; r < kRbR; r++) {   // before the number of candidates is known, masked after
        const int64_t i = base + r * kWave;
        x[r] = i < n ? wt[i] : 0;
        v[r] = i < n ? id[i] : 0u;
    }
    const int64_t cnt = *nc;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        bs[0] = 0;
        if (cnt == 0) *ne = 0;
    }
    if (t0 >= cnt) return;
#pragma unroll
    for (int r = 0; r < kRbR; r++) x[r] = base + r * kWave < cnt ? x[r] : 0;
#pragma unroll 8
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kRbTBS) {
        nb += tevn[i];
        wb += tevw[i];
    }
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        const uint64_t m = __ballot(x[r] > 0);
        rk[r] = n0 + __popcll(m & lanemask_lt());
        n0 += __popcll(m);
        pre[r] = wave_inclusive_scan((int64_t)x[r]) + run;
        run = wave_read(pre[r], kWave - 1);
    }
    nb = wave_sum(nb);
    wb = wave_sum(wb);
    if (lane == 0) {
        sh[w] = run;
        shp[w] = wb;
        shn[w] = n0;
        shm[w] = nb;
    }
    __syncthreads();
    int64_t off = 0;
    int32_t at = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kRbTBS / kWave; i++) {
        off += shp[i] + (i < w ? sh[i] : 0);
        at += shm[i] + (i < w ? shn[i] : 0);
        all += shm[i] + shn[i];
    }
#pragma unroll
    for (int r = 0; r < kRbR; r++) {
        if (x[r] > 0) {
            elist[at + rk[r]] = (int32_t)v[r];
            bs[at + rk[r] + 1] = off + pre[r];
        }
    }
    if (t0 + kRbTile >= cnt && threadIdx.x == 0) *ne = all;   // the last tile
}

__global__ void __launch_bounds__(kWave) k_rb_cookie(RbView A, const int64_t *__restrict__ ne,
                                                     const int64_t *__restrict__ bs, int32_t *__restrict__ es,
                                                     int32_t *__restrict__ ee)
{
    extern __shared__ int64_t room[];
    const int64_t maxwgt = A.ctl->maxwgt;
    for (int32_t p = lane_id(); p < A.k; p += kWave) room[p] = maxwgt > A.pwgts[p] ? maxwgt - A.pwgts[p] : 0;
    wave_lds_sync();
    cut_cookies(A.k, (int32_t)*ne, bs, room, es, ee);
}

__global__ void k_rb_assign(RbView A, const int64_t *__restrict__ ne, const int32_t *__restrict__ elist,
                            const int32_t *__restrict__ es, const int32_t *__restrict__ ee)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < *ne) assign_evicted(A, (int32_t)i, elist[i], es, ee);
}

}  // namespace

RbScratch rebalance_scratch(Ctx &c, int32_t n, int32_t k)
{
    RbScratch s{};
    const size_t N = (size_t)(n > 0 ? n : 1), K = (size_t)k;
    s.bs = c.arena.ralloc<int64_t>(N + 1);
    if (n <= kRbBlockN && k <= kRbBS) return s;   // one block keeps the rest in LDS
    const size_t tiles = (N + kRbTile - 1) / kRbTile, stiles = (N + kRbSR * kRbBS - 1) / (kRbSR * kRbBS);
    for (int b = 0; b < 2; b++) {
        s.key[b] = c.arena.ralloc<uint32_t>(N);
        s.id[b] = c.arena.ralloc<uint32_t>(N);
    }
    s.hist = c.arena.ralloc<uint32_t>((stiles + 1) * 256);
    s.ptile = c.arena.ralloc<int32_t>(K);
    s.phead = c.arena.ralloc<int64_t>(K);
    s.w = c.arena.ralloc<int32_t>(N);
    s.tsum = c.arena.ralloc<int64_t>(tiles);
    s.tevw = c.arena.ralloc<int64_t>(tiles);
    s.tevn = c.arena.ralloc<int32_t>(tiles);
    s.elist = c.arena.ralloc<int32_t>(N);
    s.es = c.arena.ralloc<int32_t>(K);
    s.ee = c.arena.ralloc<int32_t>(K);
    s.cnt = c.arena.ralloc<int64_t>(2);
    return s;
}

void rebalance(Ctx &c, const RbView &v, const RbScratch &s, int32_t mode)
{
    const int32_t n = v.n, k = v.k;
    const int bits = bits_for((uint64_t)k * kMaxBuckets - 1);   // of the largest candidate key
    const uint32_t nokey = (uint32_t)k * kMaxBuckets;
    if (n <= kRbBlockN && k <= kRbBS) {
        // rows a wave by the level's size (less LDS and fewer registers on the small ones)
        KScope ks(c, "k_rb_block", 24.0 * (double)n);
        const size_t lds = sizeof(int64_t) * (size_t)k;
        if (n <= 4 * kRbBS) k_rb_block<4><<<1, kRbBS, lds, c.stream>>>(v, bits, s.bs);
        else if (n <= 8 * kRbBS) k_rb_block<8><<<1, kRbBS, lds, c.stream>>>(v, bits, s.bs);
        else k_rb_block<16><<<1, kRbBS, lds, c.stream>>>(v, bits, s.bs);
        HGP_LAUNCH_CHECK();
        return;
    }
    const int32_t ntiles = (int32_t)(((int64_t)n + kRbBS * kRbSR - 1) / (kRbBS * kRbSR));
    const bool columns = ntiles > kRbFuseTiles;
    int cur = -1;   // buffer that holds the sorted candidates (-1: none yet)
    for (int shift = 0; shift < bits; shift += 8) {
        const bool first = cur < 0;
        const uint32_t *kin = first ? v.key : s.key[cur], *vin = first ? nullptr : s.id[cur];
        const int64_t *nc = first ? nullptr : s.cnt;
        const int out = first ? 0 : cur ^ 1;
        {
            KScope ks(c, "k_rb_hist", 4.0 * (double)n);
            k_rb_hist<kRbSR><<<ntiles, kRbBS, 0, c.stream>>>(kin, n, nc, nokey, shift, s.hist);
            HGP_LAUNCH_CHECK();
        }
        if (columns) {
            k_rb_columns<<<256, kRowBS, 0, c.stream>>>(ntiles, s.hist);
            HGP_LAUNCH_CHECK();
        }
        {
            KScope ks(c, "k_rb_scatter", 12.0 * (double)n);
            const bool last = shift + 8 >= bits;
            k_rb_scatter<kRbSR><<<ntiles, kRbBS, 0, c.stream>>>(kin, vin, n, nc, nokey, shift, ntiles, s.hist, columns,
                                                                s.key[out], s.id[out], first ? s.cnt : nullptr,
                                                                v.vwgt, last ? s.w : nullptr);
            HGP_LAUNCH_CHECK();
        }
        cur = out;
    }
    const unsigned tiles = (unsigned)(((int64_t)n + kRbTile - 1) / kRbTile);
    k_rb_sums<<<tiles, kRbTBS, 0, c.stream>>>(n, s.cnt, s.key[cur], s.w, s.tsum, s.ptile, s.phead);
    HGP_LAUNCH_CHECK();
    k_rb_evict<<<tiles, kRbTBS, sizeof(int64_t) * (size_t)k, c.stream>>>(v, s.cnt, s.key[cur], s.id[cur], s.w, s.tsum,
                                                                        s.ptile, s.phead, s.tevn, s.tevw);
    HGP_LAUNCH_CHECK();
    if (mode != kModeRS) return;
    k_rb_elist<<<tiles, kRbTBS, 0, c.stream>>>(n, s.cnt, s.id[cur], s.w, s.tevn, s.tevw, s.elist, s.bs, s.cnt + 1);
    HGP_LAUNCH_CHECK();
    {
        KScope ks(c, "k_rb_cookie", 0.0);
        k_rb_cookie<<<1, kWave, sizeof(int64_t) * (size_t)k, c.stream>>>(v, s.cnt + 1, s.bs, s.es, s.ee);
        HGP_LAUNCH_CHECK();
    }
    k_rb_assign<<<grid_for(n, kRowBS), kRowBS, 0, c.stream>>>(v, s.cnt + 1, s.elist, s.es, s.ee);
    HGP_LAUNCH_CHECK();
}

}  // namespace hgp
