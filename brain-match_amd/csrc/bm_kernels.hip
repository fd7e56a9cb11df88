/*
 * gfx950 support kernels around the delta kernels (bm_delta.hip):
 * candidate generation (uniform streams and the reference's changed-first
 * enumerations), candidate validation, reductions over deltas (stats, rank
 * picks), deterministic disjoint acceptance, and single-move application.
 */
#include "bm_device.h"
#include "bm_devutil.h"
#include "bm_rng.h"
#include "bm_rowtab.h"

#include <hipcub/hipcub.hpp>

using namespace bmd;

namespace {

/* ------------------------------------------------------------------ */
/* Candidate generation and validation                                 */
/* ------------------------------------------------------------------ */

__global__ void k_gen_pairs(int32_t n, uint64_t seed, int64_t k, int2* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride) {
        int32_t u, v;
        bm_uniform_pair(seed, (uint64_t)c, n, &u, &v);
        cand[c] = make_int2(u, v);
    }
}

__global__ void k_gen_triples(int32_t n, uint64_t seed, int64_t k, int4* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride) {
        int32_t a, b, d;
        bm_uniform_triple(seed, (uint64_t)c, n, &a, &b, &d);
        cand[c] = make_int4(a, b, d, 0);
    }
}

/* Lexicographic pair t of C(c,2) -> (i, j), i < j < c. */
__device__ __forceinline__ void pair_of(int64_t t, int64_t c, int64_t* i, int64_t* j) {
    /* row i starts at s(i) = i*(2c-i-1)/2 */
    const double b = 2.0 * (double)c - 1.0;
    int64_t r = (int64_t)((b - sqrt(b * b - 8.0 * (double)t)) * 0.5);
    if (r < 0) r = 0;
    if (r > c - 2) r = c - 2;
    while (r > 0 && r * (2 * c - r - 1) / 2 > t) r--;
    while (r + 1 <= c - 2 && (r + 1) * (2 * c - r - 2) / 2 <= t) r++;
    *i = r;
    *j = r + 1 + (t - r * (2 * c - r - 1) / 2);
}

__global__ void k_gen_changed_pairs(int32_t n, int32_t c, const int32_t* __restrict__ reorder, int64_t P,
                                    int2* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t cc = (int64_t)c * (c - 1) / 2;
    const int64_t nu = (int64_t)n - c;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < P; idx += stride) {
        int64_t i, j;
        if (idx < cc) {
            pair_of(idx, c, &i, &j);
            cand[idx] = make_int2(reorder[i], reorder[j]);
        } else {
            const int64_t t = idx - cc;
            i = t / nu;
            j = t - i * nu;
            cand[idx] = make_int2(reorder[i], reorder[c + j]);
        }
    }
}

/* The 3-section enumeration of calculateThreeNodeSwapKernel
 * (src/graph-re-alignment-gpu-3-swap.cu:67-150), with the same order. */
__global__ void k_gen_changed_triples(int32_t n, int32_t c, const int32_t* __restrict__ reorder, int64_t T,
                                      int4* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t s1 = (int64_t)c * (c - 1) * (c - 2) / 6;
    const int64_t cc = (int64_t)c * (c - 1) / 2;
    const int64_t s2 = s1 + cc * ((int64_t)n - c);
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < T; idx += stride) {
        int32_t a, b, d;
        if (idx < s1) {
            /* lexicographic triple of the c changed positions */
            int64_t t = idx, i = 0, rem = (int64_t)(c - 1) * (c - 2) / 2;
            while (t >= rem) { t -= rem; i++; rem = (int64_t)(c - 1 - i) * (c - 2 - i) / 2; }
            int64_t j = i + 1, r2 = c - i - 2;
            while (t >= r2) { t -= r2; j++; r2--; }
            a = reorder[i];
            b = reorder[j];
            d = reorder[j + 1 + t];
        } else if (idx < s2) {
            const int64_t t = idx - s1;
            const int64_t m3 = t / cc;
            int64_t i, j;
            pair_of(t - m3 * cc, c, &i, &j);
            a = reorder[i];
            b = reorder[j];
            d = reorder[c + m3];
        } else {
            const int64_t t = idx - s2;
            const int64_t rest = (int64_t)n - c - 1;
            const int64_t i = t / rest, j = t - i * rest;
            a = reorder[i];
            b = reorder[c + j];
            d = reorder[c + j + 1];
        }
        cand[idx] = make_int4(a, b, d, 0);
    }
}

__global__ void k_check_pairs(int32_t n, const int2* __restrict__ cand, int64_t k, int32_t* bad) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int badl = 0;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride) {
        const int2 p = cand[c];
        badl |= (p.x < 1) | (p.x > n) | (p.y < 1) | (p.y > n);
    }
    if (badl) atomicOr(bad, 1);
}

__global__ void k_check_triples(int32_t n, const int4* __restrict__ cand, int64_t k, int32_t* bad) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int badl = 0;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride) {
        const int4 p = cand[c];
        badl |= (p.x < 1) | (p.x > n) | (p.y < 1) | (p.y > n) | (p.z < 1) | (p.z > n);
        badl |= (p.x == p.y) | (p.x == p.z) | (p.y == p.z);
    }
    if (badl) atomicOr(bad, 1);
}

/* ------------------------------------------------------------------ */
/* Reductions                                                          */
/* ------------------------------------------------------------------ */

/* A batch's deltas are read once by at most kRedBlocks blocks, one chunk of a
 * power of two each, so that the one block which combines the partial results
 * has at most eight per thread; up to 2^25 deltas the chunk is 4,096.  What
 * bounds both passes is the read: 16-byte loads, eight in flight per thread,
 * and shuffles instead of an LDS tree (2^28 deltas: stats 465 + 165 us ->
 * 378 + 12 us; the pick's count 405 us -> 342 us). */
constexpr int kRedThreads = 256;
constexpr int kRedWaves = kRedThreads / BM_WAVE;
constexpr int64_t kRedChunk = 4096;    /* smallest chunk */
constexpr int64_t kRedBlocks = 8192;
constexpr int kRedLoads = 8;
constexpr int kFinThreads = 1024;
constexpr int kFinWaves = kFinThreads / BM_WAVE;

int64_t red_chunk(int64_t k) {
    int64_t chunk = kRedChunk;
    while (chunk * kRedBlocks < k) chunk *= 2;
    return chunk;
}

struct Stats {
    int64_t sum, max, arg, pos, zero;   /* arg: first index of max, -1 none */
};

__device__ __forceinline__ void stats_join(Stats& a, const Stats& b) {
    a.sum += b.sum;
    a.pos += b.pos;
    a.zero += b.zero;
    if (b.arg >= 0 && (a.arg < 0 || b.max > a.max || (b.max == a.max && b.arg < a.arg))) {
        a.max = b.max;
        a.arg = b.arg;
    }
}

/* All threads' results joined in thread 0; s: one entry per wave. */
template <int WAVES>
__device__ __forceinline__ Stats stats_block(Stats a, Stats* s) {
#pragma unroll
    for (int o = BM_WAVE / 2; o > 0; o >>= 1) {
        const Stats b = {__shfl_down(a.sum, o), __shfl_down(a.max, o), __shfl_down(a.arg, o), __shfl_down(a.pos, o),
                         __shfl_down(a.zero, o)};
        stats_join(a, b);   /* lanes past the wave's end repeat their own: only lane 0 counts */
    }
    if ((threadIdx.x & (BM_WAVE - 1)) == 0) s[threadIdx.x / BM_WAVE] = a;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < WAVES; w++) stats_join(a, s[w]);
    return a;
}

__device__ __forceinline__ void stats_put(const Stats& a, int64_t k, int64_t* out) {
    out[0] = k; out[1] = a.sum; out[2] = a.max; out[3] = a.arg; out[4] = a.pos; out[5] = a.zero;
}

/* Partial results of chunk b at part[field * blocks + b]; a single chunk's
 * are the answer. */
__global__ void __launch_bounds__(kRedThreads) k_stats_part(const int64_t* __restrict__ d, int64_t k, int64_t chunk,
                                                            int64_t* __restrict__ part, int64_t* __restrict__ out) {
    __shared__ Stats s[kRedWaves];
    const int64_t base = (int64_t)blockIdx.x * chunk;
    const int64_t end = k - base < chunk ? k : base + chunk;
    Stats a = {0, INT64_MIN, -1, 0, 0};
    int32_t pos = 0, zero = 0;
    auto take = [&](int64_t x, int64_t i) {
        a.sum += x;
        pos += x > 0;
        zero += x == 0;
        if (x > a.max) { a.max = x; a.arg = i; }
    };
    int64_t i = base;
    constexpr int64_t kStep = 2 * kRedThreads * kRedLoads;
    for (; i + kStep <= end; i += kStep) {
        longlong2 x[kRedLoads];
#pragma unroll
        for (int j = 0; j < kRedLoads; j++)
            x[j] = reinterpret_cast<const longlong2*>(d + i)[j * kRedThreads + threadIdx.x];
#pragma unroll
        for (int j = 0; j < kRedLoads; j++) {
            const int64_t at = i + 2 * (j * kRedThreads + threadIdx.x);
            take(x[j].x, at);
            take(x[j].y, at + 1);
        }
    }
    for (i += threadIdx.x; i < end; i += kRedThreads) take(d[i], i);
    a.pos = pos;
    a.zero = zero;
    a = stats_block<kRedWaves>(a, s);
    if (threadIdx.x) return;
    const int64_t nb = gridDim.x;
    if (nb == 1) {
        stats_put(a, k, out);
        return;
    }
    int64_t* o = part + blockIdx.x;
    o[0] = a.sum; o[nb] = a.max; o[2 * nb] = a.arg; o[3 * nb] = a.pos; o[4 * nb] = a.zero;
}

__global__ void __launch_bounds__(kFinThreads) k_stats_final(const int64_t* __restrict__ part, int64_t nb, int64_t k,
                                                             int64_t* __restrict__ out) {
    __shared__ Stats s[kFinWaves];
    Stats a = {0, INT64_MIN, -1, 0, 0};
#pragma unroll 4
    for (int64_t b = threadIdx.x; b < nb; b += kFinThreads) {
        const int64_t* p = part + b;
        stats_join(a, {p[0], p[nb], p[2 * nb], p[3 * nb], p[4 * nb]});
    }
    a = stats_block<kFinWaves>(a, s);
    if (threadIdx.x == 0) stats_put(a, k, out);
}

__device__ __forceinline__ bool picked(int64_t x, int32_t kind) { return kind ? x > 0 : x == 0; }

__global__ void __launch_bounds__(kRedThreads) k_pick_count(const int64_t* __restrict__ d, int64_t k, int32_t kind,
                                                            int64_t chunk, int64_t* __restrict__ cnt) {
    __shared__ int32_t s[kRedWaves];
    const int64_t base = (int64_t)blockIdx.x * chunk;
    const int64_t end = k - base < chunk ? k : base + chunk;
    int32_t c = 0;
    int64_t i = base;
    constexpr int64_t kStep = 2 * kRedThreads * kRedLoads;
    for (; i + kStep <= end; i += kStep) {
        longlong2 x[kRedLoads];
#pragma unroll
        for (int j = 0; j < kRedLoads; j++)
            x[j] = reinterpret_cast<const longlong2*>(d + i)[j * kRedThreads + threadIdx.x];
#pragma unroll
        for (int j = 0; j < kRedLoads; j++) c += picked(x[j].x, kind) + picked(x[j].y, kind);
    }
    for (i += threadIdx.x; i < end; i += kRedThreads) c += picked(d[i], kind);
#pragma unroll
    for (int o = BM_WAVE / 2; o > 0; o >>= 1) c += __shfl_down(c, o);
    if ((threadIdx.x & (BM_WAVE - 1)) == 0) s[threadIdx.x / BM_WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t all = 0;
        for (int w = 0; w < kRedWaves; w++) all += s[w];
        cnt[blockIdx.x] = all;
    }
}

/* Block scan of one value per thread: the sum before this thread's. */
__device__ __forceinline__ int64_t fin_scan(int64_t x, int64_t* s) {
    const int lane = threadIdx.x & (BM_WAVE - 1), wave = threadIdx.x / BM_WAVE;
    int64_t inc = x;
#pragma unroll
    for (int o = 1; o < BM_WAVE; o <<= 1) {
        const int64_t y = __shfl_up(inc, o);
        inc += lane >= o ? y : 0;
    }
    __syncthreads();   /* s may still be read */
    if (lane == BM_WAVE - 1) s[wave] = inc;
    __syncthreads();
    for (int w = 0; w < wave; w++) inc += s[w];
    return inc - x;
}

/* One block: locate the chunk holding the rank-th match (a single chunk has
 * no counts), then the wave's share of it, then the element. */
__global__ void __launch_bounds__(kFinThreads) k_pick_find(const int64_t* __restrict__ d, int64_t k, int32_t kind,
                                                           int64_t chunk, const int64_t* __restrict__ cnt, int64_t nb,
                                                           int64_t rank, int64_t* __restrict__ out) {
    __shared__ int64_t s[kFinWaves];
    __shared__ int64_t s_chunk, s_before, s_hit;
    const int t = threadIdx.x, lane = t & (BM_WAVE - 1), wave = t / BM_WAVE;
    if (t == 0) {
        s_hit = -1;
        s_chunk = nb == 1 ? 0 : -1;
        s_before = 0;
    }
    if (nb > 1) {
        const int64_t per = (nb + kFinThreads - 1) / kFinThreads;
        const int64_t b0 = (int64_t)t * per, b1 = b0 + per < nb ? b0 + per : nb;
        int64_t mine = 0;
        for (int64_t b = b0; b < b1; b++) mine += cnt[b];
        int64_t acc = fin_scan(mine, s);
        if (rank >= acc && rank < acc + mine)
            for (int64_t b = b0; b < b1; b++) {
                if (rank < acc + cnt[b]) { s_chunk = b; s_before = acc; break; }
                acc += cnt[b];
            }
    }
    __syncthreads();
    if (s_chunk >= 0) {   /* block-uniform */
        const int64_t share = chunk / kFinWaves;   /* a multiple of the wave */
        const int64_t base = s_chunk * chunk + wave * share;
        int64_t mine = 0;
#pragma unroll 4
        for (int64_t q = 0; q < share; q += BM_WAVE) {
            const int64_t i = base + q + lane;
            mine += __popcll(__ballot(i < k && picked(i < k ? d[i] : -1, kind)));
        }
        int64_t at = s_before + fin_scan(lane == 0 ? mine : 0, s);
        at = __shfl(at, 0);
        if (rank >= at && rank < at + mine)
            for (int64_t q = 0; q < share; q += BM_WAVE) {
                const int64_t i = base + q + lane;
                const bool hit = i < k && picked(i < k ? d[i] : -1, kind);
                const uint64_t m = __ballot(hit);
                if (hit && at + __popcll(m & ((1ull << lane) - 1)) == rank) s_hit = i;
                at += __popcll(m);
            }
        __syncthreads();
    }
    if (t == 0) out[0] = s_hit;
}

/* ------------------------------------------------------------------ */
/* Disjoint acceptance                                                 */
/* ------------------------------------------------------------------ */

struct PosDelta {
    const int64_t* d;
    __host__ __device__ bool operator()(const int64_t& i) const { return d[i] > 0; }
};

__global__ void k_gather_keys(const int64_t* __restrict__ d, const int64_t* __restrict__ idx, int64_t m,
                              int64_t* __restrict__ keys) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) keys[i] = d[idx[i]];
}

/* Order of a small batch's positive candidates: (delta desc, index asc), by
 * counting.  Every block holds all k deltas in LDS; 16 lanes per candidate
 * count the ones before it.  One launch and no host round trip, where
 * compaction, gather and radix sort take seven launches with the count read
 * back in between (4,096 candidates: 8 us against 30 us of kernels and the gaps). */
constexpr int kOrderMax = 8192, kOrderThreads = 256, kOrderLanes = 16, kOrderKeys = kOrderThreads / kOrderLanes;

__global__ void __launch_bounds__(kOrderThreads) k_accept_order(const int64_t* __restrict__ d, int32_t k,
                                                                int64_t* __restrict__ order,
                                                                int64_t* __restrict__ npos) {
    extern __shared__ longlong2 sd[];
    const int32_t words = (k + 2 * kOrderLanes - 1) / (2 * kOrderLanes) * kOrderLanes;
    int32_t pos = 0;
    const longlong2* dv = reinterpret_cast<const longlong2*>(d);
    for (int32_t b = 0; b < words; b += 8 * kOrderThreads) {   /* eight loads in flight */
        longlong2 x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int32_t i = b + j * kOrderThreads + threadIdx.x;
            x[j] = make_longlong2(0, 0);
            if (2 * i + 1 < k) x[j] = dv[i];
            else if (2 * i < k) x[j].x = d[2 * i];
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int32_t i = b + j * kOrderThreads + threadIdx.x;
            if (i < words) sd[i] = x[j];
            pos += (x[j].x > 0) + (x[j].y > 0);
        }
    }
    __shared__ int32_t s_pos;
    if (threadIdx.x == 0) s_pos = 0;
    __syncthreads();
    if (blockIdx.x == 0) {
        if (pos) atomicAdd(&s_pos, pos);
        __syncthreads();
        if (threadIdx.x == 0) *npos = s_pos;
    }
    const int32_t i = blockIdx.x * kOrderKeys + threadIdx.x / kOrderLanes, part = threadIdx.x % kOrderLanes;
    const int64_t me = i < k ? reinterpret_cast<const int64_t*>(sd)[i] : 0;
    if (!__ballot(me > 0)) return;
    int32_t rank = 0;
#pragma unroll 8
    for (int32_t q = part; q < words; q += kOrderLanes) {
        const longlong2 x = sd[q];   /* an equal delta counts when its index is smaller */
        rank += x.x > (2 * q < i ? me - 1 : me) ? 1 : 0;
        rank += x.y > (2 * q + 1 < i ? me - 1 : me) ? 1 : 0;
    }
#pragma unroll
    for (int o = 1; o < kOrderLanes; o <<= 1) rank += __shfl_xor(rank, o, BM_WAVE);
    if (part == 0 && me > 0) order[rank] = i;
}

constexpr int kAccThreads = 1024, kAccWaves = kAccThreads / BM_WAVE;
constexpr int kAccBatch = 16;   /* free candidates decided together */

/* Sequential greedy in priority order, one block.  lock[] is a bitmap of
 * vertices in the closed neighbourhood of accepted swaps (LDS, n+1 bits).
 * The candidates are taken 1,024 at a time, one per thread.  A round takes
 * the first 16 of them whose endpoints are unlocked; whether one's acceptance
 * would lock another follows from row-table lookups among their endpoints
 * (120 pairs x 8 lookups, one per thread), one thread decides the 16 in
 * order, and the waves lock the accepted swaps' neighbourhoods.  That is
 * the decision of the one-at-a-time loop: a later candidate of the 16 is
 * rejected exactly when an earlier accepted one locks an endpoint.  One
 * candidate per round (five barriers and a list walk each) took 150 us for
 * the 50 swaps of an early climb round at n = 18,524, this 55 us with one wave per list. */
template <bool PACKED>
__global__ void __launch_bounds__(kAccThreads) k_accept_greedy(BmDevGraph g, int32_t* __restrict__ pi,
                                                               int32_t* __restrict__ inv,
                                                               const int2* __restrict__ cand,
                                                               const int64_t* __restrict__ d,
                                                               const int64_t* __restrict__ order,
                                                               const int64_t* __restrict__ npos_at, int64_t max_accept,
                                                               int64_t* __restrict__ acc_idx,
                                                               int64_t* __restrict__ meta, int64_t* __restrict__ host,
                                                               int4* __restrict__ moves) {
    extern __shared__ uint32_t lock[];
    __shared__ int32_t s_cnt[kAccWaves];
    __shared__ int2 s_end[kAccBatch];        /* endpoints of the round's candidates */
    __shared__ int64_t s_ci[kAccBatch], s_d[kAccBatch];
    __shared__ uint32_t s_conf[kAccBatch];   /* earlier candidates of the round that would lock it */
    __shared__ uint32_t s_acc;               /* accepted candidates of the round */
    __shared__ int32_t s_last;               /* thread of the round's last candidate */
    __shared__ int64_t s_nacc, s_gain;
    const int t = threadIdx.x, lane = t & (BM_WAVE - 1), wave = t / BM_WAVE;
    const int64_t npos = *npos_at;
    const int words = (g.n + 32) / 32;
    for (int i = t; i < words; i += kAccThreads) lock[i] = 0;
    if (t == 0) { s_nacc = 0; s_gain = 0; }
    /* this thread's lookup in a round: candidates qi < qj, endpoints and direction */
    int qi = -1, qj = -1;
    if (t < kAccBatch * (kAccBatch - 1) / 2 * 8) {
        const int pr = t >> 3;
        qj = 1;
        while (qj * (qj + 1) / 2 <= pr) qj++;
        qi = pr - qj * (qj - 1) / 2;
    }
    __syncthreads();
    for (int64_t base = 0; base < npos; base += kAccThreads) {
        if (s_nacc >= max_accept) break;   /* or every later tile is loaded and scanned for nothing */
        const int64_t i = base + t;
        const bool valid = i < npos;
        int64_t ci = -1, di = 0;
        int32_t u = 0, v = 0;
        if (valid) {
            ci = order[i];
            const int2 p = cand[ci];
            di = d[ci];
            u = p.x;
            v = p.y;
        }
        int start = 0;
        for (;;) {
            if (s_nacc >= max_accept) break;
            const bool free_ = valid && t >= start && u != v && !((lock[u >> 5] >> (u & 31)) & 1u) &&
                               !((lock[v >> 5] >> (v & 31)) & 1u);
            const uint64_t m = __ballot(free_);
            if (lane == 0) s_cnt[wave] = __popcll(m);
            if (t < kAccBatch) s_conf[t] = 0;
            __syncthreads();
            int before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < kAccWaves; w++) {
                const int c = s_cnt[w];
                before += w < wave ? c : 0;
                total += c;
            }
            if (total == 0) break;
            const int q = before + __popcll(m & ((1ull << lane) - 1ull));
            if (free_ && q < kAccBatch) {
                s_end[q] = make_int2(u, v);
                s_ci[q] = ci;
                s_d[q] = di;
                if (q == kAccBatch - 1 || q == total - 1) s_last = t;
            }
            __syncthreads();
            const int cnt = total < kAccBatch ? total : kAccBatch;
            /* lane l of every wave: list l % 4 (u out, v out, u in, v in) of candidate l / 4 */
            int64_t l0 = 0, l1 = 0;
            int32_t end = 0;
            if ((lane >> 2) < cnt) {
                end = (lane & 1) ? s_end[lane >> 2].y : s_end[lane >> 2].x;
                const int64_t* ptr = (lane & 2) ? g.m_in_ptr : g.m_out_ptr;
                l0 = ptr[end];
                l1 = ptr[end + 1];
            }
            if (qj >= 0 && qj < cnt) {
                const int2 a = s_end[qi], b = s_end[qj];
                const int32_t x = (t & 1) ? a.y : a.x, y = (t & 2) ? b.y : b.x;
                const int32_t row = (t & 4) ? y : x, key = (t & 4) ? x : y;
                if (x == y || row_find<PACKED>(g.m_out_t.tab, g.m_out_t.desc[row], key) != BM_ABSENT)
                    atomicOr(&s_conf[qj], 1u << qi);
            }
            __syncthreads();
            if (t == 0) {
                uint32_t acc = 0;
                int64_t nacc = s_nacc, gain = s_gain;
                for (int z = 0; z < cnt && nacc < max_accept; z++)
                    if (!(s_conf[z] & acc)) {
                        acc |= 1u << z;
                        acc_idx[nacc++] = s_ci[z];
                        gain += s_d[z];
                    }
                s_acc = acc;
                s_nacc = nacc;
                s_gain = gain;
            }
            __syncthreads();
            /* lock the accepted swaps' neighbourhoods: their lists in units of
             * 256 entries, taken by the waves in turn, so that a hub's list
             * does not hang on one wave */
            const bool on = (s_acc >> (lane >> 2)) & 1u;
            if (on && lane % 4 < 2 && wave == 0) atomicOr(&lock[end >> 5], 1u << (end & 31));
            const int32_t units = on ? (int32_t)((l1 - l0 + 255) / 256) : 0;
            int32_t incl = units;
#pragma unroll
            for (int o = 1; o < BM_WAVE; o <<= 1) {
                const int32_t y = __shfl_up(incl, o, BM_WAVE);
                if (lane >= o) incl += y;
            }
            const int32_t all = __builtin_amdgcn_readlane(incl, BM_WAVE - 1);
            for (int32_t unit = wave; unit < all; unit += kAccWaves) {
                const int l = __popcll(__ballot(incl <= unit));
                const int64_t first = __shfl(l0, l, BM_WAVE), last = __shfl(l1, l, BM_WAVE);
                const int64_t o = first + (int64_t)(unit - __shfl(incl - units, l, BM_WAVE)) * 256 + lane;
                const int2* adj = (l & 2) ? g.m_in : g.m_out;
                int32_t y[4];
#pragma unroll
                for (int z = 0; z < 4; z++) y[z] = o + BM_WAVE * z < last ? adj[o + BM_WAVE * z].x : 0;
#pragma unroll
                for (int z = 0; z < 4; z++)
                    if (y[z]) atomicOr(&lock[y[z] >> 5], 1u << (y[z] & 31));
            }
            start = s_last + 1;
            __syncthreads();
        }
        __syncthreads();
    }
    __syncthreads();
    const int64_t nacc = s_nacc;
    for (int64_t a = t; a < nacc; a += kAccThreads) {
        const int2 p = cand[acc_idx[a]];
        const int32_t fu = pi[p.x], fv = pi[p.y];
        if (moves) {
            moves[2 * a] = make_int4(p.x, fu, fv, 0);
            moves[2 * a + 1] = make_int4(p.y, fv, fu, 0);
        }
        pi[p.x] = fv;
        pi[p.y] = fu;
        if (fv) inv[fv] = p.x;
        if (fu) inv[fu] = p.y;
    }
    if (t == 0) {
        meta[0] = nacc; meta[1] = s_gain; meta[2] = 2 * nacc;
        host[0] = nacc; host[1] = s_gain;
    }
}

__global__ void k_apply_swap(int32_t* pi, int32_t* inv, int32_t u, int32_t v) {
    const int32_t fu = pi[u], fv = pi[v];
    pi[u] = fv;
    pi[v] = fu;
    if (fv) inv[fv] = u;
    if (fu) inv[fu] = v;
}

/* apply_permutation (src/graph-re-alignment-gpu-3-swap.cu:925-956). */
__global__ void k_apply_perm3(int32_t* pi, int32_t* inv, int32_t a, int32_t b, int32_t c, int32_t p) {
    const int32_t f[3] = {pi[a], pi[b], pi[c]}, v[3] = {a, b, c};
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int32_t x = f[perm_of(p, i)];
        pi[v[i]] = x;
        if (x) inv[x] = v[i];
    }
}

/* ---- u-major uniform stream (bm_umajor_first / bm_umajor_partner) ---- */

__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t count, int32_t v) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = v;
}

/* counts[u] += #{c : first vertex of draw c is u}; a block-private histogram
 * in LDS (n+1 ints) when it fits, merged with one global atomic per bin. */
__global__ void __launch_bounds__(1024) k_umajor_hist(int32_t n, uint64_t seed, int64_t k, int32_t* __restrict__ counts,
                                                     int use_lds) {
    extern __shared__ int32_t h[];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    if (use_lds) {
        for (int32_t x = threadIdx.x; x <= n; x += blockDim.x) h[x] = 0;
        __syncthreads();
        for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride)
            atomicAdd(&h[bm_umajor_first(seed, (uint64_t)c, n)], 1);
        __syncthreads();
        for (int32_t x = threadIdx.x; x <= n; x += blockDim.x)
            if (h[x]) atomicAdd(&counts[x], h[x]);
    } else {
        for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride)
            atomicAdd(&counts[bm_umajor_first(seed, (uint64_t)c, n)], 1);
    }
}

/* off[0] = off[1] = 0, off[u + 1] = off[u] + counts[u] (u = 1..n): one block,
 * each thread a contiguous run, then a block scan of the run sums. */
__global__ void __launch_bounds__(1024) k_umajor_offsets(int32_t n, const int32_t* __restrict__ counts,
                                                        int64_t* __restrict__ off) {
    __shared__ int64_t part[1024];
    const int t = threadIdx.x;
    const int64_t per = ((int64_t)n + 1023) / 1024;
    const int64_t a = 1 + (int64_t)t * per, b = a + per < (int64_t)n + 1 ? a + per : (int64_t)n + 1;
    int64_t sum = 0;
    for (int64_t x = a; x < b; x++) sum += counts[x];
    part[t] = sum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int64_t y = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += y;
        __syncthreads();
    }
    int64_t run = t ? part[t - 1] : 0;
    if (t == 0) {
        off[0] = 0;
        off[1] = 0;
    }
    for (int64_t x = a; x < b; x++) {
        run += counts[x];
        off[x + 1] = run;
    }
}

__global__ void k_gen_umajor(int32_t n, uint64_t seed, const int64_t* __restrict__ off, int64_t k,
                             int2* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < k; i += stride) {
        const int32_t u = umajor_owner(off, n, i);
        cand[i] = make_int2(u, bm_umajor_partner(seed, (uint64_t)i, u, n));
    }
}

/* a-major triples: entry i of the stream (seed) is (a, b, c, 0), a the
 * owner of i in the offsets of the first-vertex draws. */
__global__ void k_gen_amajor(int32_t n, uint64_t seed, const int64_t* __restrict__ off, int64_t k,
                             int4* __restrict__ cand) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < k; i += stride) {
        const int32_t a = umajor_owner(off, n, i);
        int32_t b, c;
        bm_amajor_partners(seed, (uint64_t)i, a, n, &b, &c);
        cand[i] = make_int4(a, b, c, 0);
    }
}

/* A block per row at a time: every entry takes the first empty slot from its
 * home bucket on (compare-and-swap; keys are unique in a row).  Within a bucket
 * slots fill in order, which the lookups rely on. */
template <bool PACKED>
__global__ void __launch_bounds__(256) k_rowtab_fill(const int64_t* __restrict__ ptr, const int2* __restrict__ adj,
                                                     int32_t n, const uint64_t* __restrict__ desc,
                                                     uint4* __restrict__ tab) {
    for (int64_t row = blockIdx.x; row <= n; row += gridDim.x) {
        const int64_t b = ptr[row], e = ptr[row + 1];
        const uint64_t d = desc[row];
        const uint32_t lb = (uint32_t)(d & 63u);
        const uint32_t per = RowSlots<PACKED>::kPerBucket, smask = (per << lb) - 1u;
        for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) {
            const int2 x = adj[i];
            uint32_t s = row_home(x.x, lb) * per;
            if (PACKED) {
                uint32_t* T = reinterpret_cast<uint32_t*>(tab + (d >> 6));
                const uint32_t v = ((uint32_t)x.x << 15) | (uint32_t)x.y;
                while (atomicCAS(&T[s], 0u, v) != 0u) s = (s + 1u) & smask;
            } else {
                unsigned long long* T = reinterpret_cast<unsigned long long*>(tab + (d >> 6));
                const unsigned long long v = ((unsigned long long)(uint32_t)x.y << 32) | (uint32_t)x.x;
                while (atomicCAS(&T[s], 0ull, v) != 0ull) s = (s + 1u) & smask;
            }
        }
    }
}

int grid_for(int64_t work, int threads) {
    int64_t b = (work + threads - 1) / threads;
    if (b < 1) b = 1;
    if (b > 65536) b = 65536;
    return (int)b;
}

}  // namespace

/* ------------------------------------------------------------------ */
/* Launchers                                                           */
/* ------------------------------------------------------------------ */

static hipError_t set_lds(const void* fn, size_t bytes) {
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

hipError_t bm_launch_rowtab_fill(int packed, const int64_t* ptr, const int2* adj, int32_t n, const uint64_t* desc,
                                 uint4* tab, hipStream_t s) {
    auto k = packed ? k_rowtab_fill<true> : k_rowtab_fill<false>;
    /* a launch of 2^32 threads or more is cut short without an error */
    const int64_t rows = (int64_t)n + 1, blocks = rows < (1 << 20) ? rows : 1 << 20;
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), 0, s, ptr, adj, n, desc, tab);
    return hipGetLastError();
}

hipError_t bm_launch_gen_pairs(int32_t n, uint64_t seed, int64_t k, int2* cand, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_pairs, dim3(grid_for(k, 256)), dim3(256), 0, s, n, seed, k, cand);
    return hipGetLastError();
}

hipError_t bm_launch_gen_triples(int32_t n, uint64_t seed, int64_t k, int4* cand, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_triples, dim3(grid_for(k, 256)), dim3(256), 0, s, n, seed, k, cand);
    return hipGetLastError();
}

hipError_t bm_launch_gen_changed_pairs(int32_t n, int32_t c, const int32_t* reorder, int64_t P, int2* cand,
                                       hipStream_t s) {
    if (P <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_changed_pairs, dim3(grid_for(P, 256)), dim3(256), 0, s, n, c, reorder, P, cand);
    return hipGetLastError();
}

hipError_t bm_launch_gen_changed_triples(int32_t n, int32_t c, const int32_t* reorder, int64_t T, int4* cand,
                                         hipStream_t s) {
    if (T <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_changed_triples, dim3(grid_for(T, 256)), dim3(256), 0, s, n, c, reorder, T, cand);
    return hipGetLastError();
}

hipError_t bm_launch_check_pairs(int32_t n, const int2* cand, int64_t k, int32_t* bad, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_check_pairs, dim3(grid_for(k, 256)), dim3(256), 0, s, n, cand, k, bad);
    return hipGetLastError();
}

hipError_t bm_launch_check_triples(int32_t n, const int4* cand, int64_t k, int32_t* bad, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_check_triples, dim3(grid_for(k, 256)), dim3(256), 0, s, n, cand, k, bad);
    return hipGetLastError();
}

int64_t bm_stats_blocks(int64_t k) {
    const int64_t nb = (k + kRedChunk - 1) / kRedChunk;
    return nb < 1 ? 1 : nb < kRedBlocks ? nb : kRedBlocks;
}

hipError_t bm_launch_stats(const int64_t* d, int64_t k, int64_t* part, int64_t* out6, hipStream_t s) {
    if (k <= 0) return hipErrorInvalidValue;
    const int64_t chunk = red_chunk(k), nb = (k + chunk - 1) / chunk;
    hipLaunchKernelGGL(k_stats_part, dim3((unsigned)nb), dim3(kRedThreads), 0, s, d, k, chunk, part, out6);
    if (nb > 1) hipLaunchKernelGGL(k_stats_final, dim3(1), dim3(kFinThreads), 0, s, part, nb, k, out6);
    return hipGetLastError();
}

hipError_t bm_launch_pick(const int64_t* d, int64_t k, int32_t kind, int64_t rank, int64_t* cnt, int64_t* out,
                          hipStream_t s) {
    if (k <= 0) return hipErrorInvalidValue;
    const int64_t chunk = red_chunk(k), nb = (k + chunk - 1) / chunk;
    if (nb > 1) hipLaunchKernelGGL(k_pick_count, dim3((unsigned)nb), dim3(kRedThreads), 0, s, d, k, kind, chunk, cnt);
    hipLaunchKernelGGL(k_pick_find, dim3(1), dim3(kFinThreads), 0, s, d, k, kind, chunk, cnt, nb, rank, out);
    return hipGetLastError();
}

/* Scratch layout: [idx k][keys k][sorted keys k][sorted idx k][count 1][cub temp ...] */
static size_t cub_temp_bytes(int64_t k) {
    size_t a = 0, b = 0;
    hipcub::CountingInputIterator<int64_t> it(0);
    PosDelta pred{nullptr};
    (void)hipcub::DeviceSelect::If(nullptr, a, it, (int64_t*)nullptr, (int64_t*)nullptr, (int)k, pred);
    (void)hipcub::DeviceRadixSort::SortPairsDescending(nullptr, b, (const int64_t*)nullptr, (int64_t*)nullptr,
                                                 (const int64_t*)nullptr, (int64_t*)nullptr, (int)k);
    return a > b ? a : b;
}

size_t bm_accept_scratch_bytes(int64_t k) {
    if (k < 1) k = 1;
    return (size_t)k * 4 * sizeof(int64_t) + 256 + cub_temp_bytes(k) + 256;
}

hipError_t bm_launch_accept(const BmDevGraph& g, int32_t* pi_rw, int32_t* inv_rw, const int2* cand, const int64_t* d,
                            int64_t k, int64_t max_accept, void* scratch, size_t scratch_bytes, int64_t* out_acc_idx,
                            int64_t* out_meta, int64_t* host_meta, int4* out_moves, hipStream_t s) {
    char* p = (char*)scratch;
    int64_t* idx = (int64_t*)p;
    int64_t* keys = idx + k;
    int64_t* skeys = keys + k;
    int64_t* sidx = skeys + k;
    int64_t* cnt = sidx + k;
    hipError_t e;
    if (k <= kOrderMax) {
        const size_t lds = (size_t)((k + 2 * kOrderLanes - 1) / (2 * kOrderLanes) * kOrderLanes) * sizeof(longlong2);
        if (lds > 48 * 1024) {
            e = set_lds((const void*)k_accept_order, lds);
            if (e != hipSuccess) return e;
        }
        int64_t blocks = (k + kOrderKeys - 1) / kOrderKeys;
        if (blocks < 1) blocks = 1;
        hipLaunchKernelGGL(k_accept_order, dim3((unsigned)blocks), dim3(kOrderThreads), lds, s, d, (int32_t)k, sidx, cnt);
    } else {
        char* temp = (char*)(cnt) + 256;
        const size_t temp_bytes = scratch_bytes - ((size_t)(temp - p));
        hipcub::CountingInputIterator<int64_t> it(0);
        PosDelta pred{d};
        size_t tb = temp_bytes;
        e = hipcub::DeviceSelect::If(temp, tb, it, idx, cnt, (int)k, pred, s);
        if (e != hipSuccess) return e;
        int64_t npos = 0;
        e = hipMemcpyAsync(&npos, cnt, sizeof(int64_t), hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) return e;
        e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        if (npos > 0) {
            size_t need = 0;
            e = hipcub::DeviceRadixSort::SortPairsDescending(nullptr, need, (const int64_t*)nullptr, (int64_t*)nullptr,
                                                             (const int64_t*)nullptr, (int64_t*)nullptr, (int)npos, 0,
                                                             64, s);
            if (e != hipSuccess) return e;
            if (need > temp_bytes) return hipErrorInvalidValue;
            hipLaunchKernelGGL(k_gather_keys, dim3(grid_for(npos, 256)), dim3(256), 0, s, d, idx, npos, keys);
            tb = temp_bytes;
            e = hipcub::DeviceRadixSort::SortPairsDescending(temp, tb, keys, skeys, idx, sidx, (int)npos, 0, 64, s);
            if (e != hipSuccess) return e;
        }
    }
    const size_t lds = (size_t)((g.n + 32) / 32) * sizeof(uint32_t);
    auto greedy = g.packed ? k_accept_greedy<true> : k_accept_greedy<false>;
    if (lds > 48 * 1024) {
        e = set_lds((const void*)greedy, lds);
        if (e != hipSuccess) return e;
    }
    if (max_accept <= 0) max_accept = INT64_MAX;
    hipLaunchKernelGGL(greedy, dim3(1), dim3(kAccThreads), lds, s, g, pi_rw, inv_rw, cand, d, sidx, cnt, max_accept,
                       out_acc_idx, out_meta, host_meta, out_moves);
    return hipGetLastError();
}

hipError_t bm_launch_apply_swap(int32_t* pi, int32_t* inv, int32_t u, int32_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_apply_swap, dim3(1), dim3(1), 0, s, pi, inv, u, v);
    return hipGetLastError();
}

hipError_t bm_launch_apply_perm3(int32_t* pi, int32_t* inv, int32_t a, int32_t b, int32_t c, int32_t p, hipStream_t s) {
    hipLaunchKernelGGL(k_apply_perm3, dim3(1), dim3(1), 0, s, pi, inv, a, b, c, p);
    return hipGetLastError();
}

hipError_t bm_launch_umajor_offsets(int32_t n, uint64_t seed, int64_t k, int32_t* counts, int64_t* off,
                                    int32_t num_cus, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_for((int64_t)n + 1, 256)), dim3(256), 0, s, counts, (int64_t)n + 1, 0);
    const size_t lds = ((size_t)n + 1) * sizeof(int32_t);
    const int use_lds = lds <= 150 * 1024 ? 1 : 0;
    if (use_lds) {
        hipError_t e = hipFuncSetAttribute((const void*)k_umajor_hist, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds);
        if (e != hipSuccess) return e;
    }
    int64_t blocks = (k + 1023) / 1024;
    const int64_t cap = (int64_t)(num_cus > 0 ? num_cus : 256);
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    if (k > 0)
        hipLaunchKernelGGL(k_umajor_hist, dim3((unsigned)blocks), dim3(1024), use_lds ? lds : 0, s, n, seed, k, counts,
                           use_lds);
    hipLaunchKernelGGL(k_umajor_offsets, dim3(1), dim3(1024), 0, s, n, counts, off);
    return hipGetLastError();
}

hipError_t bm_launch_gen_amajor(int32_t n, uint64_t seed, const int64_t* off, int64_t k, int4* cand, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_amajor, dim3(grid_for(k, 256)), dim3(256), 0, s, n, seed, off, k, cand);
    return hipGetLastError();
}

hipError_t bm_launch_gen_umajor(int32_t n, uint64_t seed, const int64_t* off, int64_t k, int2* cand, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_umajor, dim3(grid_for(k, 256)), dim3(256), 0, s, n, seed, off, k, cand);
    return hipGetLastError();
}
