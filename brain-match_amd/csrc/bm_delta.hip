/*
 * gfx950 delta kernels: exact swap deltas, exact 3-vertex permutation deltas,
 * the full score and the annealing chains.
 *
 * A move's delta is a sum of terms (male vertex x, female f): the edges of x's
 * out- or in-list that land on edges of f's row under the matching.  A wave
 * (or the four waves of a block, for batches too small to fill the device)
 * takes one candidate: lanes set up its lists in parallel, then the wave walks
 * all of them as one index space, the shorter side of every term, and looks
 * each entry up in the other side's row table (bm_rowtab.h).  Sums over all
 * male lists (score, current contributions, features) go by fixed chunks.
 *
 * The reference kernels scan a dense (n+1)^2 int16 matrix row per vertex,
 * O(n) per pair (src/graph-re-alignment-gpu-swap.cu:198-233,
 * src/graph-re-alignment-gpu-3-swap.cu:186-248); here the work is at most
 * O(min degree) per term and exact for any int32 weights.
 */
#include <type_traits>

#include "bm_detexp.h"
#include "bm_device.h"
#include "bm_devutil.h"
#include "bm_rng.h"
#include "bm_rowtab.h"

using namespace bmd;

namespace {

/* ---- list intersections -------------------------------------------- */

/* One term of a delta: the edges of one list of a male vertex x (out or in)
 * that land on edges of the matching row of a female f.  The wave walks the
 * shorter of the two (the male list, mapped by pi, or the female row, mapped
 * by the inverse matching) and looks each mapped id up in the other's row
 * table, so a hub placed on an ordinary female costs the female's degree. */
struct alignas(16) ScanList {
    const int2* rows;    /* entries walked */
    const uint4* tab;    /* buckets of the row probed */
    uint32_t meta;       /* log2 buckets | kSideF | kIn | kNew */
    int32_t start;       /* first position in the wave's index space */
    int32_t term;        /* 3-vertex moves: 3 i + j for vertex i on female j */
    int32_t pad;
};
constexpr uint32_t kSideF = 64u, kIn = 128u, kNew = 256u;

/* List of (male x, female f, direction) into t; returns its length.  The
 * female row is walked only where the matching has an inverse. */
__device__ __forceinline__ int32_t scan_list(const BmDevGraph& g, bool inverse, int32_t x, int32_t f, bool in,
                                             ScanList& t) {
    const int64_t* mp = in ? g.m_in_ptr : g.m_out_ptr;
    const int64_t* fp = in ? g.f_in_ptr : g.f_out_ptr;
    const int64_t m0 = mp[x], m1 = mp[x + 1], a0 = fp[f], a1 = fp[f + 1];
    const uint64_t md = (in ? g.m_in_t.desc : g.m_out_t.desc)[x];
    const uint64_t fd = (in ? g.f_in_t.desc : g.f_out_t.desc)[f];
    const int32_t dm = (int32_t)(m1 - m0), df = (int32_t)(a1 - a0);
    const bool side = inverse && df < dm;
    const uint64_t d = side ? md : fd;
    t.rows = side ? (in ? g.f_in : g.f_out) + a0 : (in ? g.m_in : g.m_out) + m0;
    t.tab = (side ? (in ? g.m_in_t.tab : g.m_out_t.tab) : (in ? g.f_in_t.tab : g.f_out_t.tab)) + (d >> 6);
    t.meta = (uint32_t)(d & 63u) | (side ? kSideF : 0u) | (in ? kIn : 0u);
    return side ? df : (df == 0 ? 0 : dm);
}

/* Sum of contributions new - old of the lists of a swap (u on f2, v on f1:
 * new; with NT = 4 also u on f1, v on f2: old), the lane's share of wave wv
 * of W.  An out-list prices an edge to u or v at that endpoint's image in
 * the matching it belongs to (which makes u <-> v edges and self-loops
 * exact); an in-list leaves edges from u or v out (counted by the out-list).
 * Positions in 32 bits: 8 lists of at most n entries each. */
template <bool PACKED, int NT, int U, int W>
__device__ __forceinline__ typename std::conditional<PACKED, int32_t, int64_t>::type
swap_lists(const BmDevGraph& g, const int32_t* pi, const int32_t* inv, int32_t u, int32_t v, int32_t f1, int32_t f2, ScanList* L, int lane,
           int wv) {
    typedef typename std::conditional<PACKED, int32_t, int64_t>::type Acc;
    constexpr int NL = 2 * NT;
    int32_t len = 0;
    ScanList t;
    t.term = t.pad = 0;
    if (lane < NL) {
        const int q = lane >> 1;
        const bool onu = (q & 1) == 0;
        len = scan_list(g, inv != nullptr, onu ? u : v, (q == 0 || q == 3) ? f2 : f1, lane & 1, t);
        if (q < 2) t.meta |= kNew;
    }
    int32_t incl = len;
#pragma unroll
    for (int o = 1; o < NL; o <<= 1) {
        const int32_t y = __shfl_up(incl, o, BM_WAVE);
        if (lane >= o) incl += y;
    }
    t.start = incl - len;
    wave_sync();
    if (lane < NL) L[lane] = t;
    wave_sync();
    int32_t st[NL];
#pragma unroll
    for (int q = 1; q < NL; q++) st[q] = __builtin_amdgcn_readlane(t.start, q);
    const int32_t total = __builtin_amdgcn_readlane(incl, NL - 1);
    Acc acc = 0;
    for (int32_t base = wv * BM_WAVE * U; base < total; base += W * BM_WAVE * U) {
        const uint4* T[U];
        uint32_t meta[U];
        int2 e[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int32_t i = base + BM_WAVE * j + lane;
            int q = 0;
#pragma unroll
            for (int z = 1; z < NL; z++) q += i >= st[z] ? 1 : 0;
            const ScanList l = L[q];
            T[j] = l.tab;
            meta[j] = l.meta;
            e[j] = i < total ? l.rows[i - l.start] : make_int2(0, 0);
        }
        int32_t key[U];
#pragma unroll
        for (int j = 0; j < U; j++) key[j] = ((meta[j] & kSideF) ? inv : pi)[e[j].x];
        uint32_t b[U];
        uint32_t pend = 0;
#pragma unroll
        for (int j = 0; j < U; j++) {
            const bool side = meta[j] & kSideF;
            const int32_t id = e[j].x;
            const bool ha = id == (side ? f1 : u), hb = id == (side ? f2 : v);
            if (ha || hb) {
                if (meta[j] & kIn) key[j] = 0;
                else if (meta[j] & kNew) key[j] = side ? (ha ? v : u) : (ha ? f2 : f1);
            }
            if (id == 0) key[j] = 0;
            b[j] = row_home(key[j], meta[j] & 63u);
            pend |= (key[j] != 0 ? 1u : 0u) << j;
        }
        while (pend) {
            uint4 x[U];
#pragma unroll
            for (int j = 0; j < U; j++)
                if ((pend >> j) & 1u) x[j] = T[j][b[j]];
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (!((pend >> j) & 1u)) continue;
                int32_t w;
                if (row_bucket<PACKED>(x[j], key[j], w)) {
                    const int32_t c = contrib(e[j].y, w);
                    acc += (meta[j] & kNew) ? (Acc)c : -(Acc)c;
                    pend &= ~(1u << j);
                } else {
                    b[j] = (b[j] + 1u) & ((1u << (meta[j] & 63u)) - 1u);
                }
            }
        }
    }
    return acc;
}

/* Exact swap deltas.  What bounds it is the lookups: each is a 16-byte gather
 * (and a 4-byte gather of the matching), about 2e11 a second, so the shorter
 * side of every term is walked and the current terms are shared where a batch
 * is large enough.  At n = 18,524 with 4M edges a pair takes 555 lookups with
 * diag (1,322 without) and no hub pair more than 21,000; scanning both
 * vertices' lists against LDS copies of the four female rows took 1,728
 * lookups and 860 inserts, and up to 74,000 for a hub pair, which set the time
 * of small batches (4,096 pairs: 1,263 us, now 111; 65,536: 1,457, now 476;
 * 2^20: 12 ms, now 4.5).
 * W = 1: one wave per candidate, any number of waves per
 * block; W = 4: the four waves of a block share a candidate (batches too
 * small to fill the device, where the longest list sets the time).  DIAG:
 * the current contributions of u and v come from diag (bm_launch_diag), so only the
 * lists of the new images are walked; their edges u <-> v, counted by both,
 * are looked up. */
template <int MODE, bool PACKED, int U, int W, bool DIAG>
__global__ void __launch_bounds__(W == 1 ? 512 : 64 * W) k_swap(BmDevGraph g, const int2* __restrict__ cand,
                                                                const int64_t* __restrict__ off, uint64_t seed,
                                                                int64_t k, int64_t* __restrict__ delta,
                                                                const int64_t* __restrict__ diag) {
    constexpr int NT = DIAG ? 2 : 4;
    __shared__ ScanList s_lists[8][2 * NT];
    __shared__ int64_t s_part[2][W];
    const int lane = threadIdx.x & (BM_WAVE - 1);
    const int wave = uni(threadIdx.x / BM_WAVE);
    const int wpb = W == 1 ? (int)(blockDim.x / BM_WAVE) : 1;
    const int64_t nw = (int64_t)gridDim.x * wpb;
    int par = 0;
    for (int64_t c = (int64_t)blockIdx.x * wpb + (W == 1 ? wave : 0); c < k; c += nw) {
        int32_t u, v;
        if (MODE == BM_CAND_LIST) {
            const int2 p = cand[c];
            u = p.x;
            v = p.y;
        } else if (MODE == BM_CAND_UMAJOR) {
            u = umajor_owner(off, g.n, c);
            v = bm_umajor_partner(seed, (uint64_t)c, u, g.n);
        } else {
            bm_uniform_pair(seed, (uint64_t)c, g.n, &u, &v);
        }
        u = uni(u);
        v = uni(v);
        if (u == v) {
            if (threadIdx.x % (BM_WAVE * W) == 0) delta[c] = 0;
            continue;
        }
        const int32_t f1 = uni(g.pi[u]), f2 = uni(g.pi[v]);
        int64_t acc = (int64_t)swap_lists<PACKED, NT, U, W>(g, g.pi, g.inv, u, v, f1, f2, s_lists[wave], lane, W == 1 ? 0 : wave);
        if (DIAG && (W == 1 || wave == 0)) {
            if (lane < 2) {   /* edge u -> v (lane 0), v -> u (lane 1) at its current images */
                const int32_t a = lane ? v : u, b = lane ? u : v, fa = lane ? f2 : f1, fb = lane ? f1 : f2;
                acc -= diag[a];
                const int32_t w = row_find<PACKED>(g.m_out_t.tab, g.m_out_t.desc[a], b);
                if (w != BM_ABSENT) acc += contrib(w, row_find<PACKED>(g.f_out_t.tab, g.f_out_t.desc[fa], fb));
            }
        }
        acc = wave_sum64(acc);
        if (W == 1) {
            if (lane == 0) delta[c] = acc;
        } else {
            /* two buffers: thread 0 has read one before the barrier after which it is written again */
            if (lane == 0) s_part[par][wave] = acc;
            __syncthreads();
            if (threadIdx.x == 0) {
                int64_t sum = 0;
#pragma unroll
                for (int q = 0; q < W; q++) sum += s_part[par][q];
                delta[c] = sum;
            }
            par ^= 1;
        }
    }
}

/* ------------------------------------------------------------------ */
/* 3-vertex permutation deltas                                         */
/* ------------------------------------------------------------------ */

/* The lane's share (wave wv of W) of the deltas d[p], p = 1..5, of the five
 * non-identity permutations of the images f of the distinct vertices vtx; the
 * caller sums them over the waves (d[0] = 0).  18 lists: vertex i on female j,
 * out and in, edges inside the triple left out.  A lane's entries come in
 * list order, so it keeps one running sum and files it under the term when
 * the term changes.  Edges inside the triple (self-loops included) are looked
 * up by nine lanes and priced per permutation. */
template <bool PACKED, int U, int W>
__device__ __forceinline__ void rot3_lists(const BmDevGraph& g, const int32_t* pi, const int32_t* inv,
                                           const int32_t* vtx, const int32_t* f, ScanList* L,
                                           int lane, int wv, int64_t* d) {
    typedef typename std::conditional<PACKED, int32_t, int64_t>::type Acc;
    constexpr int NL = 18;
    int32_t len = 0;
    ScanList t;
    t.term = t.pad = 0;
    if (lane < NL) {
        const int i = lane / 6, j = (lane >> 1) % 3;
        len = scan_list(g, inv != nullptr, sel3(i, vtx[0], vtx[1], vtx[2]), sel3(j, f[0], f[1], f[2]), lane & 1, t);
        t.term = 3 * i + j;
    }
    int32_t incl = len;
#pragma unroll
    for (int o = 1; o < NL; o <<= 1) {
        const int32_t y = __shfl_up(incl, o, BM_WAVE);
        if (lane >= o) incl += y;
    }
    t.start = incl - len;
    wave_sync();
    if (lane < NL) L[lane] = t;
    wave_sync();
    const int32_t total = __builtin_amdgcn_readlane(incl, NL - 1);
    Acc s[9];
#pragma unroll
    for (int q = 0; q < 9; q++) s[q] = 0;
    int32_t cur = 0;
    Acc run = 0;
    int q0 = 0;   /* list of this lane's last entry: entries only move forward */
    for (int32_t base = wv * BM_WAVE * U; base < total; base += W * BM_WAVE * U) {
        const uint4* T[U];
        uint32_t meta[U];
        int32_t term[U];
        int2 e[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int32_t i = base + BM_WAVE * j + lane;
            while (q0 + 1 < NL && i >= L[q0 + 1].start) q0++;
            const ScanList l = L[q0];
            T[j] = l.tab;
            meta[j] = l.meta;
            term[j] = l.term;
            e[j] = i < total ? l.rows[i - l.start] : make_int2(0, 0);
        }
        int32_t key[U];
#pragma unroll
        for (int j = 0; j < U; j++) key[j] = ((meta[j] & kSideF) ? inv : pi)[e[j].x];
        uint32_t b[U];
        uint32_t pend = 0;
#pragma unroll
        for (int j = 0; j < U; j++) {
            const bool side = meta[j] & kSideF;
            const int32_t id = e[j].x;
            if (id == 0 || id == (side ? f[0] : vtx[0]) || id == (side ? f[1] : vtx[1]) || id == (side ? f[2] : vtx[2]))
                key[j] = 0;   /* no entry, or an edge inside the triple */
            b[j] = row_home(key[j], meta[j] & 63u);
            pend |= (key[j] != 0 ? 1u : 0u) << j;
        }
        int32_t c[U];
#pragma unroll
        for (int j = 0; j < U; j++) c[j] = 0;
        while (pend) {
            uint4 x[U];
#pragma unroll
            for (int j = 0; j < U; j++)
                if ((pend >> j) & 1u) x[j] = T[j][b[j]];
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (!((pend >> j) & 1u)) continue;
                int32_t w;
                if (row_bucket<PACKED>(x[j], key[j], w)) {
                    c[j] = contrib(e[j].y, w);
                    pend &= ~(1u << j);
                } else {
                    b[j] = (b[j] + 1u) & ((1u << (meta[j] & 63u)) - 1u);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < U; j++) {
            if (term[j] != cur) {
#pragma unroll
                for (int q = 0; q < 9; q++)
                    if (q == cur) s[q] += run;
                run = 0;
                cur = term[j];
            }
            run += c[j];
        }
    }
#pragma unroll
    for (int q = 0; q < 9; q++)
        if (q == cur) s[q] += run;
    d[0] = 0;
#pragma unroll
    for (int p = 1; p <= 5; p++) {
        int64_t x = 0;
#pragma unroll
        for (int i = 0; i < 3; i++) x += (int64_t)s[3 * i + perm_of(p, i)] - s[3 * i + i];
        d[p] = x;
    }
    if (W > 1 && wv != 0) return;
    /* edges inside the triple: lane 3 a + b has vtx[a] -> vtx[b] and the
     * female weight f[a] -> f[b] */
    const int ia = lane < 9 ? lane / 3 : 0, ib = lane < 9 ? lane % 3 : 0;
    int32_t w = BM_ABSENT;
    if (lane < 9)
        w = row_find<PACKED>(g.m_out_t.tab, g.m_out_t.desc[sel3(ia, vtx[0], vtx[1], vtx[2])],
                             sel3(ib, vtx[0], vtx[1], vtx[2]));
    if (__ballot(w != BM_ABSENT) == 0) return;
    int32_t fw = BM_ABSENT;
    if (lane < 9)
        fw = row_find<PACKED>(g.f_out_t.tab, g.f_out_t.desc[sel3(ia, f[0], f[1], f[2])], sel3(ib, f[0], f[1], f[2]));
#pragma unroll
    for (int p = 1; p <= 5; p++) {
        const int na = ia == 0 ? perm_of(p, 0) : (ia == 1 ? perm_of(p, 1) : perm_of(p, 2));
        const int nb = ib == 0 ? perm_of(p, 0) : (ib == 1 ? perm_of(p, 1) : perm_of(p, 2));
        const int32_t nw = __shfl(fw, 3 * na + nb, BM_WAVE);
        if (w != BM_ABSENT) d[p] += (int64_t)contrib(w, nw) - contrib(w, fw);
    }
}

/* Best permutation of every triple, bound by lookups like k_swap (2,800 a
 * triple at n = 18,524 with 4M edges, against 3,900 and the building of six
 * LDS tables before: the 3-swap tool's enumerations 1.7x faster): W = 1, one wave per triple; W = 4, the
 * four waves of a block (see k_swap). */
template <bool PACKED, int U, int W>
__global__ void __launch_bounds__(W == 1 ? 512 : 64 * W) k_rot3(BmDevGraph g, int4* __restrict__ cand, int64_t k,
                                                                int64_t* __restrict__ best, uint8_t* __restrict__ perm,
                                                                int write_perm_into_cand) {
    __shared__ ScanList s_lists[8][18];
    __shared__ int64_t s_part[2][W][5];
    const int lane = threadIdx.x & (BM_WAVE - 1);
    const int wave = uni(threadIdx.x / BM_WAVE);
    const int wpb = W == 1 ? (int)(blockDim.x / BM_WAVE) : 1;
    const int64_t nw = (int64_t)gridDim.x * wpb;
    int par = 0;
    for (int64_t c = (int64_t)blockIdx.x * wpb + (W == 1 ? wave : 0); c < k; c += nw) {
        const int4 q = cand[c];
        const int32_t vtx[3] = {uni(q.x), uni(q.y), uni(q.z)};
        const int32_t f[3] = {uni(g.pi[vtx[0]]), uni(g.pi[vtx[1]]), uni(g.pi[vtx[2]])};
        int64_t d5[6];
        rot3_lists<PACKED, U, W>(g, g.pi, g.inv, vtx, f, s_lists[wave], lane, W == 1 ? 0 : wave, d5);
#pragma unroll
        for (int p = 1; p <= 5; p++) d5[p] = wave_sum64(d5[p]);
        if (W > 1) {
            /* two buffers: thread 0 has read one before the barrier after which it is written again */
            if (lane == 0) {
#pragma unroll
                for (int p = 1; p <= 5; p++) s_part[par][wave][p - 1] = d5[p];
            }
            __syncthreads();
            if (threadIdx.x == 0) {
#pragma unroll
                for (int p = 1; p <= 5; p++) {
                    d5[p] = 0;
#pragma unroll
                    for (int z = 0; z < W; z++) d5[p] += s_part[par][z][p - 1];
                }
            }
            par ^= 1;
        }
        if (lane == 0 && (W == 1 || wave == 0)) {
            int64_t bd = 0;
            int bp = 0;
#pragma unroll
            for (int p = 1; p <= 5; p++)
                if (d5[p] > bd) { bd = d5[p]; bp = p; }
            best[c] = bd;
            if (perm) perm[c] = (uint8_t)bp;
            if (write_perm_into_cand) cand[c].w = bp;
        }
    }
}

/* ------------------------------------------------------------------ */
/* Sums over the male lists: full score, current contributions, features */
/* ------------------------------------------------------------------ */

enum { kSumScore = 0, kSumDiag = 1, kSumFeature = 2 };
constexpr int kStageBuckets = 256;   /* largest row table staged per wave: 4 KB */

/* One wave per chunk of at most BM_EDGE_CHUNK entries of one vertex's male
 * list (the chunks depend only on the male graph), so a hub's lists spread
 * over many waves: every entry's contribution under the matching is a lookup
 * in the female row of the vertex's image.  Four entries per lane, each level
 * of their loads issued together.  A row table of at most 4 KB is first
 * copied to the wave's LDS slice: the 216 lookups of an average in-list hit
 * 2 KB of table, but with 32 waves' tables competing for a 32 KB L1 most of
 * them would each fetch a 128-byte line from L2 (both lists of the 4M-edge
 * pair: 78 us without the copy, 58 us with it).  What remains is the gather of
 * pi and the hubs' tables, which no LDS slice holds.  n = 18,524, 4M edges:
 * score 47 us (one wave per vertex, building its table first: 350-800 us, the
 * longest out-list set the time), features 58 us (8-byte linear-probing
 * tables, one dependent load per lane: 132 us).
 *   SCORE:   out-lists only, everything into out[0];
 *   DIAG:    out[x] += the contributions of x's out-edges and of its other
 *            in-edges (a self-loop counts once);
 *   FEATURE: out + 4 x += {contributions, weights, entries contributing 0}. */
template <bool PACKED, int MODE>
__global__ void __launch_bounds__(256) k_edge_sums(BmDevGraph g, const int4* __restrict__ chunks, int64_t nchunks,
                                                   int64_t* __restrict__ out) {
    constexpr int U = BM_EDGE_CHUNK / BM_WAVE;
    __shared__ uint4 s_tab[4][kStageBuckets];
    __shared__ int64_t s_part[4];
    const int lane = threadIdx.x & (BM_WAVE - 1);
    const int wave = uni(threadIdx.x / BM_WAVE);
    uint4* S = s_tab[wave];
    const int64_t nw = (int64_t)gridDim.x * 4;
    int64_t total = 0;
    for (int64_t ci = (int64_t)blockIdx.x * 4 + wave; ci < nchunks; ci += nw) {
        const int4 ch = chunks[ci];
        const int32_t x = uni(ch.x);
        const bool in = uni(ch.y) != 0;
        const int32_t cnt = uni(ch.w);
        const int2* __restrict__ adj = (in ? g.m_in + g.m_in_ptr[x] : g.m_out + g.m_out_ptr[x]) + uni(ch.z);
        int2 e[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int32_t i = lane + BM_WAVE * j;
            e[j] = i < cnt ? adj[i] : make_int2(0, 0);
        }
        const BmRowTab t = in ? g.f_in_t : g.f_out_t;
        const uint64_t d = (uint64_t)uni64((int64_t)t.desc[uni(g.pi[x])]);
        const uint4* __restrict__ T = t.tab + (d >> 6);
        const uint32_t lb = (uint32_t)(d & 63u), mask = (1u << lb) - 1u;
        int32_t key[U];
#pragma unroll
        for (int j = 0; j < U; j++) key[j] = g.pi[e[j].x];
        /* a copy costs one 16-byte load per bucket, a lookup about one and a half */
        const bool staged = (mask + 1u) <= (uint32_t)kStageBuckets && (int32_t)mask < 2 * cnt;
        if (staged) {
            wave_sync();
            for (uint32_t q = lane; q <= mask; q += BM_WAVE) S[q] = T[q];
            wave_sync();
        }
        uint32_t b[U], pend = 0;
#pragma unroll
        for (int j = 0; j < U; j++) {
            if (e[j].x == 0 || (MODE != kSumScore && in && e[j].x == x)) key[j] = 0;
            b[j] = row_home(key[j], lb);
            pend |= (key[j] != 0 ? 1u : 0u) << j;
        }
        int64_t sum = 0, ws = 0, hit = 0, used = 0;
        while (pend) {
            uint4 y[U];
#pragma unroll
            for (int j = 0; j < U; j++)
                if ((pend >> j) & 1u) y[j] = staged ? S[b[j]] : T[b[j]];
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (!((pend >> j) & 1u)) continue;
                int32_t w;
                if (row_bucket<PACKED>(y[j], key[j], w)) {
                    const int32_t c = contrib(e[j].y, w);
                    sum += c;
                    if (MODE == kSumFeature) hit += c != 0;
                    pend &= ~(1u << j);
                } else {
                    b[j] = (b[j] + 1u) & mask;
                }
            }
        }
        if (MODE == kSumScore) {
            total += sum;
            continue;
        }
        if (MODE == kSumFeature) {
#pragma unroll
            for (int j = 0; j < U; j++)
                if (e[j].x != 0 && !(in && e[j].x == x)) {
                    ws += e[j].y;
                    used++;
                }
        }
        sum = wave_sum64(sum);
        if (MODE == kSumDiag) {
            if (lane == 0 && sum != 0)
                atomicAdd(reinterpret_cast<unsigned long long*>(&out[x]), (unsigned long long)sum);
        } else {
            ws = wave_sum64(ws);
            const int64_t miss = wave_sum64(used - hit);
            if (lane < 3)
                atomicAdd(reinterpret_cast<unsigned long long*>(&out[4 * (int64_t)x + lane]),
                          (unsigned long long)(lane == 0 ? sum : (lane == 1 ? ws : miss)));
        }
    }
    if (MODE == kSumScore) {
        total = wave_sum64(total);
        if (lane == 0) s_part[wave] = total;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int64_t all = s_part[0] + s_part[1] + s_part[2] + s_part[3];
            if (all != 0) atomicAdd(reinterpret_cast<unsigned long long*>(out), (unsigned long long)all);
        }
    }
}

__global__ void __launch_bounds__(256) k_zero64(int64_t* __restrict__ p, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = 0;
}

/* ------------------------------------------------------------------ */
/* Annealing chains                                                    */
/* ------------------------------------------------------------------ */

/* One wave per chain (W = 1), or the four waves of a block (W = 4).  A step is
 * a chain of dependent loads (pi, list bounds, entries, pi or inverse,
 * buckets), so few chains are bound by its latency and many by the lookups:
 * four instances of n = 1,013 to 5,003 with 200 edges a vertex, 200 steps,
 * 1,024 chains 10.2 -> 4.5 ms, 8,192 chains 6.7e7 steps a second.  Step s of
 * a chain with stream seed q:
 *   kind:  r_k = rand(q2, s); a 3-vertex move if lo32(r_k) < p_rot3 (n >= 3);
 *   pool:  with a proposal pool of P pairs for the chain's instance,
 *          r_l = rand(q4, s); the move is built on pool entry
 *          range(hi32(r_l), P) if lo32(r_l) < p_pool;
 *   swap:  (u, v) = that pool pair, else uniform pair s of stream q0;
 *          delta exact;
 *   3-move: (a, b) = that pool pair and c = bm_third_vertex(q3, s, n, a, b),
 *          else (a, b, c) = uniform triple s of stream q3; permutation
 *          p = 1 + range(hi32(r_k), 5), delta of that permutation exact;
 *   accept if delta >= 0, else if U < exp(delta * beta_s) with
 *          U = (rand(q1, s) >> 11) * 2^-53 and beta_s = beta0 * exp(s * lam),
 *          exp being the deterministic bm_det_exp;
 * with q_i = rand(q, i).  The best matching is kept lazily: a chain standing
 * on its best score copies the matching aside only when it accepts a move
 * that lowers the score (the best is the latest matching reaching the
 * maximum).  The Metropolis rule and the geometric schedule follow
 * simulated_annealing (src/best-swap/score-lookup.c:345-400); its delta
 * comes from a lookup table and its stream from xoshiro256**, here the
 * delta is recomputed exactly every step and the streams are counter-based.
 * MIN = 4 holds the four-wave form to 128 registers, four blocks a CU instead
 * of three (one instance of n = 12,000, 200 edges a vertex, 10% 3-vertex moves,
 * 100 steps: 1,024 chains 2.71 -> 1.97 ms, 4,096 8.74 -> 7.50); its spills cost
 * up to 3% where three blocks hold all chains.
 * Each chain also sums the male degrees of the vertices of its moves (the
 * byte model of the delta kernels) and counts its 3-vertex and pool moves. */
template <bool PACKED, int U, bool ROT, int W, int MIN = 1>
__global__ void __launch_bounds__(W == 1 ? 512 : 64 * W, MIN) k_anneal(const BmDevGraph* __restrict__ insts,
                                                                  BmChain* __restrict__ chains, int64_t n_chains,
                                                                  int32_t* pool, int64_t steps, BmAnnealSched sc,
                                                                  int64_t* __restrict__ traj,
                                                                  const BmProposalPool* __restrict__ props) {
    __shared__ ScanList s_lists[8][ROT ? 18 : 8];
    __shared__ int64_t s_part[2][W];
    const int lane = threadIdx.x & (BM_WAVE - 1);
    const int wave = uni(threadIdx.x / BM_WAVE);
    const int wpb = W == 1 ? (int)(blockDim.x / BM_WAVE) : 1;
    ScanList* L = s_lists[wave];
    const int64_t nw = (int64_t)gridDim.x * wpb;
    int par = 0;
    for (int64_t c = (int64_t)blockIdx.x * wpb + (W == 1 ? wave : 0); c < n_chains; c += nw) {
        const BmChain ch = chains[c];
        const BmDevGraph& g = insts[uni(ch.inst)];
        const int32_t n = g.n;
        int32_t* pi = pool + uni64(ch.pi_off);
        int32_t* pib = pi + ((int64_t)n + 1);
        int32_t* inv = pib + ((int64_t)n + 1);
        const int32_t* ginv = g.inv ? inv : nullptr;   /* images are distinct, and stay so */
        const uint64_t q = (uint64_t)uni64((int64_t)ch.seed);
        const uint64_t q0 = bm_rand_at(q, 0), q1 = bm_rand_at(q, 1), q2 = bm_rand_at(q, 2), q3 = bm_rand_at(q, 3);
        const uint64_t q4 = bm_rand_at(q, 4);
        int64_t score = uni64(ch.score), best = uni64(ch.best), nacc = uni64(ch.accepted);
        int at_best = uni(ch.at_best);
        const int64_t s0 = uni64(ch.step);
        /* the instance's proposal pool (count 0: every move uniform) */
        const int2* pp = nullptr;
        int64_t pcount = 0;
        if (sc.p_pool && props) {
            pp = reinterpret_cast<const int2*>(uni64((int64_t)reinterpret_cast<uintptr_t>(props[uni(ch.inst)].pairs)));
            pcount = uni64(props[uni(ch.inst)].count);
        }
        int64_t dsw = 0, drt = 0, nrt = 0, npool = 0;
        for (int64_t s = s0; s < s0 + steps; s++) {
            const uint64_t rk = bm_rand_at(q2, (uint64_t)s);
            /* ROT = false: swap-only chains (p_rot3 == 0), built without the
             * 3-vertex path and its registers */
            const bool rot = ROT && n >= 3 && (uint64_t)(uint32_t)rk < sc.p_rot3;
            /* a move from the pool: entry range(hi32, count) of draw s of stream q4 */
            int2 from = make_int2(0, 0);
            if (pcount > 0) {
                const uint64_t rl = bm_rand_at(q4, (uint64_t)s);
                if ((uint64_t)(uint32_t)rl < sc.p_pool) {
                    from = pp[(int64_t)(((uint64_t)(uint32_t)(rl >> 32) * (uint64_t)pcount) >> 32)];
                    from.x = uni(from.x);
                    from.y = uni(from.y);
                    npool++;
                }
            }
            int32_t vtx[3] = {0, 0, 0}, f[3] = {0, 0, 0};
            int64_t d;
            int p = 0;
            if (!rot) {
                if (from.x) {
                    vtx[0] = from.x;
                    vtx[1] = from.y;
                } else {
                    bm_uniform_pair(q0, (uint64_t)s, n, &vtx[0], &vtx[1]);
                }
                dsw += uni64((g.m_out_ptr[vtx[0] + 1] - g.m_out_ptr[vtx[0]]) + (g.m_in_ptr[vtx[0] + 1] - g.m_in_ptr[vtx[0]]) +
                             (g.m_out_ptr[vtx[1] + 1] - g.m_out_ptr[vtx[1]]) + (g.m_in_ptr[vtx[1] + 1] - g.m_in_ptr[vtx[1]]));
                f[0] = uni(pi[vtx[0]]);
                f[1] = uni(pi[vtx[1]]);
                if (PACKED || g.packed)
                    d = (int64_t)swap_lists<true, 4, U, W>(g, pi, ginv, vtx[0], vtx[1], f[0], f[1], L, lane, W == 1 ? 0 : wave);
                else
                    d = swap_lists<false, 4, U, W>(g, pi, ginv, vtx[0], vtx[1], f[0], f[1], L, lane, W == 1 ? 0 : wave);
            } else {
                if (from.x) {
                    vtx[0] = from.x;
                    vtx[1] = from.y;
                    vtx[2] = bm_third_vertex(q3, (uint64_t)s, n, from.x, from.y);
                } else {
                    bm_uniform_triple(q3, (uint64_t)s, n, &vtx[0], &vtx[1], &vtx[2]);
                }
                nrt++;
#pragma unroll
                for (int i = 0; i < 3; i++)
                    drt += uni64((g.m_out_ptr[vtx[i] + 1] - g.m_out_ptr[vtx[i]]) + (g.m_in_ptr[vtx[i] + 1] - g.m_in_ptr[vtx[i]]));
#pragma unroll
                for (int i = 0; i < 3; i++) f[i] = uni(pi[vtx[i]]);
                int64_t d5[6];
                if (PACKED || g.packed)
                    rot3_lists<true, U, W>(g, pi, ginv, vtx, f, L, lane, W == 1 ? 0 : wave, d5);
                else
                    rot3_lists<false, U, W>(g, pi, ginv, vtx, f, L, lane, W == 1 ? 0 : wave, d5);
                p = 1 + (int)bm_range32((uint32_t)(rk >> 32), 5u);
                d = d5[1];
#pragma unroll
                for (int j = 2; j <= 5; j++)
                    if (p == j) d = d5[j];
            }
            d = wave_sum64(d);
            if (W > 1) {   /* two buffers, as in k_swap; every wave takes the same decision */
                if (lane == 0) s_part[par][wave] = d;
                __syncthreads();
                d = 0;
#pragma unroll
                for (int z = 0; z < W; z++) d += s_part[par][z];
                d = uni64(d);
                par ^= 1;
            }
            bool accept = d >= 0;
            if (!accept) {
                const double beta = sc.beta0 * bm_det_exp((double)s * sc.lam);
                const double x = (double)d * beta;
                const double r = (double)(bm_rand_at(q1, (uint64_t)s) >> 11) * 0x1p-53;
                accept = r < bm_det_exp(x);
            }
            if (!accept) continue;
            if (at_best && d < 0) {
                for (int64_t i = (W == 1 ? 0 : wave * BM_WAVE) + lane; i <= n; i += W * BM_WAVE) pib[i] = pi[i];
                at_best = 0;
                if (W > 1) __syncthreads();   /* copied before the move below changes it */
            }
            if (lane == 0 && (W == 1 || wave == 0)) {
                if (!rot) {
                    pi[vtx[0]] = f[1];
                    pi[vtx[1]] = f[0];
                    if (f[1]) inv[f[1]] = vtx[0];
                    if (f[0]) inv[f[0]] = vtx[1];
                } else {
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        const int32_t x = sel3(perm_of(p, i), f[0], f[1], f[2]);
                        pi[vtx[i]] = x;
                        if (x) inv[x] = vtx[i];
                    }
                }
            }
            __threadfence_block();
            if (W > 1) __syncthreads();
            score += d;
            nacc++;
            if (score >= best) {
                best = score;
                at_best = 1;
            }
        }
        if (lane == 0 && (W == 1 || wave == 0)) {
            BmChain o = ch;
            o.score = score;
            o.best = best;
            o.accepted = nacc;
            o.step = s0 + steps;
            o.at_best = at_best;
            o.deg_swap += dsw;
            o.deg_rot3 += drt;
            o.n_rot3 += nrt;
            o.n_learned += npool;
            if (traj && o.nseg < sc.traj_cap) traj[c * sc.traj_cap + o.nseg] = score;
            o.nseg++;
            chains[c] = o;
        }
    }
}

/* Persistent grid: never more blocks than can be resident at once. */
template <typename K>
hipError_t grid_of(K kernel, const BmLaunch& L, int64_t work, int waves, int per_block, dim3* grid, dim3* block) {
    *block = dim3(waves * BM_WAVE);
    int occ = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void*)kernel, (int)block->x, 0);
    if (e != hipSuccess) return e;
    int per_cu = L.blocks_per_cu < occ ? L.blocks_per_cu : occ;
    if (per_cu < 1) per_cu = 1;
    int64_t blocks = (work + per_block - 1) / per_block;
    const int64_t cap = (int64_t)per_cu * (L.num_cus > 0 ? L.num_cus : 256);
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    *grid = dim3((unsigned)blocks);
    return hipSuccess;
}

}  // namespace

template <int M, bool P, int U, int W, bool D>
static hipError_t launch_swap_one(const BmDevGraph& g, const BmLaunch& L, const int2* cand, const int64_t* off,
                                  uint64_t seed, int64_t k, int64_t* delta, const int64_t* diag, hipStream_t s) {
    const int waves = W == 1 ? L.waves_per_block : W;
    dim3 grid, block;
    const hipError_t e = grid_of(k_swap<M, P, U, W, D>, L, k, waves, W == 1 ? waves : 1, &grid, &block);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_swap<M, P, U, W, D>), grid, block, 0, s, g, cand, off, seed, k, delta, diag);
    return hipGetLastError();
}

template <int M, bool P, bool D>
static hipError_t launch_swap_u(const BmDevGraph& g, const BmLaunch& L, const int2* cand, const int64_t* off,
                                uint64_t seed, int64_t k, int64_t* delta, const int64_t* diag, hipStream_t s) {
    if (L.coop) return launch_swap_one<M, P, 4, 4, D>(g, L, cand, off, seed, k, delta, diag, s);
    if (L.unroll == 2) return launch_swap_one<M, P, 2, 1, D>(g, L, cand, off, seed, k, delta, diag, s);
    if (L.unroll == 8) return launch_swap_one<M, P, 8, 1, D>(g, L, cand, off, seed, k, delta, diag, s);
    return launch_swap_one<M, P, 4, 1, D>(g, L, cand, off, seed, k, delta, diag, s);
}

template <int M>
static hipError_t launch_swap_mode(const BmDevGraph& g, const BmLaunch& L, const int2* cand, const int64_t* off,
                                   uint64_t seed, int64_t k, int64_t* delta, const int64_t* diag, hipStream_t s) {
    if (g.packed)
        return diag ? launch_swap_u<M, true, true>(g, L, cand, off, seed, k, delta, diag, s)
                    : launch_swap_u<M, true, false>(g, L, cand, off, seed, k, delta, diag, s);
    return diag ? launch_swap_u<M, false, true>(g, L, cand, off, seed, k, delta, diag, s)
                : launch_swap_u<M, false, false>(g, L, cand, off, seed, k, delta, diag, s);
}

hipError_t bm_launch_swap(const BmDevGraph& g, const BmLaunch& L, int mode, const int2* cand, const int64_t* off,
                          uint64_t seed, int64_t k, int64_t* delta, const int64_t* diag, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    if (mode == BM_CAND_LIST) return launch_swap_mode<BM_CAND_LIST>(g, L, cand, off, seed, k, delta, diag, s);
    if (mode == BM_CAND_UMAJOR) return launch_swap_mode<BM_CAND_UMAJOR>(g, L, cand, off, seed, k, delta, diag, s);
    return launch_swap_mode<BM_CAND_UNIFORM>(g, L, cand, off, seed, k, delta, diag, s);
}

template <bool P, int U, int W>
static hipError_t launch_rot3_one(const BmDevGraph& g, const BmLaunch& L, const int4* cand, int64_t k, int64_t* best,
                                  uint8_t* perm, int4* cand_out_perm, hipStream_t s) {
    const int waves = W == 1 ? L.waves_per_block : W;
    dim3 grid, block;
    const hipError_t e = grid_of(k_rot3<P, U, W>, L, k, waves, W == 1 ? waves : 1, &grid, &block);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_rot3<P, U, W>), grid, block, 0, s, g, const_cast<int4*>(cand), k, best, perm,
                       cand_out_perm ? 1 : 0);
    return hipGetLastError();
}

/* 3-vertex kernel: 2 or 4 list entries per lane in flight (L.unroll). */
hipError_t bm_launch_rot3(const BmDevGraph& g, const BmLaunch& L, const int4* cand, int64_t k, int64_t* best,
                          uint8_t* perm, int4* cand_out_perm, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    if (g.packed) {
        if (L.coop) return launch_rot3_one<true, 4, 4>(g, L, cand, k, best, perm, cand_out_perm, s);
        return L.unroll == 2 ? launch_rot3_one<true, 2, 1>(g, L, cand, k, best, perm, cand_out_perm, s)
                             : launch_rot3_one<true, 4, 1>(g, L, cand, k, best, perm, cand_out_perm, s);
    }
    if (L.coop) return launch_rot3_one<false, 4, 4>(g, L, cand, k, best, perm, cand_out_perm, s);
    return L.unroll == 2 ? launch_rot3_one<false, 2, 1>(g, L, cand, k, best, perm, cand_out_perm, s)
                         : launch_rot3_one<false, 4, 1>(g, L, cand, k, best, perm, cand_out_perm, s);
}

/* Annealing chains: 2 or 4 list entries per lane in flight (L.unroll), or four
 * waves a chain (L.coop; 2: in 128 registers). */
template <typename F>
static hipError_t with_anneal(int packed, int rot, const BmLaunch& L, F f) {
#define BM_ANNEAL_W(P, R) \
    (L.coop ? (R && L.coop == 2 ? f(k_anneal<P, 4, R, 4, R ? 4 : 1>) : f(k_anneal<P, 4, R, 4>)) : (L.unroll == 2 ? f(k_anneal<P, 2, R, 1>) : f(k_anneal<P, 4, R, 1>)))
    if (packed) return rot ? BM_ANNEAL_W(true, true) : BM_ANNEAL_W(true, false);
    return rot ? BM_ANNEAL_W(false, true) : BM_ANNEAL_W(false, false);
#undef BM_ANNEAL_W
}

hipError_t bm_anneal_grid(int packed, int rot, const BmLaunch& L, int64_t n_chains, dim3* grid, dim3* block) {
    const int waves = L.coop ? 4 : L.waves_per_block;
    return with_anneal(packed, rot, L, [&](auto kern) {
        return grid_of(kern, L, n_chains, waves, L.coop ? 1 : waves, grid, block);
    });
}

hipError_t bm_launch_anneal(const BmDevGraph* insts, int packed, BmChain* chains, int64_t n_chains, int32_t* pool,
                            int64_t steps, const BmAnnealSched& sc, int64_t* traj, const BmProposalPool* proposals,
                            const BmLaunch& L, dim3 grid, dim3 block, hipStream_t s) {
    if (n_chains <= 0 || steps <= 0) return hipSuccess;
    return with_anneal(packed, sc.p_rot3 != 0, L, [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, block, 0, s, insts, chains, n_chains, pool, steps, sc, traj, proposals);
        return hipGetLastError();
    });
}

/* Chains back to their start: a block per chain at a time copies its
 * instance's matching (n+1, then its inverse) to the chain's current and best
 * matchings and inverse. */
__global__ void __launch_bounds__(256) k_anneal_reset(const BmDevGraph* __restrict__ insts,
                                                      const BmChain* __restrict__ chains, int64_t n_chains,
                                                      const int32_t* __restrict__ init,
                                                      const int64_t* __restrict__ init_off, int32_t* __restrict__ pool) {
    for (int64_t c = blockIdx.x; c < n_chains; c += gridDim.x) {
        const BmChain& ch = chains[c];
        const int64_t len = (int64_t)insts[ch.inst].n + 1;
        const int32_t* from = init + init_off[ch.inst];
        int32_t* to = pool + ch.pi_off;
        for (int64_t i = threadIdx.x; i < len; i += blockDim.x) {
            const int32_t f = from[i];
            to[i] = f;
            to[len + i] = f;
            to[2 * len + i] = from[len + i];
        }
    }
}

hipError_t bm_launch_anneal_reset(const BmDevGraph* insts, const BmChain* chains, int64_t n_chains,
                                  const int32_t* init, const int64_t* init_off, int32_t* pool, hipStream_t s) {
    /* fewer than 2^32 threads, whatever the number of chains */
    const int64_t blocks = n_chains < (1 << 20) ? n_chains : 1 << 20;
    hipLaunchKernelGGL(k_anneal_reset, dim3((unsigned)blocks), dim3(256), 0, s, insts, chains, n_chains, init, init_off, pool);
    return hipGetLastError();
}

template <int MODE>
static hipError_t launch_edge_sums(const BmDevGraph& g, const int4* chunks, int64_t nchunks, int64_t* out,
                                   int32_t num_cus, hipStream_t s) {
    if (nchunks <= 0) return hipSuccess;
    int64_t blocks = (nchunks + 3) / 4;
    const int64_t cap = (int64_t)(num_cus > 0 ? num_cus : 256) * 8;
    if (blocks > cap) blocks = cap;
    auto kern = g.packed ? k_edge_sums<true, MODE> : k_edge_sums<false, MODE>;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, s, g, chunks, nchunks, out);
    return hipGetLastError();
}

hipError_t bm_launch_score(const BmDevGraph& g, const int4* chunks, int64_t n_out_chunks, int64_t* acc,
                           int32_t num_cus, hipStream_t s) {
    return launch_edge_sums<kSumScore>(g, chunks, n_out_chunks, acc, num_cus, s);
}

hipError_t bm_launch_diag(const BmDevGraph& g, const int4* chunks, int64_t nchunks, int64_t* diag, int32_t num_cus,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_zero64, dim3((unsigned)((g.n + 256) / 256)), dim3(256), 0, s, diag, (int64_t)g.n + 1);
    return launch_edge_sums<kSumDiag>(g, chunks, nchunks, diag, num_cus, s);
}

hipError_t bm_launch_feature_sums(const BmDevGraph& g, const int4* chunks, int64_t nchunks, int64_t* acc,
                                  int32_t num_cus, hipStream_t s) {
    return launch_edge_sums<kSumFeature>(g, chunks, nchunks, acc, num_cus, s);
}
