/*
 * Deltas of the reference's changed-first enumerations
 * (src/graph-re-alignment-gpu-swap.cu:163-195,
 * src/graph-re-alignment-gpu-3-swap.cu:67-150) from placement rows.
 *
 * All candidates of an enumeration share a few changed vertices, so instead of
 * intersecting lists per candidate (bm_delta.hip) each changed vertex u with
 * image f gets two rows, computed once:
 *   R_u(f') = G(u, f')  u placed on every female f', and
 *   K_u(v)  = G(v, f)   every male v placed on f,
 * where G(x, y) is the score of x's incident edges (self-loops excluded) with
 * x alone moved to y (bm_gain.hip).  R_u adds min(w, w_F) over the female rows
 * of u's mapped neighbours, K_u over the male lists of f's mapped neighbours.
 * With the current contribution of every vertex (bm_launch_diag) a pair is
 * then two reads and its edge and self-loop corrections, a triple six.  At
 * n = 18,524 with 4M edges a row is about 0.9M additions, a vertex's 18,523
 * pairs 10M lookups: the 3.7M pairs of 200 changed vertices 83 ms by list
 * scans, 1.2 ms here; 37,045 pairs of two 1-8 ms, 0.1 ms; 280,000 triples of
 * five 8-22 ms, 0.2 ms.
 */
#include "bm_device.h"
#include "bm_devutil.h"
#include "bm_rowtab.h"

using namespace bmd;

namespace {

constexpr int kRowThreads = 512, kRowWaves = kRowThreads / BM_WAVE;
constexpr int kRowEdges = 256;   /* source edges set up together */
constexpr int kRowUnit = 256;    /* target entries per wave and step: four per lane */

/* Bound by the LDS additions and, for a few changed vertices, by the latency of
 * the set-up: 4 rows of ordinary vertices 20 us, 26 rows 52 us, 400 rows of
 * hub-biased vertices 0.8 ms (n = 18,524, 4M edges).
 * Block (r, s): split s of row r (r < g: R of changed[r]; else K of
 * changed[r - g]) into its partial row.  The split's source edges are taken
 * 256 at a time: a thread finds its edge's target list, a block scan numbers
 * the lists' 256-entry units, and the waves take units in turn (so a hub's
 * long list spreads over them), the next unit's entries loading while the
 * last one's are added to the LDS row.  Two blocks per CU up to n = 18,911. */
__global__ void __launch_bounds__(kRowThreads) k_place_rows(BmDevGraph g, const int32_t* __restrict__ changed,
                                                            int32_t ng, int32_t splits, int32_t stride,
                                                            int32_t* __restrict__ rows) {
    extern __shared__ int32_t acc[];
    __shared__ int64_t s_base[kRowEdges];
    __shared__ int32_t s_len[kRowEdges], s_w[kRowEdges], s_x[kRowEdges];
    __shared__ alignas(16) int32_t s_incl[kRowEdges];
    __shared__ int32_t s_wave[kRowEdges / BM_WAVE];
    const int t = threadIdx.x, lane = t & (BM_WAVE - 1), wave = uni(t / BM_WAVE);
    const int32_t r = blockIdx.x / splits, split = blockIdx.x % splits;
    const bool col = r >= ng;
    const int32_t u = changed[col ? r - ng : r];
    const int32_t from = col ? g.pi[u] : u;
    const int32_t* map = col ? g.inv : g.pi;
    for (int32_t i = t; i < stride; i += kRowThreads) acc[i] = 0;
    __syncthreads();
    for (int dir = 0; dir < 2; dir++) {
        /* out-edges of the source reach the in-lists of the other graph and the reverse */
        const int64_t* sp = col ? (dir ? g.f_in_ptr : g.f_out_ptr) : (dir ? g.m_in_ptr : g.m_out_ptr);
        const int2* sa = col ? (dir ? g.f_in : g.f_out) : (dir ? g.m_in : g.m_out);
        const int64_t* tp = col ? (dir ? g.m_out_ptr : g.m_in_ptr) : (dir ? g.f_out_ptr : g.f_in_ptr);
        const int2* ta = col ? (dir ? g.m_out : g.m_in) : (dir ? g.f_out : g.f_in);
        const int64_t b = sp[from], n_edges = sp[from + 1] - b;
        const int64_t e0 = b + n_edges * split / splits, e1 = b + n_edges * (split + 1) / splits;
        for (int64_t eb = e0; eb < e1; eb += kRowEdges) {
            if (t < kRowEdges) {
                int32_t len = 0, w = 0, x = 0;
                int64_t base = 0;
                if (eb + t < e1) {
                    const int2 e = sa[eb + t];
                    w = e.y;
                    x = map[e.x];
                    base = tp[x];
                    len = (int32_t)(tp[x + 1] - base);
                    if (!col && e.x == u) len = 0;   /* a self-loop */
                }
                const int32_t units = (len + kRowUnit - 1) / kRowUnit;
                int32_t incl = units;
#pragma unroll
                for (int o = 1; o < BM_WAVE; o <<= 1) {
                    const int32_t y = __shfl_up(incl, o, BM_WAVE);
                    if (lane >= o) incl += y;
                }
                s_base[t] = base;
                s_len[t] = len;
                s_w[t] = w;
                s_x[t] = col ? x : 0;   /* an entry equal to x is a male self-loop */
                s_incl[t] = incl;
                if (lane == BM_WAVE - 1) s_wave[wave] = incl;
            }
            __syncthreads();
            /* lane l holds the running unit counts of edges 4 l .. 4 l + 3 */
            int4 v = *reinterpret_cast<const int4*>(&s_incl[4 * lane]);
            int32_t add = 0, total = 0;
#pragma unroll
            for (int q = 0; q < kRowEdges / BM_WAVE; q++) {
                if (q < lane / 16) add += s_wave[q];
                total += s_wave[q];
            }
            v.x += add;
            v.y += add;
            v.z += add;
            v.w += add;
            total = uni(total);
            int2 nx[4];
            int32_t nw = 0, nself = 0;
            const auto load = [&](int32_t unit) {
                const int l = __popcll(__ballot(v.w <= unit));
                const int32_t a = __builtin_amdgcn_readlane(v.x, l), c = __builtin_amdgcn_readlane(v.y, l),
                              d = __builtin_amdgcn_readlane(v.z, l);
                const int idx = 4 * l + (a <= unit) + (c <= unit) + (d <= unit);
                const int32_t prev = (a > unit) ? (l ? __builtin_amdgcn_readlane(v.w, l - 1) : 0)
                                                : ((c > unit) ? a : ((d > unit) ? c : d));
                const int32_t off = (unit - prev) * kRowUnit, len = s_len[idx];
                const int2* p = ta + s_base[idx] + off;
                nw = s_w[idx];
                nself = s_x[idx];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int32_t i = BM_WAVE * j + lane;
                    nx[j] = off + i < len ? p[i] : make_int2(0, 0);
                }
            };
            if (wave < total) load(wave);
            for (int32_t unit = wave; unit < total; unit += kRowWaves) {
                int2 e[4];
#pragma unroll
                for (int j = 0; j < 4; j++) e[j] = nx[j];
                const int32_t w = nw, self = nself;
                if (unit + kRowWaves < total) load(unit + kRowWaves);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (e[j].x != 0 && e[j].x != self) atomicAdd(&acc[e[j].x], w < e[j].y ? w : e[j].y);
            }
            __syncthreads();
        }
    }
    int4* out = reinterpret_cast<int4*>(rows + (int64_t)blockIdx.x * stride);
    const int4* in = reinterpret_cast<const int4*>(acc);
    for (int32_t i = t; i < stride / 4; i += kRowThreads) out[i] = in[i];
}

/* The partials of each row summed into its first one. */
__global__ void __launch_bounds__(256) k_sum_rows(int32_t n_rows, int32_t splits, int32_t stride,
                                                  int32_t* __restrict__ rows) {
    const int32_t quads = stride / 4;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n_rows * quads) return;
    const int32_t r = (int32_t)(i / quads), q = (int32_t)(i % quads);
    int4* p = reinterpret_cast<int4*>(rows + (int64_t)r * splits * stride) + q;
    int4 sum = p[0];
#pragma unroll 8
    for (int32_t s = 1; s < splits; s++) {
        const int4 x = p[(int64_t)s * quads];
        sum.x += x.x;
        sum.y += x.y;
        sum.z += x.z;
        sum.w += x.w;
    }
    p[0] = sum;
}

struct PlaceRows {
    const int32_t* rows;
    const int32_t* changed;   /* this group's vertices, ascending */
    int64_t pitch;            /* splits x stride */
    int32_t ng;
    const int64_t* diag;
    const int32_t* m_self;
    const int32_t* f_self;
};

__device__ __forceinline__ int32_t place_index(const PlaceRows& P, int32_t u) {
    int32_t lo = 0, hi = P.ng - 1;
    while (lo < hi) {
        const int32_t m = (lo + hi) >> 1;
        if (P.changed[m] < u) lo = m + 1; else hi = m;
    }
    return lo;
}
__device__ __forceinline__ int64_t place_r(const PlaceRows& P, int32_t i, int32_t f) { return P.rows[i * P.pitch + f]; }
__device__ __forceinline__ int64_t place_k(const PlaceRows& P, int32_t i, int32_t v) {
    return P.rows[(P.ng + i) * P.pitch + v];
}

/* Weights of the male edges x -> y and y -> x from x's two row tables. */
template <bool PACKED>
__device__ __forceinline__ void edges_between(const BmDevGraph& g, int32_t x, int32_t y, int32_t& xy, int32_t& yx) {
    xy = row_find<PACKED>(g.m_out_t.tab, g.m_out_t.desc[x], y);
    yx = row_find<PACKED>(g.m_in_t.tab, g.m_in_t.desc[x], y);
}
template <bool PACKED>
__device__ __forceinline__ int32_t female_w(const BmDevGraph& g, int32_t a, int32_t b) {
    return row_find<PACKED>(g.f_out_t.tab, g.f_out_t.desc[a], b);
}

/* Pairs [a0, a0 + la) and [b0, b0 + lb) of the enumeration, all with their
 * first vertex in the group.  u on f2 and v on f1, every other vertex where it
 * is: R_u(f2) + K_u(v) price an edge u <-> v against the partner's old image
 * and leave self-loops out; both are put right from the four female weights
 * among f1 and f2.  The current contributions count an edge u <-> v twice. */
template <bool PACKED>
__global__ void __launch_bounds__(256) k_changed_pairs(BmDevGraph g, PlaceRows P, const int2* __restrict__ cand,
                                                       int64_t a0, int64_t la, int64_t b0, int64_t lb,
                                                       int64_t* __restrict__ delta) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < la + lb; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t idx = t < la ? a0 + t : b0 + (t - la);
        const int2 c = cand[idx];
        const int32_t u = c.x, v = c.y, f1 = g.pi[u], f2 = g.pi[v];
        const int32_t i = place_index(P, u);
        int64_t d = place_r(P, i, f2) + place_k(P, i, v) - P.diag[u] - P.diag[v];
        int32_t uv, vu;
        edges_between<PACKED>(g, u, v, uv, vu);
        const int32_t su = P.m_self[u], sv = P.m_self[v];
        if (uv != BM_ABSENT || vu != BM_ABSENT) {
            const int32_t F12 = female_w<PACKED>(g, f1, f2), F21 = female_w<PACKED>(g, f2, f1), F11 = P.f_self[f1],
                          F22 = P.f_self[f2];
            if (uv != BM_ABSENT)
                d += (int64_t)contrib(uv, F21) - contrib(uv, F22) - contrib(uv, F11) + contrib(uv, F12);
            if (vu != BM_ABSENT)
                d += (int64_t)contrib(vu, F12) - contrib(vu, F11) - contrib(vu, F22) + contrib(vu, F21);
        }
        if (su != BM_ABSENT) d += contrib(su, P.f_self[f2]);
        if (sv != BM_ABSENT) d += contrib(sv, P.f_self[f1]);
        delta[idx] = d;
    }
}

/* G(x, f) and G(y, f') of the neighbouring unchanged vertices of the third
 * section: wave j takes (x, y) = (r_j, r_{j+1}), their images crossed, and
 * walks the shorter side of each list (k_swap's lists, self-loops left out).
 * out[2 j] = G(x, pi(y)), out[2 j + 1] = G(y, pi(x)). */
template <bool PACKED>
__global__ void __launch_bounds__(256) k_cross_terms(BmDevGraph g, const int4* __restrict__ cand, int32_t count,
                                                     int64_t* __restrict__ out) {
    const int lane = threadIdx.x & (BM_WAVE - 1);
    const int32_t nw = (int32_t)(gridDim.x * (blockDim.x / BM_WAVE));
    for (int32_t j = (int32_t)(blockIdx.x * (blockDim.x / BM_WAVE)) + uni(threadIdx.x / BM_WAVE); j < count; j += nw) {
        const int4 q = cand[j];
#pragma unroll
        for (int z = 0; z < 2; z++) {
            const int32_t x = uni(z ? q.z : q.y), y = uni(z ? q.y : q.z), f = uni(g.pi[y]);
            int64_t sum = 0;
#pragma unroll
            for (int in = 0; in < 2; in++) {
                const int64_t* mp = in ? g.m_in_ptr : g.m_out_ptr;
                const int64_t* fp = in ? g.f_in_ptr : g.f_out_ptr;
                const int64_t m0 = mp[x], f0 = fp[f];
                const int32_t dm = (int32_t)(mp[x + 1] - m0), df = (int32_t)(fp[f + 1] - f0);
                const bool side = df < dm;
                const int2* rows = side ? (in ? g.f_in : g.f_out) + f0 : (in ? g.m_in : g.m_out) + m0;
                const BmRowTab& t = side ? (in ? g.m_in_t : g.m_out_t) : (in ? g.f_in_t : g.f_out_t);
                const uint64_t desc = (uint64_t)uni64((int64_t)t.desc[side ? x : f]);
                const int32_t len = side ? df : (df ? dm : 0);
                const uint4* T = t.tab + (desc >> 6);
                const uint32_t lb = (uint32_t)(desc & 63u), mask = (1u << lb) - 1u;
                for (int32_t i0 = lane; i0 < len; i0 += 4 * BM_WAVE) {   /* four entries in flight */
                    int2 e[4];
                    int32_t key[4];
                    uint32_t b[4], pend = 0;
#pragma unroll
                    for (int u = 0; u < 4; u++) e[u] = i0 + BM_WAVE * u < len ? rows[i0 + BM_WAVE * u] : make_int2(0, 0);
#pragma unroll
                    for (int u = 0; u < 4; u++) key[u] = (side ? g.inv : g.pi)[e[u].x];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        if (e[u].x == 0 || (side ? key[u] : e[u].x) == x) key[u] = 0;
                        b[u] = row_home(key[u], lb);
                        pend |= (key[u] != 0 ? 1u : 0u) << u;
                    }
                    while (pend) {
                        uint4 y[4];
#pragma unroll
                        for (int u = 0; u < 4; u++)
                            if ((pend >> u) & 1u) y[u] = T[b[u]];
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            if (!((pend >> u) & 1u)) continue;
                            int32_t w;
                            if (row_bucket<PACKED>(y[u], key[u], w)) {
                                sum += contrib(e[u].y, w);
                                pend &= ~(1u << u);
                            } else {
                                b[u] = (b[u] + 1u) & mask;
                            }
                        }
                    }
                }
            }
            sum = wave_sum64(sum);
            if (lane == 0) out[2 * (int64_t)j + z] = sum;
        }
    }
}

/* Best permutation of every triple of the enumeration: a is changed; b too in
 * the first two sections (idx < s2); in the third b and d are neighbours in
 * the unchanged order, whose two terms come from `cross` (rest of them). */
template <bool PACKED>
__global__ void __launch_bounds__(256) k_changed_triples(BmDevGraph g, PlaceRows P, int4* __restrict__ cand, int64_t k,
                                                         int64_t s2, int64_t rest, const int64_t* __restrict__ cross,
                                                         int64_t* __restrict__ best, uint8_t* __restrict__ perm) {
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < k; idx += (int64_t)gridDim.x * blockDim.x) {
        const int4 q = cand[idx];
        const int32_t vtx[3] = {q.x, q.y, q.z};
        int32_t f[3], s[3], fs[3];
        int64_t Gv[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            f[i] = g.pi[vtx[i]];
            s[i] = P.m_self[vtx[i]];
            fs[i] = P.f_self[f[i]];
            Gv[i][i] = P.diag[vtx[i]] - (s[i] != BM_ABSENT ? contrib(s[i], fs[i]) : 0);
        }
        const int32_t i = place_index(P, vtx[0]);
        Gv[0][1] = place_r(P, i, f[1]);
        Gv[0][2] = place_r(P, i, f[2]);
        Gv[2][0] = place_k(P, i, vtx[2]);
        if (idx < s2) {
            const int32_t j = place_index(P, vtx[1]);
            Gv[1][0] = place_r(P, j, f[0]);
            Gv[1][2] = place_r(P, j, f[2]);
            Gv[2][1] = place_k(P, j, vtx[2]);
        } else {
            const int64_t j = (idx - s2) % rest;
            Gv[1][0] = place_k(P, i, vtx[1]);
            Gv[1][2] = cross[2 * j];
            Gv[2][1] = cross[2 * j + 1];
        }
        int32_t w[3][3], F[3][3];
#pragma unroll
        for (int x = 0; x < 3; x++)
#pragma unroll
            for (int y = 0; y < 3; y++) w[x][y] = F[x][y] = BM_ABSENT;
        edges_between<PACKED>(g, vtx[0], vtx[1], w[0][1], w[1][0]);
        edges_between<PACKED>(g, vtx[0], vtx[2], w[0][2], w[2][0]);
        edges_between<PACKED>(g, vtx[1], vtx[2], w[1][2], w[2][1]);
        bool any = false;
#pragma unroll
        for (int x = 0; x < 3; x++)
#pragma unroll
            for (int y = 0; y < 3; y++) any = any || (x != y && w[x][y] != BM_ABSENT);
        if (any) {
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int y = 0; y < 3; y++) F[x][y] = x == y ? fs[x] : female_w<PACKED>(g, f[x], f[y]);
        }
        int64_t bd;
        int bp;
        rot3_from_gains(Gv, w, F, s, fs, bd, bp);
        best[idx] = bd;
        perm[idx] = (uint8_t)bp;
        cand[idx].w = bp;
    }
}

unsigned blocks_for(int64_t work, int threads) {
    int64_t b = (work + threads - 1) / threads;
    if (b < 1) b = 1;
    return (unsigned)(b > 65536 ? 65536 : b);
}

}  // namespace

size_t bm_place_lds(int64_t stride) {
    return (size_t)stride * sizeof(int32_t) + kRowEdges * (sizeof(int64_t) + 4 * sizeof(int32_t)) + 64;
}

/* Splits of each of 2 ng rows: enough blocks to fill the device several
 * times over (a hub's row is five times an ordinary one), at most 32 partials
 * per row to add up. */
int32_t bm_place_splits(int32_t ng) {
    const int32_t s = BM_PLACE_ROWS / (2 * ng);
    return s > 32 ? 32 : (s < 1 ? 1 : s);
}

hipError_t bm_launch_place_rows(const BmDevGraph& g, const int32_t* changed, int32_t ng, int64_t stride, int32_t* rows,
                                hipStream_t s) {
    const int32_t splits = bm_place_splits(ng);
    const size_t lds = (size_t)stride * sizeof(int32_t);
    const hipError_t e = hipFuncSetAttribute((const void*)k_place_rows, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_place_rows, dim3((unsigned)(2 * ng * splits)), dim3(kRowThreads), lds, s, g, changed, ng, splits,
                       (int32_t)stride, rows);
    if (splits > 1)
        hipLaunchKernelGGL(k_sum_rows, dim3((unsigned)((2 * (int64_t)ng * (stride / 4) + 255) / 256)), dim3(256), 0, s,
                           2 * ng, splits, (int32_t)stride, rows);
    return hipGetLastError();
}

static PlaceRows place_rows(const BmPlace& p) {
    PlaceRows P;
    P.rows = p.rows;
    P.changed = p.changed;
    P.pitch = (int64_t)bm_place_splits(p.ng) * p.stride;
    P.ng = p.ng;
    P.diag = p.diag;
    P.m_self = p.m_self;
    P.f_self = p.f_self;
    return P;
}

hipError_t bm_launch_changed_pairs(const BmDevGraph& g, const BmPlace& p, const int2* cand, int64_t a0, int64_t la,
                                   int64_t b0, int64_t lb, int64_t* delta, hipStream_t s) {
    if (la + lb <= 0) return hipSuccess;
    auto kern = g.packed ? k_changed_pairs<true> : k_changed_pairs<false>;
    hipLaunchKernelGGL(kern, dim3(blocks_for(la + lb, 256)), dim3(256), 0, s, g, place_rows(p), cand, a0, la, b0, lb,
                       delta);
    return hipGetLastError();
}

hipError_t bm_launch_changed_triples(const BmDevGraph& g, const BmPlace& p, int4* cand, int64_t k, int64_t s2,
                                     int64_t rest, int64_t* cross, int64_t* best, uint8_t* perm, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    if (k > s2) {
        auto terms = g.packed ? k_cross_terms<true> : k_cross_terms<false>;
        hipLaunchKernelGGL(terms, dim3(blocks_for(rest, 4)), dim3(256), 0, s, g, cand + s2, (int32_t)rest, cross);
    }
    auto kern = g.packed ? k_changed_triples<true> : k_changed_triples<false>;
    hipLaunchKernelGGL(kern, dim3(blocks_for(k, 256)), dim3(256), 0, s, g, place_rows(p), cand, k, s2, rest > 0 ? rest : 1,
                       cross, best, perm);
    return hipGetLastError();
}
