/*
 * Small device helpers shared by the kernel translation units.
 */
#ifndef BM_DEVUTIL_H
#define BM_DEVUTIL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#define BM_ABSENT INT32_MIN
#define BM_WAVE 64

namespace bmd {

/* Exact contribution of a male edge of weight w whose image is a female
 * lookup result fw: min(w, fw) when the female edge exists, else 0. */
__device__ __forceinline__ int32_t contrib(int32_t w, int32_t fw) {
    return fw == BM_ABSENT ? 0 : (w < fw ? w : fw);
}

__device__ __forceinline__ int32_t uni(int32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint32_t uniu(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ int64_t uni64(int64_t x) {
    uint32_t lo = uniu((uint32_t)x), hi = uniu((uint32_t)((uint64_t)x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

/* Compiler fence for wave-private LDS: a wave's LDS operations execute in
 * order, so only reordering by the compiler has to be prevented. */
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int64_t wave_sum64(int64_t x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        int lo = __shfl_xor((int)(uint32_t)x, o, BM_WAVE);
        int hi = __shfl_xor((int)(uint32_t)((uint64_t)x >> 32), o, BM_WAVE);
        x += (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
    }
    return x;
}

/* New female index (0..2) of position i under permutation p (1..5), in the
 * numbering of calculateThreeNodeSwapKernel's table
 * (src/graph-re-alignment-gpu-3-swap.cu:167-174):
 * 1 (f1,f3,f2)  2 (f2,f1,f3)  3 (f2,f3,f1)  4 (f3,f1,f2)  5 (f3,f2,f1). */
__host__ __device__ __forceinline__ int perm_of(int p, int i) {
    switch (p) {
        case 1: return i == 0 ? 0 : (i == 1 ? 2 : 1);
        case 2: return i == 0 ? 1 : (i == 1 ? 0 : 2);
        case 3: return i == 0 ? 1 : (i == 1 ? 2 : 0);
        case 4: return i == 0 ? 2 : (i == 1 ? 0 : 1);
        case 5: return i == 0 ? 2 : (i == 1 ? 1 : 0);
        default: return i;
    }
}

/* Entry i (< off[n+1]) of a u-major pair stream with offsets off[1..n+1]:
 * the vertex u whose range [off[u], off[u+1]) holds i. */
__device__ __forceinline__ int32_t umajor_owner(const int64_t* __restrict__ off, int32_t n, int64_t i) {
    int32_t lo = 1, hi = n;   /* smallest u with off[u + 1] > i */
    while (lo < hi) {
        const int32_t m = (lo + hi) >> 1;
        if (off[m + 1] > i) hi = m; else lo = m + 1;
    }
    return lo;
}

template <typename T>
__device__ __forceinline__ T sel3(int j, const T& a, const T& b, const T& c) {
    return j == 0 ? a : (j == 1 ? b : c);
}

/* Best of the five permutations of a triple from its nine gains Gv[i][j] =
 * G(vtx_i, f_j), the male self-loops s and female self-loops fs of f_0..f_2
 * (BM_ABSENT when missing), the male weights w[i][j] of edges inside the
 * triple and the female weights F[x][y] = w_F(f_x, f_y) (needed only where a
 * male edge exists).  An edge i -> j is corrected exactly: under permutation
 * p it contributes c(w, F(f_pi, f_pj)) where the gains counted
 * c(w, F(f_pi, f_j)) and c(w, F(f_i, f_pj)) and the old score
 * c(w, F(f_i, f_j)); all of these are among the nine F[x][y].  bd = the
 * largest positive delta (0 if none), bp its permutation (first p on ties). */
__device__ __forceinline__ void rot3_from_gains(const int64_t (*Gv)[3], const int32_t (*w)[3], const int32_t (*F)[3],
                                                const int32_t* s, const int32_t* fs, int64_t& bd, int& bp) {
    bd = 0;
    bp = 0;
#pragma unroll
    for (int p = 1; p <= 5; p++) {
        int64_t d = 0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int pi = perm_of(p, i);
            d += sel3(pi, Gv[i][0], Gv[i][1], Gv[i][2]) - Gv[i][i];
            if (s[i] != BM_ABSENT) d += contrib(s[i], fs[pi]) - (int64_t)contrib(s[i], fs[i]);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                if (i == j) continue;
                const int pj = perm_of(p, j);
                const int32_t x = w[i][j];
                if (x != BM_ABSENT)
                    d += (int64_t)contrib(x, F[pi][pj]) - contrib(x, F[pi][j]) - contrib(x, F[i][pj]) +
                         contrib(x, F[i][j]);
            }
        }
        if (d > bd) { bd = d; bp = p; }
    }
}

}  // namespace bmd

#endif
