/*
 * Learned swap proposal (gfx950): a 16 -> 128 -> 128 -> 1 perceptron in BF16
 * with FP32 accumulation on the matrix cores, with hand-written forward and
 * backward kernels.  It scores candidate pairs from per-vertex features of
 * the current matching; a search sends only the top candidates of a large
 * pool to the exact delta kernels, so the score stays exact whatever the
 * network predicts.  There is no counterpart in the reference (its proposals
 * are uniform, score-weighted or 2-hop: src/graph-re-alignment-gpu-swap.cu:816-887,
 * src/refine-twohop-random.c:676-693).
 *
 * Model (x = the 16 pair features, bf() = rounding to bfloat16, nearest even):
 *   z1 = bf(x) @ bf(W1) + b1          W1: 16 x 128
 *   h1 = bf(relu(z1))
 *   z2 = h1 @ bf(W2) + b2             W2: 128 x 128
 *   h2 = relu(z2)                     (fp32)
 *   y  = h2 . w3 + b3                 (fp32)
 * Loss: mean (y - t)^2 with t = sign(delta) log(1 + |delta|).  Backward:
 *   dy = 2 (y - t) / B;  dw3 = sum h2 dy;  db3 = sum dy
 *   g2 = bf(dy w3 * [z2 > 0]);  dW2 = h1^T g2;  db2 = sum g2 (unrounded)
 *   g1 = bf((g2 @ bf(W2)^T) * [z1 > 0]);  dW1 = bf(x)^T g1;  db1 = sum g1 (unrounded)
 * Products with K = 16 (layer 1) run on v_mfma_f32_16x16x16_bf16, those with
 * K = 128 or K = the batch (layer 2, the backward through W2, the weight
 * gradients) on gfx950's v_mfma_f32_16x16x32_bf16.  The scoring kernel
 * computes the transposed products (z^T = W^T x^T: the weights are the A
 * operand), so each lane ends a layer holding four consecutive hidden units of
 * one pair: h1 goes to LDS in 8-byte stores and the output layer's sum over
 * hidden units is one in-lane sum plus two shuffles.  The weight-gradient
 * products use activations stored transposed (feature-major) so that every
 * operand fragment is one 16-byte load.
 *
 * Fragment layouts (64 lanes, l = lane, q = l / 16):
 *   16x16x16: A lane l holds A[l % 16][4q + i], B holds B[4q + i][l % 16], i < 4;
 *   16x16x32: A lane l holds A[l % 16][8q + i], B holds B[8q + i][l % 16], i < 8;
 *   both:     D lane l holds D[4q + j][l % 16], j < 4.
 * Weights are kept in "fragment order": for a K x N matrix W and k-steps of
 * KB = 16 or 32 rows, fragment (s, t) (rows KB s.., columns 16 t..) stores
 * lane l's KB / 4 values W[KB s + (KB / 4) q + i][16 t + l % 16] contiguously.
 * The same array serves as the B operand of W and as the A operand of W^T.
 *
 * Per-vertex features (8 per vertex; a pair's 16 are u's then v's):
 *   log1p d_out, log1p d_in, log1p (weight sum), L / (weight sum + 1),
 *   unmatched-edge fraction, log1p d_out_F(pi), log1p d_in_F(pi), log1p L,
 * with L = the score carried by the vertex's incident edges under pi and an
 * edge "unmatched" when its contribution is 0.
 */
#include "bm_device.h"
#include "bm_devutil.h"
#include "bm_rng.h"

#include <hipcub/hipcub.hpp>

using namespace bmd;

namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kF = 16;     /* features per pair */
constexpr int kH = 128;    /* hidden width */
constexpr int kT = kH / 16;   /* 16-wide tiles per hidden layer */
constexpr int kS = kH / 32;   /* 32-deep k-steps over a hidden layer */
/* parameter layout */
constexpr int kOffW1 = 0, kOffB1 = kF * kH, kOffW2 = kOffB1 + kH, kOffB2 = kOffW2 + kH * kH, kOffW3 = kOffB2 + kH,
              kOffB3 = kOffW3 + kH, kParams = kOffB3 + 1;

/* bfloat16 bits of x, rounded to nearest even (v_cvt_pk_bf16_f32). */
__device__ __forceinline__ short bf16_of(float x) { return __builtin_bit_cast(short, (__bf16)x); }

__device__ __forceinline__ v4f mfma(v4s a, v4s b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v4f mfma32(v8s a, v8s b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0,
                                                    0);
}

/* Second half of the per-vertex features: one thread per vertex turns the
 * exact integer sums of its edges (bm_launch_feature_sums: contributions,
 * weights, entries contributing 0) into the 8 floats and clears them. */
__global__ void k_feature_finish(BmDevGraph g, longlong4* __restrict__ acc, float4* __restrict__ vf) {
    for (int32_t x = blockIdx.x * blockDim.x + threadIdx.x; x <= g.n; x += gridDim.x * blockDim.x) {
        if (x == 0) {
            vf[0] = make_float4(0.f, 0.f, 0.f, 0.f);
            vf[1] = make_float4(0.f, 0.f, 0.f, 0.f);
            continue;
        }
        const longlong4 a = acc[x];
        acc[x] = make_longlong4(0, 0, 0, 0);
        const int64_t L = a.x, wsum = a.y, miss = a.z;
        const int32_t fx = g.pi[x];
        const float dout = (float)(g.m_out_ptr[x + 1] - g.m_out_ptr[x]), din = (float)(g.m_in_ptr[x + 1] - g.m_in_ptr[x]);
        const float fo = fx ? (float)(g.f_out_ptr[fx + 1] - g.f_out_ptr[fx]) : 0.f;
        const float fi = fx ? (float)(g.f_in_ptr[fx + 1] - g.f_in_ptr[fx]) : 0.f;
        const float ws = (float)(wsum > 0 ? wsum : 0);
        const float Lf = (float)(L > 0 ? L : 0);
        vf[2 * (int64_t)x] = make_float4(log1pf(dout), log1pf(din), log1pf(ws), Lf / (ws + 1.f));
        vf[2 * (int64_t)x + 1] = make_float4((float)miss / (dout + din + 1.f), log1pf(fo), log1pf(fi), log1pf(Lf));
    }
}

/* Weights in fragment order with k-steps of KB rows (16 or 32), for a KK x NN
 * matrix M:
 * frag[((s * (NN / 16) + t) * 64 + l) * (KB / 4) + i] = M[KB s + (KB / 4) (l / 16) + i][16 t + l % 16].
 * Place of element (r, c) there. */
template <int KB>
__device__ __forceinline__ int frag_at(int r, int c, int NN) {
    constexpr int per = KB / 4;
    const int s = r / KB, rr = r % KB;
    return ((s * (NN / 16) + c / 16) * 64 + 16 * (rr / per) + c % 16) * per + rr % per;
}

/* The bf16 copies of parameter i with value x: W1 once, W2 as itself and
 * transposed; biases and w3 stay fp32. */
__device__ __forceinline__ void pack_param(short* __restrict__ W1f, short* __restrict__ W2f, short* __restrict__ W2Tf,
                                           int i, float x) {
    if (i < kF * kH) {
        W1f[frag_at<16>(i / kH, i % kH, kH)] = bf16_of(x);
    } else if (i >= kOffW2 && i < kOffW2 + kH * kH) {
        const int r = (i - kOffW2) / kH, c = (i - kOffW2) % kH;
        W2f[frag_at<32>(r, c, kH)] = bf16_of(x);
        W2Tf[frag_at<32>(c, r, kH)] = bf16_of(x);
    }
}

__global__ void k_mlp_pack(const float* __restrict__ p, short* __restrict__ W1f, short* __restrict__ W2f,
                           short* __restrict__ W2Tf) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < kParams; i += gridDim.x * blockDim.x)
        pack_param(W1f, W2f, W2Tf, i, p[i]);
}

struct MlpDev {
    const v4s* W1f;     /* 1 x 8 fragments (k-step 16) of W1 (16 x 128) */
    const v8s* W2f;     /* 4 x 8 fragments (k-step 32) of W2 (128 x 128) */
    const v8s* W2Tf;    /* 4 x 8 fragments (k-step 32) of W2^T */
    const float* b1;
    const float* b2;
    const float* w3;
    const float* b3;
};

/* Candidate pair p of a proposal source. */
struct PairSrc {
    const int2* list;   /* explicit pairs, or NULL for the uniform stream */
    uint64_t seed;
    int32_t n;
};

__device__ __forceinline__ int2 pair_at(const PairSrc& ps, int64_t p) {
    if (ps.list) return ps.list[p];
    int32_t u, v;
    bm_uniform_pair(ps.seed, (uint64_t)p, ps.n, &u, &v);
    return make_int2(u, v);
}

constexpr int kHistBins = 4096;   /* first 12 bits of the order-preserving score bits */
constexpr int kHPad = kH + 8;   /* padded bf16 row of a staged 16 x 128 tile (272 bytes: 16-byte reads hit distinct banks) */

template <typename Shared>
__device__ __forceinline__ void stage_weights(Shared& S, const MlpDev& M) {
    for (int q = threadIdx.x; q < kT * 64; q += blockDim.x) S.W1[q] = M.W1f[q];
    for (int q = threadIdx.x; q < kS * kT * 64; q += blockDim.x) S.W2[q] = M.W2f[q];
    for (int q = threadIdx.x; q < kH; q += blockDim.x) {
        S.b1[q] = M.b1[q];
        S.b2[q] = M.b2[q];
        S.w3[q] = M.w3[q];
    }
}

/* Input fragment of a 16-pair tile: lane l holds features 4 (l / 16) .. +3
 * of pair l % 16 (u's features 0..7, v's 8..15) -- the A operand of x W1
 * and, equally, the B operand of W1^T x^T. */
__device__ __forceinline__ v4s input_frag(const float4* __restrict__ vf, int2 uv, bool valid, int lane) {
    const int q = lane / 16;
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) f = vf[2 * (int64_t)(q < 2 ? uv.x : uv.y) + (q & 1)];
    v4s a;
    a[0] = bf16_of(f.x);
    a[1] = bf16_of(f.y);
    a[2] = bf16_of(f.z);
    a[3] = bf16_of(f.w);
    return a;
}

/* Layer 1 for one tile in the pair-major form (training): z1 (D layout:
 * lane l has pairs 4 (l / 16) + j of hidden unit 16 t + l % 16, kept for the
 * backward mask) and h1 into the wave's LDS tile. */
template <typename Shared>
__device__ __forceinline__ void layer1(const Shared& S, short (*Ht)[kHPad], v4s xa, v4f* z1, int lane) {
#pragma unroll
    for (int t = 0; t < kT; t++) {
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        acc = mfma(xa, S.W1[t * 64 + lane], acc);
        const int col = 16 * t + (lane % 16);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] += S.b1[col];
            Ht[4 * (lane / 16) + j][col] = bf16_of(acc[j] > 0.f ? acc[j] : 0.f);
        }
        z1[t] = acc;
    }
}

/* 32-deep fragments (kS k-steps) of the wave's staged 16 x 128 bf16 tile:
 * lane l gets row l % 16, columns 32 s + 8 (l / 16) .. +7 (one 16-byte read). */
__device__ __forceinline__ void load_tile32(const short (*Ht)[kHPad], v8s* a, int lane) {
#pragma unroll
    for (int s = 0; s < kS; s++) a[s] = *reinterpret_cast<const v8s*>(&Ht[lane % 16][32 * s + 8 * (lane / 16)]);
}

/* Forward: scores of k pairs, in the transposed form: z1^T = W1^T x^T (A =
 * W1^T fragments, B = the input fragment) leaves lane l with hidden units
 * 16 t + 4 (l / 16) .. +3 of pair l % 16, stored to the pair's LDS row in one
 * 8-byte write per t; z2^T = W2^T h1^T takes h1^T fragments as 16-byte reads
 * of those rows; the output layer sums the lane's 32 hidden units, then over
 * the four lanes of the pair.
 *
 * A tile is 640 MFMA cycles but reads 36 KB of weights and 1.5 KB of biases
 * from LDS (290 cycles of the CU's one LDS port per wave, so four SIMDs wait
 * for it), so a wave takes kFwdTiles tiles with each weight read, and one
 * block of 16 waves per CU shares one copy of the weights (four waves per
 * SIMD; with 4-wave blocks the 54 KB per block left two).  The next tiles'
 * features load while this one's products run.  2^20 pairs: 104 -> 58 us
 * (three or four tiles per weight read spill). */
constexpr int kScoreThreads = 1024, kScoreWaves = kScoreThreads / BM_WAVE, kFwdTiles = 2;

struct ScoreShared {
    v4s W1[kT * 64];
    v8s W2[kS * kT * 64];
    float b1[kH], b2[kH], w3[kH];
    short Ht[kScoreWaves][16][kHPad];
};

template <bool HIST>
__global__ void __launch_bounds__(kScoreThreads) k_mlp_forward(const float4* __restrict__ vf, PairSrc ps, int64_t k,
                                                               MlpDev M, float* __restrict__ score,
                                                               uint32_t* __restrict__ hist) {
    extern __shared__ uint4 smem[];
    ScoreShared& S = *reinterpret_cast<ScoreShared*>(smem);
    uint32_t* h0 = reinterpret_cast<uint32_t*>(&S + 1);   /* HIST: first digit of the ranking select */
    if (HIST)
        for (int i = threadIdx.x; i < kHistBins; i += blockDim.x) h0[i] = 0;
    stage_weights(S, M);
    __syncthreads();
    const int lane = threadIdx.x & (BM_WAVE - 1), wave = threadIdx.x / BM_WAVE;
    const int q = lane / 16;
    short(*Ht)[kHPad] = S.Ht[wave];
    const float b3 = M.b3[0];
    const int64_t groups = (k + 16 * kFwdTiles - 1) / (16 * kFwdTiles);
    const int64_t step = (int64_t)gridDim.x * kScoreWaves;
    int64_t gr = (int64_t)wave * gridDim.x + blockIdx.x;   /* few groups go to as many blocks */
    v4s xn[kFwdTiles];
#pragma unroll
    for (int z = 0; z < kFwdTiles; z++) {
        const int64_t p = (gr * kFwdTiles + z) * 16 + (lane % 16);
        xn[z] = input_frag(vf, p < k ? pair_at(ps, p) : make_int2(0, 0), p < k, lane);
    }
    for (; gr < groups; gr += step) {
        v4s xb[kFwdTiles];
#pragma unroll
        for (int z = 0; z < kFwdTiles; z++) {
            xb[z] = xn[z];
            const int64_t p = ((gr + step) * kFwdTiles + z) * 16 + (lane % 16);
            xn[z] = input_frag(vf, p < k ? pair_at(ps, p) : make_int2(0, 0), p < k, lane);
        }
        v8s hb[kFwdTiles][kS];
#pragma unroll
        for (int z = 0; z < kFwdTiles; z++) {
#pragma unroll 4
            for (int t = 0; t < kT; t++) {
                v4f acc = {0.f, 0.f, 0.f, 0.f};
                acc = mfma(S.W1[t * 64 + lane], xb[z], acc);
                const float4 b1 = *reinterpret_cast<const float4*>(&S.b1[16 * t + 4 * q]);
                const float bb[4] = {b1.x, b1.y, b1.z, b1.w};
                v4s h;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float y = acc[j] + bb[j];
                    h[j] = bf16_of(y > 0.f ? y : 0.f);
                }
                *reinterpret_cast<v4s*>(&Ht[lane % 16][16 * t + 4 * q]) = h;
            }
            wave_sync();
            load_tile32(Ht, hb[z], lane);
            wave_sync();
        }
        float part[kFwdTiles];
#pragma unroll
        for (int z = 0; z < kFwdTiles; z++) part[z] = 0.f;
#pragma unroll 2   /* fully unrolled, the weight reads move up and spill */
        for (int t = 0; t < kT; t++) {
            v4f acc[kFwdTiles];
#pragma unroll
            for (int z = 0; z < kFwdTiles; z++) acc[z] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s2 = 0; s2 < kS; s2++) {
                const v8s w = S.W2[(s2 * kT + t) * 64 + lane];
#pragma unroll
                for (int z = 0; z < kFwdTiles; z++) acc[z] = mfma32(w, hb[z][s2], acc[z]);
            }
            const float4 b2 = *reinterpret_cast<const float4*>(&S.b2[16 * t + 4 * q]);
            const float4 w3 = *reinterpret_cast<const float4*>(&S.w3[16 * t + 4 * q]);
            const float bb[4] = {b2.x, b2.y, b2.z, b2.w}, ww[4] = {w3.x, w3.y, w3.z, w3.w};
#pragma unroll
            for (int z = 0; z < kFwdTiles; z++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float h2 = acc[z][j] + bb[j];
                    part[z] += (h2 > 0.f ? h2 : 0.f) * ww[j];
                }
        }
#pragma unroll
        for (int z = 0; z < kFwdTiles; z++) {
            part[z] += __shfl_xor(part[z], 16, BM_WAVE);
            part[z] += __shfl_xor(part[z], 32, BM_WAVE);
            const int64_t p = (gr * kFwdTiles + z) * 16 + (lane % 16);
            if (lane < 16 && p < k) {
                const float y = part[z] + b3;
                score[p] = y;
                if (HIST) {
                    const uint32_t u = __float_as_uint(y);
                    atomicAdd(&h0[((u & 0x80000000u) ? ~u : (u | 0x80000000u)) >> 20], 1u);
                }
            }
        }
    }
    if (HIST) {
        __syncthreads();
        for (int i = threadIdx.x; i < kHistBins; i += blockDim.x)
            if (h0[i]) atomicAdd(&hist[i], h0[i]);
    }
}

/* Regression target of an exact int64 delta: sign(d) log(1 + |d|). */
__device__ __forceinline__ float delta_target(int64_t d) {
    const double x = (double)d;
    return (float)(x < 0 ? -log1p(-x) : log1p(x));
}

/* Training pass over a batch of B pairs (B a multiple of 32): forward, loss,
 * and the backward through the activations.  Stores bf(x)^T (16 x B), h1^T,
 * g1^T and g2^T (128 x B) for the weight-gradient products.  The bias
 * gradients, dw3 and the summed squared error stay in registers over all of a
 * wave's tiles, are summed per block in LDS and written as one partial per
 * block, which k_mlp_adam / k_mlp_reduce add up in a fixed order.  Added to
 * the gradient per 16-pair tile they were 1.6M device-wide atomics per 65,536
 * pairs, which run at about 1.3e10 a second here: 221 us, now 31 us.  Eight
 * waves per block share the weights (two per SIMD). */
struct TrainBuf {
    short* XT;      /* 16 x B */
    short* H1T;     /* 128 x B */
    short* G1T;     /* 128 x B */
    short* G2T;     /* 128 x B */
    float* wpart;   /* slices x kWParams: weight gradients (dW1 then dW2) of each slice */
    float* bpart;   /* kBParams x blocks: db1, db2, dw3, db3 and the summed squared error of each block */
    const float* target;    /* one of the two */
    const int64_t* delta;   /* targets are delta_target of these */
    int64_t B;
    int64_t ld;     /* row stride of the four */
};

/* W1 and W2 in the partials; the other parameters in bpart's order, then the loss. */
constexpr int kWParams = kF * kH + kH * kH, kBParams = 3 * kH + 2;

constexpr int kTrainThreads = 512, kTrainWaves = kTrainThreads / BM_WAVE;

struct TrainShared {
    v4s W1[kT * 64];
    v8s W2[kS * kT * 64];
    float b1[kH], b2[kH], w3[kH];
    v8s W2T[kS * kT * 64];
    float part[kTrainWaves][kBParams];
    short Ht[kTrainWaves][16][kHPad];
};

__global__ void __launch_bounds__(kTrainThreads) k_mlp_train_act(const float4* __restrict__ vf, PairSrc ps, int64_t k,
                                                                 MlpDev M, TrainBuf T) {
    extern __shared__ uint4 smem[];
    TrainShared& S = *reinterpret_cast<TrainShared*>(smem);
    stage_weights(S, M);
    for (int q = threadIdx.x; q < kS * kT * 64; q += blockDim.x) S.W2T[q] = M.W2Tf[q];
    __syncthreads();
    const int lane = threadIdx.x & (BM_WAVE - 1), wave = threadIdx.x / BM_WAVE;
    short(*Ht)[kHPad] = S.Ht[wave];
    const float b3 = M.b3[0];
    const float inv = 2.f / (float)k;
    const int64_t ld = T.ld;
    const int64_t tiles = T.B / 16;
    float ab1[kT], ab2[kT], aw3[kT], ab3 = 0.f, ase = 0.f;
#pragma unroll
    for (int t = 0; t < kT; t++) ab1[t] = ab2[t] = aw3[t] = 0.f;
    for (int64_t tile = (int64_t)blockIdx.x * kTrainWaves + wave; tile < tiles; tile += (int64_t)gridDim.x * kTrainWaves) {
        const int64_t base = tile * 16;
        const int64_t p = base + (lane % 16);
        const bool valid = p < k;
        const int2 uv = valid ? pair_at(ps, p) : make_int2(0, 0);
        const v4s xa = input_frag(vf, uv, valid, lane);
        float tg[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t q = base + 4 * (lane / 16) + j;
            tg[j] = q >= k ? 0.f : (T.delta ? delta_target(T.delta[q]) : T.target[q]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) T.XT[(int64_t)(4 * (lane / 16) + i) * ld + p] = xa[i];
        v4f z1[kT];
        layer1(S, Ht, xa, z1, lane);
        wave_sync();
        v8s a[kS];
        load_tile32(Ht, a, lane);
        /* h1^T: rows 4 (l/16) + j of column c are 4 consecutive pairs */
#pragma unroll
        for (int t = 0; t < kT; t++) {
            const int col = 16 * t + (lane % 16);
            v4s h;
#pragma unroll
            for (int j = 0; j < 4; j++) h[j] = Ht[4 * (lane / 16) + j][col];
            *reinterpret_cast<v4s*>(&T.H1T[(int64_t)col * ld + base + 4 * (lane / 16)]) = h;
        }
        v4f z2[kT];
        float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < kT; t++) {
            v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < kS; s++) acc = mfma32(a[s], S.W2[(s * kT + t) * 64 + lane], acc);
            const int col = 16 * t + (lane % 16);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[j] += S.b2[col];
                part[j] += (acc[j] > 0.f ? acc[j] : 0.f) * S.w3[col];
            }
            z2[t] = acc;
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) part[j] += __shfl_xor(part[j], o, BM_WAVE);
        /* dy for this lane's four rows (every lane of a 16-lane group has the sums) */
        float dy[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool ok = base + 4 * (lane / 16) + j < k;
            const float y = part[j] + b3;
            const float r = ok ? y - tg[j] : 0.f;
            dy[j] = r * inv;
            if ((lane % 16) == 0) {
                ase += r * r;
                ab3 += dy[j];
            }
        }
        /* g2 = bf(dy w3 [z2 > 0]); dw3 += h2 dy; db2 += dy w3 [z2 > 0] */
        wave_sync();
#pragma unroll
        for (int t = 0; t < kT; t++) {
            const int col = 16 * t + (lane % 16);
            v4s gv;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float h = z2[t][j] > 0.f ? z2[t][j] : 0.f;
                const float g = z2[t][j] > 0.f ? dy[j] * S.w3[col] : 0.f;
                ab2[t] += g;
                aw3[t] += h * dy[j];
                gv[j] = bf16_of(g);
                Ht[4 * (lane / 16) + j][col] = gv[j];
            }
            *reinterpret_cast<v4s*>(&T.G2T[(int64_t)col * ld + base + 4 * (lane / 16)]) = gv;
        }
        wave_sync();
        /* g1 = bf((g2 @ W2^T) [z1 > 0]) */
        v8s ga[kS];
        load_tile32(Ht, ga, lane);
#pragma unroll
        for (int t = 0; t < kT; t++) {
            v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < kS; s++) acc = mfma32(ga[s], S.W2T[(s * kT + t) * 64 + lane], acc);
            const int col = 16 * t + (lane % 16);
            v4s gv;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float g = z1[t][j] > 0.f ? acc[j] : 0.f;
                ab1[t] += g;
                gv[j] = bf16_of(g);
            }
            *reinterpret_cast<v4s*>(&T.G1T[(int64_t)col * ld + base + 4 * (lane / 16)]) = gv;
        }
        wave_sync();
    }
#pragma unroll
    for (int t = 0; t < kT; t++) {
        float x[3] = {ab1[t], ab2[t], aw3[t]};
#pragma unroll
        for (int j = 0; j < 3; j++) {
            x[j] += __shfl_xor(x[j], 16, BM_WAVE);
            x[j] += __shfl_xor(x[j], 32, BM_WAVE);
        }
        if (lane < 16) {
#pragma unroll
            for (int j = 0; j < 3; j++) S.part[wave][j * kH + 16 * t + lane] = x[j];
        }
    }
    ab3 += __shfl_xor(ab3, 16, BM_WAVE);
    ab3 += __shfl_xor(ab3, 32, BM_WAVE);
    ase += __shfl_xor(ase, 16, BM_WAVE);
    ase += __shfl_xor(ase, 32, BM_WAVE);
    if (lane == 0) {
        S.part[wave][3 * kH] = ab3;
        S.part[wave][3 * kH + 1] = ase;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < kBParams; q += blockDim.x) {
        float sum = 0.f;
        for (int w = 0; w < kTrainWaves; w++) sum += S.part[w][q];
        T.bpart[(int64_t)q * gridDim.x + blockIdx.x] = sum;
    }
}

/* Weight gradients: dW1 = bf(x)^T g1 (16 x 128), dW2 = h1^T g2 (128 x 128),
 * 32 batch entries per MFMA.  Work item = (block of output tiles, slice of
 * the batch), one 4-wave block each: its waves take a quarter of the slice,
 * each accumulating the whole 32 x 64 (dW2) or 16 x 64 (dW1) block, so an
 * operand fragment loaded from L2 serves two or four products; they sum in
 * LDS, in wave order, and write the slice's partial.  One tile per wave and
 * atomics into the gradient took 44 us per 65,536 pairs, bound by the
 * 590,000 atomics; now 28 us. */
constexpr int kWgRows = 2, kWgCols = 4;
constexpr int kWgItems = kT / kWgCols + (kT / kWgRows) * (kT / kWgCols);

__global__ void __launch_bounds__(256) k_mlp_wgrad(TrainBuf T, int32_t slices) {
    __shared__ float s_sum[4][kWgRows * kWgCols][256];
    const int lane = threadIdx.x & (BM_WAVE - 1), wave = threadIdx.x / BM_WAVE;
    const int64_t ld = T.ld;
    const int64_t steps = T.B / 32;
    const int item = (int)(blockIdx.x % kWgItems), slice = (int)(blockIdx.x / kWgItems);
    const bool first = item < kT / kWgCols;           /* dW1, else dW2 */
    const int it2 = item - kT / kWgCols;
    const int mt = first ? 0 : it2 / (kT / kWgCols) * kWgRows, nt = (first ? item : it2 % (kT / kWgCols)) * kWgCols;
    const int rows = first ? 1 : kWgRows;
    const short* AT = first ? T.XT : T.H1T;           /* rows = input features / neurons */
    const short* BT = first ? T.G1T : T.G2T;          /* rows = output neurons */
    const int64_t parts = 4 * (int64_t)slices, part = 4 * (int64_t)slice + wave;
    const int64_t s0 = steps * part / parts, s1 = steps * (part + 1) / parts;
    v4f acc[kWgRows][kWgCols];
#pragma unroll
    for (int r = 0; r < kWgRows; r++)
#pragma unroll
        for (int c = 0; c < kWgCols; c++) acc[r][c] = v4f{0.f, 0.f, 0.f, 0.f};
    const short* ap = AT + (int64_t)(16 * mt + lane % 16) * ld + 8 * (lane / 16);
    const short* bp = BT + (int64_t)(16 * nt + lane % 16) * ld + 8 * (lane / 16);
    v8s an[kWgRows], bn[kWgCols];   /* the next step's fragments load while this one's products run */
    const auto load = [&](int64_t s) {
#pragma unroll
        for (int r = 0; r < kWgRows; r++) an[r] = *reinterpret_cast<const v8s*>(ap + (r < rows ? 16 * r * ld : 0) + 32 * s);
#pragma unroll
        for (int c = 0; c < kWgCols; c++) bn[c] = *reinterpret_cast<const v8s*>(bp + 16 * c * ld + 32 * s);
    };
    if (s0 < s1) load(s0);
    for (int64_t s = s0; s < s1; s++) {
        v8s a[kWgRows], b[kWgCols];
#pragma unroll
        for (int r = 0; r < kWgRows; r++) a[r] = an[r];
#pragma unroll
        for (int c = 0; c < kWgCols; c++) b[c] = bn[c];
        if (s + 1 < s1) load(s + 1);
#pragma unroll
        for (int r = 0; r < kWgRows; r++)
#pragma unroll
            for (int c = 0; c < kWgCols; c++) acc[r][c] = mfma32(a[r], b[c], acc[r][c]);
    }
#pragma unroll
    for (int r = 0; r < kWgRows; r++)
#pragma unroll
        for (int c = 0; c < kWgCols; c++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                s_sum[wave][r * kWgCols + c][64 * j + lane] = acc[r][c][j];
    __syncthreads();
    float* out = T.wpart + (int64_t)slice * kWParams + (first ? 0 : kF * kH);
    for (int i = threadIdx.x; i < rows * kWgCols * 256; i += 256) {
        const int tile = i / 256, j = (i % 256) / 64, l = i % 64;
        const int r = 16 * (mt + tile / kWgCols) + 4 * (l / 16) + j, c = 16 * (nt + tile % kWgCols) + l % 16;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < 4; w++) sum += s_sum[w][tile][64 * j + l];
        out[r * kH + c] = sum;
    }
}

/* Partials of one batch's gradient. */
struct GradParts {
    const float* w;
    const float* b;
    int32_t slices, blocks;
};

constexpr int kGradThreads = 256;
/* blocks summing W1 and W2 (a thread per parameter over the slices), then one
 * wave per other parameter (and the loss) over the blocks */
constexpr int kGradWBlocks = kWParams / kGradThreads, kGradBBlocks = (kBParams + 3) / 4;

/* The gradient value of this thread's parameter and its index (-1: none;
 * kParams: the summed squared error), every slice and block added in order. */
__device__ __forceinline__ float grad_sum(const GradParts& P, int* param) {
    *param = -1;
    if ((int)blockIdx.x < kGradWBlocks) {
        const int i = blockIdx.x * kGradThreads + threadIdx.x;
        float sum = 0.f;
#pragma unroll 8
        for (int q = 0; q < P.slices; q++) sum += P.w[(int64_t)q * kWParams + i];
        *param = i < kF * kH ? kOffW1 + i : kOffW2 + (i - kF * kH);
        return sum;
    }
    const int q = ((int)blockIdx.x - kGradWBlocks) * 4 + threadIdx.x / BM_WAVE, lane = threadIdx.x & (BM_WAVE - 1);
    if (q >= kBParams) return 0.f;
    float sum = 0.f;
    for (int i = lane; i < P.blocks; i += BM_WAVE) sum += P.b[(int64_t)q * P.blocks + i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, BM_WAVE);
    if (lane == 0)
        *param = q < kH ? kOffB1 + q
                        : (q < 2 * kH ? kOffB2 + q - kH : (q < 3 * kH ? kOffW3 + q - 2 * kH : (q == 3 * kH ? kOffB3 : kParams)));
    return sum;
}

/* The whole gradient and the loss of a batch. */
__global__ void __launch_bounds__(kGradThreads) k_mlp_reduce(GradParts P, float* __restrict__ g, float* loss) {
    int i;
    const float x = grad_sum(P, &i);
    if (i == kParams) *loss = x;
    else if (i >= 0) g[i] = x;
}

/* Adam on the fp32 master parameters and their bf16 copies, from the batch's
 * partials; the summed squared error goes to *loss. */
__global__ void __launch_bounds__(kGradThreads) k_mlp_adam(GradParts P, float* __restrict__ p, float* __restrict__ m,
                                                           float* __restrict__ v, float lr, float b1c, float b2c,
                                                           short* __restrict__ W1f, short* __restrict__ W2f,
                                                           short* __restrict__ W2Tf, float* loss) {
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    int i;
    const float gi = grad_sum(P, &i);
    if (i == kParams) *loss = gi;
    if (i < 0 || i >= kParams) return;
    const float mi = beta1 * m[i] + (1.f - beta1) * gi;
    const float vi = beta2 * v[i] + (1.f - beta2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float x = p[i] - lr * (mi / b1c) / (sqrtf(vi / b2c) + eps);
    p[i] = x;
    pack_param(W1f, W2f, W2Tf, i, x);
}

__global__ void k_iota(int32_t* __restrict__ p, int64_t k) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < k; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = (int32_t)i;
}

/* Pairs of the top-ranked stream indices into a pair list. */
__global__ void k_gather_stream_pairs(uint64_t seed, int32_t n, const int32_t* __restrict__ idx, int64_t top,
                                      int2* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < top; i += (int64_t)gridDim.x * blockDim.x) {
        int32_t u, v;
        bm_uniform_pair(seed, (uint64_t)idx[i], n, &u, &v);
        out[i] = make_int2(u, v);
    }
}

/* ---- top of the ranked pool: radix select over distinct 64-bit keys ---- */

/* key(p) = order-preserving bits of score p (the float order, -0 below +0)
 * in the high half, 2^32 - 1 - p in the low half: a larger key is a larger
 * score, ties to the smaller pool index, and no two keys are equal -- the
 * order of a stable descending sort of the scores. */
__device__ __forceinline__ uint64_t rank_key(float x, int64_t p) {
    uint32_t u = __float_as_uint(x);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((uint64_t)u << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)p);
}

constexpr int kSelBits = 12, kSelBins = 1 << kSelBits, kSelThreads = 256;
static_assert(kSelBins == kHistBins, "the scoring kernel fills the first digit's histogram");
constexpr int kSelPer = 16;          /* consecutive keys per lane, loaded before any is used */
constexpr int kSortMax = 8192;       /* largest top, and keys a ranking block holds in LDS at a time */
constexpr int kSelCap = 2 * kSortMax;   /* most keys written out and ranked */

/* 2^20 scores, 4,096 wanted: 27 us with the clearing (six 11-bit passes handed
 * from block to block, a compaction and a one-block bitonic sort: 125 us).
 * The select takes two 12-bit digits: the first histogram comes out of the
 * scoring kernel, the second out of one pass over the scores; then every key
 * at or above the 24-bit threshold is written out and ranked by counting.
 * Those are the `top` and the few others that share the threshold's 24 bits.
 * Only when so many keys share them that the written set would pass kSelCap
 * (scores equal to 2^-15: a network with dead units, graphs of few distinct
 * degrees) are further digits taken, each a pass of all blocks again: the
 * score's last 8 bits (in the compaction's place), then the place in the pool,
 * coarse and, past 2^25 pairs, fine.  Their kernels leave at once otherwise.  One
 * block for these digits took 796 us for 2^20 equal scores and, with room for
 * kSortMax keys, ran for any pool when 8,192 were wanted (423 us). */
constexpr int kSelStages = 5;
struct SelState {
    uint32_t count;       /* keys written */
    uint32_t more;        /* the first two digits do not settle the select */
    uint32_t pad[62];
    uint32_t hist[kSelStages][kSelBins];
};

/* Digit of a key at a stage; sh: the pool has at most 2^(sh + 12) pairs.  A
 * smaller place is a larger digit, as in the key. */
template <int STAGE>
__device__ __forceinline__ uint32_t sel_digit(uint64_t key, int sh) {
    const uint32_t u = (uint32_t)(key >> 32), p = 0xFFFFFFFFu - (uint32_t)key;
    if (STAGE == 0) return u >> 20;
    if (STAGE == 1) return (u >> 8) & (kSelBins - 1);
    if (STAGE == 2) return u & 255u;
    if (STAGE == 3) return (kSelBins - 1) - (p >> sh);
    return (kSelBins - 1) - ((p >> (sh - kSelBits)) & (kSelBins - 1));
}

__global__ void __launch_bounds__(256) k_select_init(SelState* st) {
    uint32_t* p = reinterpret_cast<uint32_t*>(st);
    const int words = (int)(sizeof(SelState) / sizeof(uint32_t));
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) p[i] = 0;
}

/* Adds 1 to bin b of the LDS histogram for every lane with `valid`: lanes
 * sharing the first valid lane's bin (the common case: scores crowd into a
 * few bins) add together in one atomic. */
__device__ __forceinline__ void wave_hist_add(uint32_t* h, bool valid, uint32_t b, int lane) {
    const uint64_t act = __ballot(valid);
    if (!act) return;
    const int lead = __ffsll((unsigned long long)act) - 1;
    const uint32_t lb = (uint32_t)__shfl((int)b, lead, BM_WAVE);
    const uint64_t same = __ballot(valid && b == lb);
    if (lane == lead) atomicAdd(&h[lb], (uint32_t)__popcll(same));
    if (valid && b != lb) atomicAdd(&h[b], 1u);
}

/* Digit holding the rank-th largest key (1-based) of a histogram, *rank
 * reduced to the rank inside that digit and *inside its count; all NT threads
 * get the result.  A thread's bins stay in registers, its wave sums them by
 * shuffles, and two barriers cover the waves. */
struct DigitShared {
    uint32_t wave[16];
    uint32_t d, r, in;
};
template <int NT>
__device__ __forceinline__ uint32_t find_digit(const uint32_t* h, uint32_t* rank, uint32_t* inside, DigitShared& S) {
    constexpr int kPer = kSelBins / NT, kWaves = NT / BM_WAVE;
    const int t = threadIdx.x, lane = t & (BM_WAVE - 1), wave = t / BM_WAVE;
    uint32_t c[kPer], mine = 0;
#pragma unroll
    for (int j = 0; j < kPer; j += 4) {
        const uint4 q = *reinterpret_cast<const uint4*>(&h[t * kPer + j]);
        c[j] = q.x;
        c[j + 1] = q.y;
        c[j + 2] = q.z;
        c[j + 3] = q.w;
        mine += q.x + q.y + q.z + q.w;
    }
    uint32_t suffix = mine;   /* keys in this lane's and the higher lanes' bins */
#pragma unroll
    for (int o = 1; o < BM_WAVE; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_down((int)suffix, o, BM_WAVE);
        if (lane + o < BM_WAVE) suffix += y;
    }
    __syncthreads();          /* the previous call's results have been read */
    if (lane == 0) S.wave[wave] = suffix;
    __syncthreads();
    for (int w = wave + 1; w < kWaves; w++) suffix += S.wave[w];
    const uint32_t above = suffix - mine;
    if (above < *rank && *rank <= suffix) {
        uint32_t r = *rank - above;
        int d = -1;
        uint32_t in = 0;
#pragma unroll
        for (int j = kPer - 1; j >= 0; j--)
            if (d < 0) {
                if (r <= c[j]) {
                    d = j;
                    in = c[j];
                } else {
                    r -= c[j];
                }
            }
        S.d = (uint32_t)(t * kPer + d);
        S.r = r;
        S.in = in;
    }
    __syncthreads();
    *rank = S.r;
    *inside = S.in;
    return S.d;
}

/* kSelPer consecutive scores per lane from p0 on (0 past the end). */
__device__ __forceinline__ void load_scores(const float* __restrict__ sc, int64_t p0, int64_t P, float* v) {
    if (p0 + kSelPer <= P) {
#pragma unroll
        for (int j = 0; j < kSelPer; j += 4) {
            const float4 f = *reinterpret_cast<const float4*>(&sc[p0 + j]);
            v[j] = f.x;
            v[j + 1] = f.y;
            v[j + 2] = f.z;
            v[j + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < kSelPer; j++) v[j] = p0 + j < P ? sc[p0 + j] : 0.f;
    }
}

/* Second digit: every block finds the first digit from the finished first
 * histogram itself (16 KB from L2, about 2 us, against a last-block hand-over
 * and its fence in every pass), then histograms the second digit of the keys
 * that share it. */
__global__ void __launch_bounds__(kSelThreads) k_select_second(const float* __restrict__ sc, int64_t P, SelState* st,
                                                               uint32_t top) {
    __shared__ alignas(16) uint32_t h[kSelBins];
    __shared__ DigitShared S;
    const int lane = threadIdx.x & (BM_WAVE - 1);
    for (int i = threadIdx.x; i < kSelBins; i += blockDim.x) h[i] = 0;
    uint32_t r = top, in;
    const uint32_t d0 = find_digit<kSelThreads>(st->hist[0], &r, &in, S);
    /* every lane of a wave runs the same iterations (the ballots need them all) */
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / BM_WAVE) * BM_WAVE * kSelPer;
    for (int64_t w0 = ((int64_t)blockIdx.x * (blockDim.x / BM_WAVE) + threadIdx.x / BM_WAVE) * BM_WAVE * kSelPer;
         w0 < P; w0 += wstride) {
        const int64_t p0 = w0 + (int64_t)lane * kSelPer;
        float v[kSelPer];
        load_scores(sc, p0, P, v);
#pragma unroll
        for (int j = 0; j < kSelPer; j++) {
            const uint32_t u = (uint32_t)(rank_key(v[j], p0 + j) >> 32);
            wave_hist_add(h, p0 + j < P && (u >> 20) == d0, (u >> 8) & (kSelBins - 1), lane);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kSelBins; i += blockDim.x)
        if (h[i]) atomicAdd(&st->hist[1][i], h[i]);
}

/* Keys >= thr appended to out (at most kSelCap) by one block's share of the
 * pool: each wave counts its lanes' keys, the block scans its waves' counts,
 * and one global atomic per block and round reserves the slots. */
__device__ __forceinline__ void append_keys(const float* __restrict__ sc, int64_t P, uint64_t thr, uint32_t* count,
                                            uint64_t* __restrict__ out, uint32_t* wcount, uint32_t* base, int64_t block,
                                            int64_t blocks) {
    const int lane = threadIdx.x & (BM_WAVE - 1), wave = threadIdx.x / BM_WAVE, nw = blockDim.x / BM_WAVE;
    for (int64_t b0 = block * blockDim.x * kSelPer; b0 < P; b0 += blocks * blockDim.x * kSelPer) {
        const int64_t p0 = b0 + ((int64_t)wave * BM_WAVE + lane) * kSelPer;
        float v[kSelPer];
        load_scores(sc, p0, P, v);
        uint32_t inmask = 0;   /* bit j: this lane's key j is in */
#pragma unroll
        for (int j = 0; j < kSelPer; j++)
            if (p0 + j < P && rank_key(v[j], p0 + j) >= thr) inmask |= 1u << j;
        const uint32_t mine = (uint32_t)__popc(inmask);
        uint32_t incl = mine;
#pragma unroll
        for (int o = 1; o < BM_WAVE; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o, BM_WAVE);
            if (lane >= o) incl += y;
        }
        if (lane == BM_WAVE - 1) wcount[wave] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t tot = 0;
            for (int w = 0; w < nw; w++) {
                const uint32_t c = wcount[w];
                wcount[w] = tot;
                tot += c;
            }
            *base = tot ? atomicAdd(count, tot) : 0u;
        }
        __syncthreads();
        uint32_t at = *base + wcount[wave] + incl - mine;
#pragma unroll
        for (int j = 0; j < kSelPer; j++)
            if (inmask & (1u << j)) {
                if (at < (uint32_t)kSelCap) out[at] = rank_key(v[j], p0 + j);
                at++;
            }
        __syncthreads();
    }
}

/* The smallest key of the digits of stages 0 .. STAGES - 1 that hold the top-th
 * key; returns whether the keys from it on fit kSelCap (then the later stages
 * are not needed).  Stages end early once they fit. */
template <int STAGES>
__device__ __forceinline__ bool select_threshold(const SelState* st, uint32_t top, int sh, uint64_t* thr, DigitShared& S) {
    uint32_t r = top, in;
    uint32_t u = find_digit<kSelThreads>(st->hist[0], &r, &in, S) << 20;
    u |= find_digit<kSelThreads>(st->hist[1], &r, &in, S) << 8;
    *thr = (uint64_t)u << 32;
    if ((top - r) + in <= (uint32_t)kSelCap) return true;
    if (STAGES < 3) return false;
    u |= find_digit<kSelThreads>(st->hist[2], &r, &in, S);
    *thr = (uint64_t)u << 32;
    if ((top - r) + in <= (uint32_t)kSelCap) return true;
    if (STAGES < 4) return false;
    /* the last place of the digit's range has the smallest key in it */
    uint64_t place = (uint64_t)(kSelBins - 1 - find_digit<kSelThreads>(st->hist[3], &r, &in, S)) << sh;
    *thr = ((uint64_t)u << 32) | (0xFFFFFFFFull - (place + (1ull << sh) - 1));
    if ((top - r) + in <= (uint32_t)kSelCap) return true;
    if (STAGES < 5) return false;
    const int fine = sh - kSelBits;
    place += (uint64_t)(kSelBins - 1 - find_digit<kSelThreads>(st->hist[4], &r, &in, S)) << fine;
    *thr = ((uint64_t)u << 32) | (0xFFFFFFFFull - (place + (1ull << fine) - 1));
    return true;
}

/* Histogram of a further digit over the keys that share thr's earlier ones. */
template <int STAGE>
__device__ __forceinline__ void digit_pass(const float* __restrict__ sc, int64_t P, SelState* st, uint64_t thr, int sh,
                                           uint32_t* h) {
    constexpr int bins = STAGE == 2 ? 256 : kSelBins;
    for (int i = threadIdx.x; i < bins; i += blockDim.x) h[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & (BM_WAVE - 1);
    /* every lane of a wave runs the same iterations (the ballots need them all) */
    const int64_t wstride = (int64_t)gridDim.x * blockDim.x * kSelPer;
    for (int64_t w0 = ((int64_t)blockIdx.x * (blockDim.x / BM_WAVE) + threadIdx.x / BM_WAVE) * BM_WAVE * kSelPer;
         w0 < P; w0 += wstride) {
        const int64_t p0 = w0 + (int64_t)lane * kSelPer;
        float v[kSelPer];
        load_scores(sc, p0, P, v);
#pragma unroll
        for (int j = 0; j < kSelPer; j++) {
            const uint64_t k = rank_key(v[j], p0 + j);
            bool same = p0 + j < P;
            if (STAGE == 2) same = same && (k >> 40) == (thr >> 40);
            if (STAGE > 2) same = same && (k >> 32) == (thr >> 32);
            if (STAGE > 3) same = same && sel_digit<3>(k, sh) == sel_digit<3>(thr, sh);
            wave_hist_add(h, same, sel_digit<STAGE>(k, sh), lane);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < bins; i += blockDim.x)
        if (h[i]) atomicAdd(&st->hist[STAGE][i], h[i]);
}

/* The keys, where two digits settle the select; else the third digit. */
__global__ void __launch_bounds__(kSelThreads) k_select_compact(const float* __restrict__ sc, int64_t P, SelState* st,
                                                                uint64_t* __restrict__ out, uint32_t top) {
    __shared__ uint32_t h[256];
    __shared__ DigitShared S;
    __shared__ uint32_t wcount[kSelThreads / BM_WAVE];
    __shared__ uint32_t base;
    uint64_t thr;
    if (select_threshold<2>(st, top, 0, &thr, S)) {
        append_keys(sc, P, thr, &st->count, out, wcount, &base, blockIdx.x, gridDim.x);
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) st->more = 1;
    digit_pass<2>(sc, P, st, thr, 0, h);
}

template <int STAGE>
__global__ void __launch_bounds__(kSelThreads) k_select_digit(const float* __restrict__ sc, int64_t P, SelState* st,
                                                              uint32_t top, int sh) {
    __shared__ alignas(16) uint32_t h[kSelBins];
    __shared__ DigitShared S;
    if (!st->more) return;
    uint64_t thr;
    if (select_threshold<STAGE>(st, top, sh, &thr, S)) return;
    digit_pass<STAGE>(sc, P, st, thr, sh, h);
}

__global__ void __launch_bounds__(kSelThreads) k_select_rest(const float* __restrict__ sc, int64_t P, SelState* st,
                                                             uint64_t* __restrict__ out, uint32_t top, int sh) {
    __shared__ DigitShared S;
    __shared__ uint32_t wcount[kSelThreads / BM_WAVE];
    __shared__ uint32_t base;
    if (!st->more) return;
    uint64_t thr;
    (void)select_threshold<kSelStages>(st, top, sh, &thr, S);
    append_keys(sc, P, thr, &st->count, out, wcount, &base, blockIdx.x, gridDim.x);
}

/* The written keys ranked by counting: a key's place in descending order is
 * the number of larger ones (keys are distinct).  Every block goes through all
 * keys, kSortMax in LDS at a time, and ranks kRankKeys of them, 16 lanes per
 * key counting a sixteenth each; the `top` first places get their stream
 * pairs. */
constexpr int kRankLanes = 16, kRankKeys = kSelThreads / kRankLanes;

__global__ void __launch_bounds__(kSelThreads) k_select_rank(const uint64_t* __restrict__ keys, const SelState* st,
                                                             uint32_t top, uint64_t seed, int32_t n,
                                                             int2* __restrict__ out) {
    extern __shared__ ulonglong2 sk[];
    const uint32_t cnt = st->count < (uint32_t)kSelCap ? st->count : (uint32_t)kSelCap;
    if ((uint32_t)blockIdx.x * kRankKeys >= cnt) return;
    const uint32_t i = blockIdx.x * kRankKeys + threadIdx.x / kRankLanes, part = threadIdx.x % kRankLanes;
    const uint64_t me = i < cnt ? keys[i] : 0ull;
    uint32_t rank = 0;
    for (uint32_t b = 0; b < cnt; b += (uint32_t)kSortMax) {
        const uint64_t* from = keys + b;
        const uint32_t left = cnt - b < (uint32_t)kSortMax ? cnt - b : (uint32_t)kSortMax;
        /* every lane counts the same whole number of 16-byte words; key 0 is below every key */
        const uint32_t words = (left + 2 * kRankLanes - 1) / (2 * kRankLanes) * kRankLanes;
        if (b) __syncthreads();   /* the keys before have been read */
        for (uint32_t q = threadIdx.x; q < words; q += blockDim.x) {
            ulonglong2 x;
            x.x = 2 * q < left ? from[2 * q] : 0ull;
            x.y = 2 * q + 1 < left ? from[2 * q + 1] : 0ull;
            sk[q] = x;
        }
        __syncthreads();
#pragma unroll 8
        for (uint32_t q = part; q < words; q += kRankLanes) {
            const ulonglong2 x = sk[q];
            rank += (x.x > me ? 1u : 0u) + (x.y > me ? 1u : 0u);
        }
    }
#pragma unroll
    for (int o = 1; o < kRankLanes; o <<= 1) rank += (uint32_t)__shfl_xor((int)rank, o, BM_WAVE);
    if (part == 0 && i < cnt && rank < top) {
        const uint32_t p = 0xFFFFFFFFu - (uint32_t)me;
        int32_t u, v;
        bm_uniform_pair(seed, (uint64_t)p, n, &u, &v);
        out[rank] = make_int2(u, v);
    }
}

int grid_of(int64_t work, int threads, int64_t cap = 65536) {
    int64_t b = (work + threads - 1) / threads;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (int)b;
}

MlpDev mlpdev(const BmMlpDev& d) {
    MlpDev M;
    M.W1f = reinterpret_cast<const v4s*>(d.W1f);
    M.W2f = reinterpret_cast<const v8s*>(d.W2f);
    M.W2Tf = reinterpret_cast<const v8s*>(d.W2Tf);
    M.b1 = d.params + kOffB1;
    M.b2 = d.params + kOffB2;
    M.w3 = d.params + kOffW3;
    M.b3 = d.params + kOffB3;
    return M;
}

}  // namespace

int32_t bm_mlp_param_count(void) { return kParams; }

hipError_t bm_launch_vertex_features(const BmDevGraph& g, const int4* chunks, int64_t nchunks, void* acc, float* vf,
                                     int32_t num_cus, hipStream_t s) {
    const hipError_t e = bm_launch_feature_sums(g, chunks, nchunks, static_cast<int64_t*>(acc), num_cus, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_feature_finish, dim3(grid_of((int64_t)g.n + 1, 256)), dim3(256), 0, s, g,
                       static_cast<longlong4*>(acc), reinterpret_cast<float4*>(vf));
    return hipGetLastError();
}

hipError_t bm_launch_mlp_pack(const BmMlpDev& d, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(grid_of(kParams, 256)), dim3(256), 0, s, d.params, static_cast<short*>(d.W1f),
                       static_cast<short*>(d.W2f), static_cast<short*>(d.W2Tf));
    return hipGetLastError();
}

template <bool HIST>
static hipError_t launch_forward(const BmMlpDev& d, const float* vf, const int2* list, uint64_t seed, int32_t n,
                                 int64_t k, float* score, uint32_t* hist, int32_t num_cus, hipStream_t s) {
    PairSrc ps{list, seed, n};
    int64_t blocks = (k + 16 * kFwdTiles - 1) / (16 * kFwdTiles);
    const int64_t cap = num_cus > 0 ? num_cus : 256;
    if (blocks > cap) blocks = cap;
    const size_t lds = sizeof(ScoreShared) + (HIST ? kHistBins * sizeof(uint32_t) : 0);
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_forward<HIST>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mlp_forward<HIST>, dim3((unsigned)blocks), dim3(kScoreThreads), lds, s,
                       reinterpret_cast<const float4*>(vf), ps, k, mlpdev(d), score, hist);
    return hipGetLastError();
}

hipError_t bm_launch_mlp_forward(const BmMlpDev& d, const float* vf, const int2* list, uint64_t seed, int32_t n,
                                 int64_t k, float* score, int32_t num_cus, hipStream_t s) {
    if (k <= 0) return hipSuccess;
    return launch_forward<false>(d, vf, list, seed, n, k, score, nullptr, num_cus, s);
}

/* Scratch of one batch: the four activation arrays, then the partials.  The
 * rows are padded by 64 entries, so that the 16 rows a fragment reads do not
 * start a multiple of 4 KB apart. */
constexpr int kMaxSlices = 32, kMaxTrainBlocks = 1024;
static int64_t train_stride(int64_t k) { return (k + 31) / 32 * 32 + 64; }

size_t bm_mlp_train_bytes(int64_t k) {
    return (size_t)train_stride(k) * (kF + 3 * kH) * sizeof(short) +
           ((size_t)kMaxSlices * kWParams + (size_t)kBParams * kMaxTrainBlocks) * sizeof(float);
}

static int train_blocks(int64_t B, int32_t num_cus) {
    int64_t blocks = (B / 16 + kTrainWaves - 1) / kTrainWaves;
    int64_t cap = num_cus > 0 ? num_cus : 256;
    if (cap > kMaxTrainBlocks) cap = kMaxTrainBlocks;
    return (int)(blocks < cap ? blocks : cap);
}

/* a wave takes at least four 32-pair steps; 32 slices give 320 blocks */
static int train_slices(int64_t B) {
    const int64_t s = B / 32 / 16;
    return (int)(s < 1 ? 1 : (s > kMaxSlices ? kMaxSlices : s));
}

static GradParts grad_parts(void* act, int64_t k, int32_t num_cus) {
    const int64_t B = (k + 31) / 32 * 32;
    GradParts P;
    P.w = reinterpret_cast<const float*>(reinterpret_cast<const short*>(act) + (size_t)train_stride(k) * (kF + 3 * kH));
    P.b = P.w + (size_t)kMaxSlices * kWParams;
    P.slices = train_slices(B);
    P.blocks = train_blocks(B, num_cus);
    return P;
}

hipError_t bm_launch_mlp_gradient(const BmMlpDev& d, const float* vf, const int2* list, uint64_t seed, int32_t n,
                                  int64_t k, const float* target, const int64_t* delta, void* act, int32_t num_cus,
                                  hipStream_t s) {
    if (k <= 0) return hipSuccess;
    const GradParts P = grad_parts(act, k, num_cus);
    TrainBuf T;
    T.B = (k + 31) / 32 * 32;
    T.ld = train_stride(k);
    T.XT = reinterpret_cast<short*>(act);
    T.H1T = T.XT + (size_t)kF * T.ld;
    T.G1T = T.H1T + (size_t)kH * T.ld;
    T.G2T = T.G1T + (size_t)kH * T.ld;
    T.wpart = const_cast<float*>(P.w);
    T.bpart = const_cast<float*>(P.b);
    T.target = target;
    T.delta = delta;
    PairSrc ps{list, seed, n};
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_train_act, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)sizeof(TrainShared));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mlp_train_act, dim3((unsigned)P.blocks), dim3(kTrainThreads), sizeof(TrainShared), s,
                       reinterpret_cast<const float4*>(vf), ps, k, mlpdev(d), T);
    hipLaunchKernelGGL(k_mlp_wgrad, dim3((unsigned)(kWgItems * P.slices)), dim3(256), 0, s, T, P.slices);
    return hipGetLastError();
}

hipError_t bm_launch_mlp_reduce(const BmMlpDev& d, void* act, int64_t k, float* loss, int32_t num_cus, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_reduce, dim3(kGradWBlocks + kGradBBlocks), dim3(kGradThreads), 0, s,
                       grad_parts(act, k, num_cus), d.grad, loss);
    return hipGetLastError();
}

hipError_t bm_launch_mlp_adam(const BmMlpDev& d, float lr, int64_t step, void* act, int64_t k, float* loss,
                              int32_t num_cus, hipStream_t s) {
    const float b1c = 1.f - powf(0.9f, (float)step), b2c = 1.f - powf(0.999f, (float)step);
    hipLaunchKernelGGL(k_mlp_adam, dim3(kGradWBlocks + kGradBBlocks), dim3(kGradThreads), 0, s,
                       grad_parts(act, k, num_cus), d.params, d.adam_m, d.adam_v, lr, b1c, b2c,
                       static_cast<short*>(d.W1f), static_cast<short*>(d.W2f), static_cast<short*>(d.W2Tf), loss);
    return hipGetLastError();
}

size_t bm_mlp_select_bytes(int64_t pool) {
    return (size_t)pool * sizeof(float) + 512 + sizeof(SelState) + kSelCap * sizeof(uint64_t);
}

int64_t bm_mlp_select_max_top(void) { return kSortMax; }

/* Scores of the pool's pairs with the first digit's histogram, the second
 * digit, the keys at or above the threshold and their ranking; scratch holds
 * the scores, the select state and the selected keys
 * (bm_mlp_select_bytes(pool)), and the state is cleared by k_select_init, so
 * the call allocates nothing and needs no memset. */
hipError_t bm_launch_mlp_rank_select(const BmMlpDev& d, const float* vf, uint64_t seed, int32_t n, int64_t pool,
                                     int64_t top, void* scratch, size_t scratch_bytes, int2* out, int32_t num_cus,
                                     hipStream_t s) {
    if (pool <= 0 || top <= 0) return hipSuccess;
    if (top > kSortMax || top > pool || pool >= (1LL << 32) || scratch_bytes < bm_mlp_select_bytes(pool))
        return hipErrorInvalidValue;
    float* sc = static_cast<float*>(scratch);
    char* q = reinterpret_cast<char*>(sc + pool);
    q += (256 - (reinterpret_cast<uintptr_t>(q) & 255)) & 255;
    SelState* st = reinterpret_cast<SelState*>(q);
    uint64_t* keys = reinterpret_cast<uint64_t*>(st + 1);
    hipLaunchKernelGGL(k_select_init, dim3(16), dim3(256), 0, s, st);
    hipError_t e = launch_forward<true>(d, vf, nullptr, seed, n, pool, sc, st->hist[0], num_cus, s);
    if (e != hipSuccess) return e;
    const int blocks = grid_of(pool, kSelThreads * kSelPer, (int64_t)(num_cus > 0 ? num_cus : 256) * 4);
    hipLaunchKernelGGL(k_select_second, dim3(blocks), dim3(kSelThreads), 0, s, sc, pool, st, (uint32_t)top);
    hipLaunchKernelGGL(k_select_compact, dim3(blocks), dim3(kSelThreads), 0, s, sc, pool, st, keys, (uint32_t)top);
    if (pool > kSelCap) {   /* else every key fits */
        int sh = 0;
        while (((int64_t)kSelBins << sh) < pool) sh++;
        const int rest = grid_of(pool, kSelThreads * kSelPer, num_cus > 0 ? num_cus : 256);
        hipLaunchKernelGGL(k_select_digit<3>, dim3(rest), dim3(kSelThreads), 0, s, sc, pool, st, (uint32_t)top, sh);
        /* a coarse digit's 2^sh places and the keys above it fit kSelCap */
        if (sh > kSelBits + 1)
            hipLaunchKernelGGL(k_select_digit<4>, dim3(rest), dim3(kSelThreads), 0, s, sc, pool, st, (uint32_t)top, sh);
        hipLaunchKernelGGL(k_select_rest, dim3(rest), dim3(kSelThreads), 0, s, sc, pool, st, keys, (uint32_t)top, sh);
    }
    const size_t lds = kSortMax * sizeof(uint64_t);
    e = hipFuncSetAttribute((const void*)k_select_rank, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_select_rank, dim3(kSelCap / kRankKeys), dim3(kSelThreads), lds, s, keys, st, (uint32_t)top,
                       seed, n, out);
    return hipGetLastError();
}

size_t bm_mlp_rank_scratch(int64_t pool) {
    size_t temp = 0;
    (void)hipcub::DeviceRadixSort::SortPairsDescending(nullptr, temp, (const float*)nullptr, (float*)nullptr,
                                                       (const int32_t*)nullptr, (int32_t*)nullptr, (int)pool);
    const size_t sort_path = temp + 256 + (size_t)pool * (2 * sizeof(float) + 2 * sizeof(int32_t));
    const size_t select_path = bm_mlp_select_bytes(pool);
    return sort_path > select_path ? sort_path : select_path;
}

hipError_t bm_launch_mlp_rank(const BmMlpDev& d, const float* vf, uint64_t seed, int32_t n, int64_t pool, int64_t top,
                              void* scratch, size_t scratch_bytes, int2* out, int32_t num_cus, hipStream_t s) {
    if (pool <= 0 || top <= 0) return hipSuccess;
    char* p = static_cast<char*>(scratch);
    float* sc = reinterpret_cast<float*>(p);
    float* sc_sorted = sc + pool;
    int32_t* idx = reinterpret_cast<int32_t*>(sc_sorted + pool);
    int32_t* idx_sorted = idx + pool;
    char* temp = reinterpret_cast<char*>(idx_sorted + pool);
    temp += (256 - (reinterpret_cast<uintptr_t>(temp) & 255)) & 255;
    size_t temp_bytes = scratch_bytes - (size_t)(temp - p);
    /* select of the top keys, then their ranking */
    if (top <= kSortMax && pool < (1LL << 32))
        return bm_launch_mlp_rank_select(d, vf, seed, n, pool, top, scratch, scratch_bytes, out, num_cus, s);
    hipError_t e = bm_launch_mlp_forward(d, vf, nullptr, seed, n, pool, sc, num_cus, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_iota, dim3(grid_of(pool, 256)), dim3(256), 0, s, idx, pool);
    e = hipcub::DeviceRadixSort::SortPairsDescending(temp, temp_bytes, sc, sc_sorted, idx, idx_sorted, (int)pool, 0,
                                                     32, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_gather_stream_pairs, dim3(grid_of(top, 256)), dim3(256), 0, s, seed, n, idx_sorted, top, out);
    return hipGetLastError();
}
