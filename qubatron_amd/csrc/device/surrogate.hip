/*
 * surrogate.hip - the learned shadow-visibility surrogate (no reference
 * counterpart: the reference traces every shadow ray,
 * src/qubatron/shaders/octree_fsh.c:426-434).
 *
 *   training   two kernels per minibatch: features, forward (bias + ReLU +
 *              bf16 between layers), loss and output gradient, backward
 *              through the masked transposed weights and the weight and bias
 *              gradients, 64 samples per block on the matrix cores -> sum of
 *              the per-block partial gradients, Adam on fp32 master weights,
 *              bf16 repack
 *   inference  one fused kernel: weights in LDS, 16 queries per wave, the
 *              four layers chained in registers (mlp.hpp)
 *   render     the decision pass of QBT_RENDER_SURROGATE: predicted bits
 *              outside the band, the rest appended to per-light lists that
 *              the exact shadow kernel traces
 *   collect    training samples from exact renders (QBT_RENDER_COLLECT)
 *
 * Activations are feature-major ([feature][sample], bf16) so that every
 * layer is C = W H with the batch as the N dimension.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <math.h>

#include <rocprim/rocprim.hpp>

#include "mlp.hpp"
#include "pixel.hpp"
#include "qbt.h"
#include "qbt_internal.hpp"
#include "trace.hpp"

#pragma clang fp contract(off)

using namespace qbt;

#define HIPCHK(x) QBT_HIPCHK(x)

static_assert(kMlpParams == QBT_MLP_PARAMS, "parameter count");
static_assert(kMlpIn == QBT_MLP_INPUTS, "input count");

/* training sample: hit position, normal, light position, label (1 = lit) */
struct RawSample {
    float isp[3], nrm[3], light[3], label;
};
static_assert(sizeof(RawSample) == 40, "sample record");

/* a block's partial gradients (fp32): the 16 x 16 tiles of dW1, dW2, dW3 as
 * matrix-core fragments (element 256 t + 4 lane + e), dW4, the biases */
constexpr int kG2 = 12 * 256, kG3 = kG2 + 16 * 256, kG4 = kG3 + 16 * 256, kGB1 = kG4 + 64, kGB2 = kGB1 + 64,
              kGB3 = kGB2 + 64, kGB4 = kGB3 + 64, kGradN = kGB4 + 64; /* padded to 64 */
/* packed weights of the training kernel, after the inference kernels' (kP*): W2 and W3 transposed */
constexpr int kPT2 = kPackN, kPT3 = kPT2 + 64 * 64, kPackAll = kPT3 + 64 * 64;
/* biases in LDS for the fused kernels */
constexpr int kLB1 = 0, kLB2 = 64, kLB3 = 128, kLB4 = 192, kLBN = 196;

struct MlpState {
    DevBuf   params, m, v, packed, ctr; /* ctr: collected, lit (u64) */
    DevBuf   samples, perm, keys, vals, sort_tmp;
    DevBuf   X, gpart, lossbuf, io_x, io_p, io_y, io_a, io_c, flat; /* gpart: k_mlp_train's partial gradients */
    size_t   cap = 0;
    uint32_t stride = 1, phase = 0;
    int      t     = 0; /* Adam steps taken */
    float    band_lo = 0.1f, band_hi = 0.9f;
    bool     ready   = false; /* parameters initialised */
    uint64_t epoch   = 0;
    size_t   pos     = 0, perm_n = 0; /* next batch in the permutation of perm_n samples */
};

namespace {

inline unsigned nblk(size_t n, unsigned bs = 256) { return (unsigned) ((n + bs - 1) / bs); }

__global__ void k_fill_f32(float* p, size_t n, float v)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill_u64(unsigned long long* p, int n)
{
    int i = threadIdx.x;
    if (i < n) p[i] = 0ull;
}

/* splitmix64 finaliser of a counter */
__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

/* He-uniform weights (bound sqrt(6 / fan_in)), zero biases */
__global__ void k_mlp_init(float* P, uint64_t seed)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kMlpParams) return;
    float a = 0.0f;
    if (i < kB1) a = sqrtf(6.0f / 42.0f);
    else if ((i >= kW2 && i < kB2) || (i >= kW3 && i < kB3) || (i >= kW4 && i < kB4)) a = sqrtf(6.0f / 64.0f);
    float u = (float) (mix64(seed * 0x9E3779B97F4A7C15ull + (uint64_t) i) >> 40) * (1.0f / 16777216.0f);
    P[i]    = a > 0.0f ? (2.0f * u - 1.0f) * a : 0.0f;
}

/* fp32 parameters -> padded bf16 weight matrices, W2 and W3 also transposed */
__global__ void k_mlp_pack(const float* __restrict__ P, uint16_t* __restrict__ W)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kPackAll) return;
    float v = 0.0f;
    if (i >= kPackN) {
        const int k = (i - kPackN) % (64 * 64), o = k % 64, c = k / 64;
        W[i]        = f2bf(P[(i < kPT3 ? kW2 : kW3) + o * 64 + c]);
        return;
    }
    if (i < kP2) {
        int o = i / 48, c = i % 48;
        v     = c < kMlpIn ? P[kW1 + o * kMlpIn + c] : 0.0f;
    } else if (i < kP3) {
        v = P[kW2 + (i - kP2)];
    } else if (i < kP4) {
        v = P[kW3 + (i - kP3)];
    } else {
        int r = (i - kP4) / 64, c = (i - kP4) % 64;
        v     = r == 0 ? P[kW4 + c] : 0.0f;
    }
    W[i] = f2bf(v);
}

/* ------------------------------------------------------------------------ */
/* fused training forward and backward                                      */
/* ------------------------------------------------------------------------ */

constexpr int kChunk = 64; /* samples per chunk: four fragment groups of 16 */
constexpr int kRow   = 68; /* elements of a row of 64 in LDS (padded: rows start 2 banks apart) */

__device__ __forceinline__ bf16x4 lds4(const uint16_t* a) { return *reinterpret_cast<const bf16x4*>(a); }
__device__ __forceinline__ void   lds4(uint16_t* a, bf16x4 v) { *reinterpret_cast<bf16x4*>(a) = v; }

__device__ __forceinline__ bf16x4 relu_pack(f32x4 acc, const float* __restrict__ b)
{
    return pack4(acc[0] + b[0] > 0.0f ? acc[0] + b[0] : 0.0f, acc[1] + b[1] > 0.0f ? acc[1] + b[1] : 0.0f,
                 acc[2] + b[2] > 0.0f ? acc[2] + b[2] : 0.0f, acc[3] + b[3] > 0.0f ? acc[3] + b[3] : 0.0f);
}

/* dZ = (W^T dZ_next) where the layer's ReLU output is positive, bf16 */
__device__ __forceinline__ bf16x4 mask_pack(f32x4 acc, bf16x4 h)
{
    return pack4(h[0] > 0 ? acc[0] : 0.0f, h[1] > 0 ? acc[1] : 0.0f, h[2] > 0 ? acc[2] : 0.0f,
                 h[3] > 0 ? acc[3] : 0.0f);
}

/* samples of a minibatch: the store's records perm[off ..] (S not null), or
 * the feature matrix X[48][B] with labels Y */
struct TrainBatch {
    const RawSample* S;
    const uint32_t*  perm;
    size_t           off;
    float            bx, by, bz, bw;
    const uint16_t*  X;
    const float*     Y;
    int              B, n; /* columns, of which valid */
};

/* Forward and backward of a minibatch, four waves per block; block b takes
 * the 64-sample chunks b, b + gridDim.x, ... Wave w computes output features
 * 16 w .. 16 w + 15 of every layer for the chunk's four groups of 16 samples
 * (its rows of W and W^T are 24 fragments, held in registers), and the same
 * rows of the weight gradients, whose fragments stay in registers over the
 * chunks. Rounding points as the oracle's: bias, ReLU and bf16 between
 * layers, output gradient bf16((p - y) / n). Activations and gradients pass
 * between the waves through LDS twice: a sample per row (B fragments of the
 * next layer; two buffers in turn) and a feature per row (both operands of a
 * weight gradient, the samples as K). The block's gradients go to its row of
 * gp (no atomics; k_mlp_step sums the rows). loss: the summed BCE is added,
 * if not null (a training run needs that of its last step only: the double
 * logarithms are a tenth of the kernel).
 *
 * What bounds it: latency, 64 blocks at batch 4096, nine barriers. 12.6 us
 * a step's launch, features included, against 28 + 8 + 4 us (features, loss
 * reset) with every wave taking 16 samples through all features: that loaded
 * 84 weight fragments per wave, two bytes at a time for the transposed ones,
 * and summed the biases from LDS with all lanes on one bank. */
template <bool STORE>
__global__ void __launch_bounds__(256) k_mlp_train(const uint16_t* __restrict__ W, const float* __restrict__ P,
                                                   TrainBatch T, float* __restrict__ gp, double* __restrict__ loss)
{
    __shared__ __align__(16) uint16_t S0[kChunk * kRow], S1[kChunk * kRow]; /* [sample][feature], in turn */
    __shared__ __align__(16) uint16_t Xf[kMlpInPad * kRow], H1[64 * kRow], H2[64 * kRow]; /* [feature][sample] */
    __shared__ __align__(16) uint16_t F3[64 * kRow]; /* H3, later dZ2 */
    __shared__ __align__(16) uint16_t F4[64 * kRow]; /* dZ3, later dZ1 */
    __shared__ __align__(16) uint16_t dz[kChunk];
    __shared__ float                  yl[kChunk];
    const int    tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int    row = 16 * w + 4 * g; /* this lane's four output features */
    const bf16x4 zero4 = {0, 0, 0, 0}, ones = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
    const f32x4  zacc = {0.f, 0.f, 0.f, 0.f};
    bf16x4       w1[3], w2[4], w3[4], w4[4], t2[4], t3[4], t4 = zero4;
    for (int kb = 0; kb < 3; kb++) w1[kb] = *reinterpret_cast<const bf16x4*>(W + kP1 + (16 * w + r) * 48 + 16 * kb + 4 * g);
    for (int kb = 0; kb < 4; kb++) {
        const int at = (16 * w + r) * 64 + 16 * kb + 4 * g;
        w2[kb] = *reinterpret_cast<const bf16x4*>(W + kP2 + at);
        w3[kb] = *reinterpret_cast<const bf16x4*>(W + kP3 + at);
        t2[kb] = *reinterpret_cast<const bf16x4*>(W + kPT2 + at);
        t3[kb] = *reinterpret_cast<const bf16x4*>(W + kPT3 + at);
        w4[kb] = *reinterpret_cast<const bf16x4*>(W + kP4 + r * 64 + 16 * kb + 4 * g); /* the output row block */
    }
    t4[0] = g == 0 ? (short) W[kP4 + 16 * w + r] : (short) 0; /* W4^T: one column that is not zero */
    float b1[4], b2[4], b3[4];
    for (int e = 0; e < 4; e++) b1[e] = P[kB1 + row + e], b2[e] = P[kB2 + row + e], b3[e] = P[kB3 + row + e];
    const float b4 = P[kB4];
    f32x4       g1[3], g2[4], g3[4], g4 = zacc, gb1 = zacc, gb2 = zacc, gb3 = zacc; /* gradients of this wave's rows */
    for (int t = 0; t < 3; t++) g1[t] = zacc;
    for (int t = 0; t < 4; t++) g2[t] = g3[t] = zacc;
    float     gb4    = 0.0f;
    double    lsum   = 0.0;
    const int chunks = (T.B + kChunk - 1) / kChunk;
    /* one layer: rows of the wave, four sample groups: input fragments from
     * `in` ([sample][feature]), results to `out` and to feat ([feature][sample]) */
    auto put = [&](uint16_t* out, uint16_t* feat, int j, bf16x4 v) {
        if (out) lds4(out + (16 * j + r) * kRow + row, v);
        for (int e = 0; e < 4; e++) feat[(row + e) * kRow + 16 * j + r] = (uint16_t) v[e];
    };
    auto dot = [&](const bf16x4* a, int kbs, const uint16_t* in, int j) {
        f32x4 acc = zacc;
        for (int kb = 0; kb < kbs; kb++) acc = mfma16(a[kb], lds4(in + (16 * j + r) * kRow + 16 * kb + 4 * g), acc);
        return acc;
    };
    /* rows of a weight gradient: A = the wave's rows of dZ, B = rows of H, K = samples; and the bias's */
    auto grad = [&](const uint16_t* dZ, const uint16_t* H, int tiles, f32x4* acc, f32x4& gb) {
        for (int j = 0; j < kChunk / 16; j++) {
            const bf16x4 a = lds4(dZ + (16 * w + r) * kRow + 16 * j + 4 * g);
            for (int t = 0; t < tiles; t++) acc[t] = mfma16(a, lds4(H + (16 * t + r) * kRow + 16 * j + 4 * g), acc[t]);
            gb = mfma16(a, ones, gb);
        }
    };
    for (int c = blockIdx.x; c < chunks; c += gridDim.x) {
        const int base = c * kChunk, s = base + lane;
        /* features 12 w .. 12 w + 11 of sample `lane` */
        if (STORE) {
            float u[3] = {0.f, 0.f, 0.f}, nn[3] = {0.f, 0.f, 0.f}, lu[3] = {0.f, 0.f, 0.f};
            if (s < T.B) {
                const RawSample q = T.S[T.perm[T.off + (size_t) s]];
                mlp_scale(q.isp, T.bx, T.by, T.bz, T.bw, u);
                mlp_scale(q.light, T.bx, T.by, T.bz, T.bw, lu);
                nn[0] = q.nrm[0], nn[1] = q.nrm[1], nn[2] = q.nrm[2];
                if (w == 0) yl[lane] = q.label;
            }
            for (int p = 0; p < 6; p++) {
                const int f = 12 * w + 2 * p; /* uniform over the wave */
                float     a, b;
                if (f < 36) band_sincos(f / 6, pick3(u, (f % 6) >> 1), &a, &b);
                else a = mlp_feature(f, u, nn, lu), b = mlp_feature(f + 1, u, nn, lu);
                const uint16_t ab = s < T.B ? f2bf(a) : (uint16_t) 0, bb = s < T.B ? f2bf(b) : (uint16_t) 0;
                S0[lane * kRow + f]       = ab;
                S0[lane * kRow + f + 1]   = bb;
                Xf[f * kRow + lane]       = ab;
                Xf[(f + 1) * kRow + lane] = bb;
            }
        } else {
            for (int f = 12 * w; f < 12 * w + 12; f++) {
                const uint16_t v     = s < T.B ? T.X[(size_t) f * T.B + s] : (uint16_t) 0;
                S0[lane * kRow + f]  = v;
                Xf[f * kRow + lane]  = v;
            }
            if (w == 0) yl[lane] = s < T.B ? T.Y[s] : 0.0f;
        }
        __syncthreads();
        bf16x4 h1[4], h2[4], h3[4];
        for (int j = 0; j < 4; j++) put(S1, H1, j, h1[j] = relu_pack(dot(w1, 3, S0, j), b1));
        __syncthreads();
        for (int j = 0; j < 4; j++) put(S0, H2, j, h2[j] = relu_pack(dot(w2, 4, S1, j), b2));
        __syncthreads();
        for (int j = 0; j < 4; j++) put(S1, F3, j, h3[j] = relu_pack(dot(w3, 4, S0, j), b3));
        __syncthreads();
        { /* loss and output gradient of sample group w: row 0 of the output tile, lanes 0..15 */
            const f32x4 lg = dot(w4, 4, S1, w);
            const int   q  = base + 16 * w + r;
            float       d  = 0.0f;
            if (g == 0 && q < T.n) {
                const float p = 1.0f / (1.0f + expf(-(lg[0] + b4)));
                const float y = yl[16 * w + r];
                if (loss) {
                    const float pc = fminf(fmaxf(p, 1e-7f), 1.0f - 1e-7f);
                    lsum += y > 0.5f ? -log((double) pc) : -log(1.0 - (double) pc);
                }
                d = (p - y) / (float) T.n;
            }
            if (g == 0) dz[16 * w + r] = f2bf(d);
        }
        __syncthreads();
        for (int j = 0; j < 4; j++) {
            bf16x4 d4 = zero4; /* row 0 of dZ4; rows 1..15 zero */
            d4[0]     = g == 0 ? (short) dz[16 * j + r] : (short) 0;
            put(S0, F4, j, mask_pack(mfma16(t4, d4, zacc), h3[j]));
            const bf16x4 a4 = r == 0 ? lds4(dz + 16 * j + 4 * g) : zero4; /* dW4: columns 16 w .. of its row 0 */
            g4 = mfma16(a4, lds4(F3 + (16 * w + r) * kRow + 16 * j + 4 * g), g4);
        }
        if (w == 0) gb4 += bf2f(dz[lane]);
        __syncthreads();
        for (int j = 0; j < 4; j++) put(S1, F3, j, mask_pack(dot(t3, 4, S0, j), h2[j]));
        grad(F4, H2, 4, g3, gb3);
        __syncthreads();
        for (int j = 0; j < 4; j++) put(nullptr, F4, j, mask_pack(dot(t2, 4, S1, j), h1[j]));
        grad(F3, H1, 4, g2, gb2);
        __syncthreads();
        grad(F4, Xf, 3, g1, gb1);
        __syncthreads(); /* the next chunk overwrites the LDS arrays */
    }
    float* const out = gp + (size_t) blockIdx.x * kGradN;
    for (int t = 0; t < 3; t++) *reinterpret_cast<f32x4*>(out + 256 * (3 * w + t) + 4 * lane) = g1[t];
    for (int t = 0; t < 4; t++) *reinterpret_cast<f32x4*>(out + kG2 + 256 * (4 * w + t) + 4 * lane) = g2[t];
    for (int t = 0; t < 4; t++) *reinterpret_cast<f32x4*>(out + kG3 + 256 * (4 * w + t) + 4 * lane) = g3[t];
    if (g == 0) out[kG4 + 16 * w + r] = g4[0];
    if (r == 0) { /* every column of these is the same sum */
        *reinterpret_cast<f32x4*>(out + kGB1 + row) = gb1;
        *reinterpret_cast<f32x4*>(out + kGB2 + row) = gb2;
        *reinterpret_cast<f32x4*>(out + kGB3 + row) = gb3;
    }
    if (w == 0) {
        for (int o = 32; o > 0; o >>= 1) gb4 += __shfl_xor(gb4, o, 64);
        if (lane == 0) out[kGB4] = gb4;
    }
    if (loss) {
        for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
        if (lane == 0 && lsum != 0.0) atomicAdd(loss, lsum);
    }
}

/* partial-gradient element -> flat parameter index (-1: padding), and where
 * the weight's bf16 copies sit (pk; pt, W2 and W3 only) */
__device__ __forceinline__ int grad_param(int i, int& pk, int& pt)
{
    pk = pt = -1;
    if (i < kG4) {
        const int t = i < kG2 ? i / 256 : (i < kG3 ? i - kG2 : i - kG3) / 256, nts = i < kG2 ? 3 : 4;
        const int lane = (i & 255) >> 2, o = 16 * (t / nts) + 4 * (lane >> 4) + (i & 3), c = 16 * (t % nts) + (lane & 15);
        if (i < kG2) {
            if (c >= kMlpIn) return -1;
            pk = kP1 + o * 48 + c;
            return kW1 + o * kMlpIn + c;
        }
        pk = (i < kG3 ? kP2 : kP3) + o * 64 + c;
        pt = (i < kG3 ? kPT2 : kPT3) + c * 64 + o;
        return (i < kG3 ? kW2 : kW3) + o * 64 + c;
    }
    if (i < kGB1) {
        pk = kP4 + (i - kG4);
        return kW4 + (i - kG4);
    }
    if (i < kGB2) return kB1 + (i - kGB1);
    if (i < kGB3) return kB2 + (i - kGB2);
    if (i < kGB4) return kB3 + (i - kGB3);
    return i == kGB4 ? kB4 : -1;
}

struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
};

/* The sum of the blocks' partial gradients (64 elements per block, four row
 * groups), then either the gradient in flat order (grads not null), or one
 * Adam step (Kingma & Ba 2015, bias-corrected moments, fp32 master weights)
 * and the weights' new bf16 copies. 3.9 us for 64 rows, against 16 + 4.6 +
 * 4.5 for a sum by one thread per element, Adam and repack as launches. */
__global__ void __launch_bounds__(256) k_mlp_step(const float* __restrict__ gp, int rows, float* __restrict__ grads,
                                                  float* __restrict__ P, float* __restrict__ m, float* __restrict__ v,
                                                  uint16_t* __restrict__ W, AdamArgs A)
{
    __shared__ float part[4][64];
    const int        lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    const int        per = (rows + 3) / 4, lo = w * per, hi = min(rows, lo + per);
    float            acc = 0.0f;
#pragma unroll 8
    for (int b = lo; b < hi; b++) acc += gp[(size_t) b * kGradN + i];
    part[w][lane] = acc;
    __syncthreads();
    if (w != 0) return;
    int         pk, pt;
    const int   p = grad_param(i, pk, pt);
    const float g = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    if (p < 0) return;
    if (grads) {
        grads[p] = g;
        return;
    }
    const float mn = A.b1 * m[p] + (1.0f - A.b1) * g, vn = A.b2 * v[p] + (1.0f - A.b2) * g * g;
    m[p]           = mn;
    v[p]           = vn;
    const float pn = P[p] - A.lr * (mn / A.c1) / (sqrtf(vn / A.c2) + A.eps);
    P[p]           = pn;
    if (pk >= 0) W[pk] = f2bf(pn);
    if (pt >= 0) W[pt] = f2bf(pn);
}

/* supplied feature rows (n x 42 fp32) -> X; columns n..B-1 zero */
__global__ void k_copy_features(const float* __restrict__ x, int B, int n, uint16_t* __restrict__ X,
                                const float* __restrict__ yin, float* __restrict__ Y)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= B) return;
    for (int f = 0; f < kMlpInPad; f++)
        X[(size_t) f * B + s] = f2bf((s < n && f < kMlpIn) ? x[(size_t) s * kMlpIn + f] : 0.0f);
    if (Y) Y[s] = (s < n && yin) ? yin[s] : 0.0f;
}

/* random sort keys for the sample shuffle */
__global__ void k_perm_keys(uint32_t* keys, uint32_t* vals, size_t n, uint64_t seed)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = (uint32_t) mix64(seed * 0x9E3779B97F4A7C15ull + i);
    vals[i] = (uint32_t) i;
}

/* ------------------------------------------------------------------------ */
/* fused inference                                                          */
/* ------------------------------------------------------------------------ */

struct InferArgs {
    const uint16_t* W; /* packed bf16 weights */
    const float*    P; /* fp32 parameters (the biases are read) */
    float           bx, by, bz, bw;
};

/* the biases in LDS (every lane of a row group reads the same four) */
__device__ __forceinline__ void load_biases_lds(const InferArgs& ia, float* Bs)
{
    for (int i = threadIdx.x; i < kLBN; i += blockDim.x) {
        float b = 0.0f;
        if (i < 64) b = ia.P[kB1 + i];
        else if (i < 128) b = ia.P[kB2 + i - 64];
        else if (i < 192) b = ia.P[kB3 + i - 128];
        else if (i == kLB4) b = ia.P[kB4];
        Bs[i] = b;
    }
    __syncthreads();
}

/* All weights as matrix-core A fragments, held in registers for the whole
 * kernel (48 fragments, 96 VGPRs): lane l holds W[16 mt + l % 16][16 kb +
 * 4 (l / 16) + e]. */
struct MlpFrags {
    bf16x4 w1[4][3], w2[4][4], w3[4][4], w4[4];
};

__device__ __forceinline__ void load_frags(const uint16_t* __restrict__ W, int lane, MlpFrags& F)
{
    const int r = lane & 15, g = lane >> 4;
    for (int mt = 0; mt < 4; mt++) {
        for (int kb = 0; kb < 3; kb++)
            F.w1[mt][kb] = *reinterpret_cast<const bf16x4*>(W + kP1 + (16 * mt + r) * 48 + 16 * kb + 4 * g);
        for (int kb = 0; kb < 4; kb++) {
            F.w2[mt][kb] = *reinterpret_cast<const bf16x4*>(W + kP2 + (16 * mt + r) * 64 + 16 * kb + 4 * g);
            F.w3[mt][kb] = *reinterpret_cast<const bf16x4*>(W + kP3 + (16 * mt + r) * 64 + 16 * kb + 4 * g);
        }
    }
    for (int kb = 0; kb < 4; kb++) F.w4[kb] = *reinterpret_cast<const bf16x4*>(W + kP4 + r * 64 + 16 * kb + 4 * g);
}

/* B fragments of the input of 16 queries: lane l holds features 16 kb +
 * 4 (l / 16) + e of query l % 16 */
__device__ __forceinline__ void query_frag(const float u[3], const float nrm[3], const float lu[3], int g,
                                           bf16x4 xin[3])
{
    for (int kb = 0; kb < 3; kb++) {
        float f[4];
        for (int p = 0; p < 2; p++) {
            const int fi = 16 * kb + 4 * g + 2 * p; /* even */
            if (fi < 36) {
                const int k = fi / 6, a = (fi % 6) >> 1;
                band_sincos(k, pick3(u, a), &f[2 * p], &f[2 * p + 1]);
            } else {
                f[2 * p]     = mlp_feature(fi, u, nrm, lu);
                f[2 * p + 1] = mlp_feature(fi + 1, u, nrm, lu);
            }
        }
        xin[kb] = pack4(f[0], f[1], f[2], f[3]);
    }
}

__device__ __forceinline__ float relu(float v) { return v > 0.0f ? v : 0.0f; }

/* logit of the 16 queries of the fragments (valid in lanes 0..15) */
__device__ __forceinline__ float mlp_logit(const MlpFrags& F, const float* __restrict__ Bs, const bf16x4 xin[3],
                                           int lane)
{
    const int g = lane >> 4;
    bf16x4    h[4], h2[4];
    for (int mt = 0; mt < 4; mt++) { /* layer 1: 64 x 48 */
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = 0; kb < 3; kb++) acc = mfma16(F.w1[mt][kb], xin[kb], acc);
        const float4 b = *reinterpret_cast<const float4*>(Bs + kLB1 + 16 * mt + 4 * g);
        h[mt] = pack4(relu(acc[0] + b.x), relu(acc[1] + b.y), relu(acc[2] + b.z),
                      relu(acc[3] + b.w));
    }
    for (int mt = 0; mt < 4; mt++) { /* layer 2 */
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = 0; kb < 4; kb++) acc = mfma16(F.w2[mt][kb], h[kb], acc);
        const float4 b = *reinterpret_cast<const float4*>(Bs + kLB2 + 16 * mt + 4 * g);
        h2[mt] = pack4(relu(acc[0] + b.x), relu(acc[1] + b.y), relu(acc[2] + b.z),
                       relu(acc[3] + b.w));
    }
    for (int mt = 0; mt < 4; mt++) { /* layer 3 */
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = 0; kb < 4; kb++) acc = mfma16(F.w3[mt][kb], h2[kb], acc);
        const float4 b = *reinterpret_cast<const float4*>(Bs + kLB3 + 16 * mt + 4 * g);
        h[mt] = pack4(relu(acc[0] + b.x), relu(acc[1] + b.y), relu(acc[2] + b.z),
                      relu(acc[3] + b.w));
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}; /* layer 4: row 0 of 16 x 64 */
    for (int kb = 0; kb < 4; kb++) acc = mfma16(F.w4[kb], h[kb], acc);
    return acc[0] + Bs[kLB4]; /* D[0][query]: lanes 0..15, element 0 */
}

/* Logit of query 16 j + (lane % 16) of the wave's 64 (fragment group j):
 * the group's inputs are handed to the fragment lanes by shuffles, and the
 * result is returned in every lane (it is the one for this lane in the lanes
 * of group j). */
__device__ __forceinline__ float mlp_group(const MlpFrags& F, const float* __restrict__ Bs, const float u[3],
                                           const float nrm[3], const float lu[3], int lane, int j)
{
    const int r = lane & 15, g = lane >> 4;
    const int src = 16 * j + r;
    float     uj[3], nj[3], lj[3];
    for (int a = 0; a < 3; a++) {
        uj[a] = __shfl(u[a], src, 64);
        nj[a] = __shfl(nrm[a], src, 64);
        lj[a] = __shfl(lu[a], src, 64);
    }
    bf16x4 xin[3];
    query_frag(uj, nj, lj, g, xin);
    const float lg = mlp_logit(F, Bs, xin, lane);
    return __shfl(lg, r, 64); /* query 16 j + r's logit sits in lane r */
}

/* Logits of the 64 queries of a wave, one per lane: four fragment groups of 16. */
__device__ __forceinline__ float mlp_logit64(const MlpFrags& F, const float* __restrict__ Bs, const float u[3],
                                             const float nrm[3], const float lu[3], int lane)
{
    const int g   = lane >> 4;
    float     res = 0.0f;
    for (int j = 0; j < 4; j++) {
        const float got = mlp_group(F, Bs, u, nrm, lu, lane, j);
        if (g == j) res = got;
    }
    return res;
}

/* probabilities of n queries, 64 per wave. RAW: inputs from isp/nrm/light
 * (n x 3 each); else from the feature matrix X[48][B] */
template <bool RAW>
__global__ void __launch_bounds__(256) k_mlp_infer(InferArgs ia, const uint16_t* __restrict__ X, int B,
                                                   const float* __restrict__ isp, const float* __restrict__ nrm,
                                                   const float* __restrict__ light, int n, float* __restrict__ pout)
{
    __shared__ float Bs[kLBN];
    load_biases_lds(ia, Bs);
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, nw = (gridDim.x * blockDim.x) >> 6;
    const int r = lane & 15, g = lane >> 4;
    MlpFrags  F;
    load_frags(ia.W, lane, F);
    for (int q0 = wave * 64; q0 < n; q0 += nw * 64) {
        const int s = q0 + lane;
        float     logit;
        if (RAW) {
            float u[3] = {0.f, 0.f, 0.f}, nn[3] = {0.f, 0.f, 0.f}, lu[3] = {0.f, 0.f, 0.f};
            if (s < n) {
                const float p3[3] = {isp[3 * s], isp[3 * s + 1], isp[3 * s + 2]};
                const float l3[3] = {light[3 * s], light[3 * s + 1], light[3 * s + 2]};
                mlp_scale(p3, ia.bx, ia.by, ia.bz, ia.bw, u);
                mlp_scale(l3, ia.bx, ia.by, ia.bz, ia.bw, lu);
                nn[0] = nrm[3 * s], nn[1] = nrm[3 * s + 1], nn[2] = nrm[3 * s + 2];
            }
            logit = mlp_logit64(F, Bs, u, nn, lu, lane);
        } else {
            logit = 0.0f;
            for (int j = 0; j < 4; j++) {
                const int sj = q0 + 16 * j + r;
                bf16x4    xin[3];
                for (int kb = 0; kb < 3; kb++)
                    for (int e = 0; e < 4; e++)
                        xin[kb][e] = sj < n ? (short) X[(size_t) (16 * kb + 4 * g + e) * B + sj] : (short) 0;
                const float lg  = mlp_logit(F, Bs, xin, lane);
                const float got = __shfl(lg, r, 64);
                if (g == j) logit = got;
            }
        }
        if (s < n) pout[s] = 1.0f / (1.0f + expf(-logit));
    }
}

/* The decision pass: for each (shaded pixel, light) query, 64 per wave,
 * the predicted bit outside the band, LS_UNSURE inside it (those are then
 * compacted into the light's exact-trace list). Pixels of light l:
 * lists[l * lstride + i], i < *nsel. */
template <bool DUAL>
__global__ void __launch_bounds__(256) k_mlp_shadow(InferArgs ia, SceneDev s, LightsDev L,
                                                    const uint32_t* __restrict__ lists, size_t lstride,
                                                    const unsigned* __restrict__ nsel, const float4* __restrict__ isp,
                                                    const int* __restrict__ ms, const int* __restrict__ md,
                                                    uint8_t* __restrict__ lstat, size_t npix, float lo_logit,
                                                    float hi_logit,
                                                    unsigned long long* __restrict__ counters)
{
    __shared__ float Bs[kLBN];
    load_biases_lds(ia, Bs);
    const uint32_t nq     = *nsel;
    const uint32_t total  = nq * (uint32_t) L.n;
    const int      lane   = threadIdx.x & 63;
    const int      wave   = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int      nw     = (gridDim.x * blockDim.x) >> 6;
    unsigned       n_pred = 0;
    if ((uint32_t) wave * 64u >= total) return; /* uniform over the wave; no barrier follows */
    MlpFrags F;
    load_frags(ia.W, lane, F);
    /* The inputs of the wave's next 64 queries are gathered while the
     * current ones are evaluated: list entry before fragment group 0, hit
     * point and model index before group 1, normal before groups 2-3, so
     * that each dependent load is covered by a group's MFMA work. */
    const uint32_t step = (uint32_t) nw * 64u;
    uint32_t       q0   = (uint32_t) wave * 64u;
    bool           valid = q0 + (uint32_t) lane < total;
    int            l     = 0;
    uint32_t       gp    = 0;
    float          u[3] = {0.f, 0.f, 0.f}, nrm[3] = {0.f, 0.f, 0.f}, lu[3] = {0.f, 0.f, 0.f};
    if (valid) {
        const uint32_t qi = q0 + (uint32_t) lane;
        l                 = (int) (qi / nq);
        gp                = lists[(size_t) l * lstride + (qi - (uint32_t) l * nq)];
        const float4 ip    = isp[gp];
        const float  p3[3] = {ip.x, ip.y, ip.z};
        mlp_scale(p3, ia.bx, ia.by, ia.bz, ia.bw, u);
        float col[4], n4[4];
        fetch_attr(s.astat, ms[gp], col, n4);
        if (DUAL && md[gp] > 0) fetch_attr(s.adyn, md[gp], col, n4);
        nrm[0] = n4[0], nrm[1] = n4[1], nrm[2] = n4[2];
        mlp_scale(L.p[l], ia.bx, ia.by, ia.bz, ia.bw, lu);
    }
    for (; q0 < total; q0 += step) {
        const int      g      = lane >> 4;
        const uint32_t qn     = q0 + step + (uint32_t) lane;
        const bool     nvalid = qn < total;
        int            nl_    = 0;
        uint32_t       ngp    = 0;
        if (nvalid) {
            nl_ = (int) (qn / nq);
            ngp = lists[(size_t) nl_ * lstride + (qn - (uint32_t) nl_ * nq)];
        }
        float res = mlp_group(F, Bs, u, nrm, lu, lane, 0);
        float4 nip = make_float4(0.f, 0.f, 0.f, 0.f);
        int    nms = 0, nmd = 0;
        if (nvalid) {
            nip = isp[ngp];
            nms = ms[ngp];
            if (DUAL) nmd = md[ngp];
        }
        const float r1 = mlp_group(F, Bs, u, nrm, lu, lane, 1);
        float       ncol[4], n4[4] = {0.f, 0.f, 0.f, 0.f};
        if (nvalid) {
            fetch_attr(s.astat, nms, ncol, n4);
            if (DUAL && nmd > 0) fetch_attr(s.adyn, nmd, ncol, n4);
        }
        const float r2 = mlp_group(F, Bs, u, nrm, lu, lane, 2);
        const float r3 = mlp_group(F, Bs, u, nrm, lu, lane, 3);
        res = g == 1 ? r1 : res;
        res = g == 2 ? r2 : res;
        res = g == 3 ? r3 : res;
        if (valid) {
            const uint8_t d = res < lo_logit ? LS_PRED_OCC : res > hi_logit ? LS_PRED_LIT : LS_UNSURE;
            lstat[(size_t) l * npix + gp] = d;
            n_pred += d != LS_UNSURE ? 1u : 0u;
        }
        valid = nvalid;
        l     = nl_;
        gp    = ngp;
        if (nvalid) {
            const float p3[3] = {nip.x, nip.y, nip.z};
            mlp_scale(p3, ia.bx, ia.by, ia.bz, ia.bw, u);
            nrm[0] = n4[0], nrm[1] = n4[1], nrm[2] = n4[2];
            mlp_scale(L.p[nl_], ia.bx, ia.by, ia.bz, ia.bw, lu);
        }
    }
    n_pred = wave_sum(n_pred);
    if (lane == 0 && n_pred) atomicAdd(&counters[CNT_PRED], (unsigned long long) n_pred);
}

/* training samples of an exact render: queries stride * k + phase of the
 * (light, shaded pixel) sequence, label = the exact visibility */
template <bool DUAL>
__global__ void k_collect(SceneDev s, LightsDev L, const uint32_t* __restrict__ lists, size_t lstride,
                          const unsigned* __restrict__ nsel, const float4* __restrict__ isp,
                          const int* __restrict__ ms, const int* __restrict__ md, const uint8_t* __restrict__ lstat,
                          size_t npix, uint32_t stride, uint32_t phase, RawSample* __restrict__ out, size_t cap,
                          unsigned long long* __restrict__ ctr)
{
    const uint64_t nq    = *nsel;
    const uint64_t qi    = ((uint64_t) blockIdx.x * blockDim.x + threadIdx.x) * stride + phase;
    const int      lane  = threadIdx.x & 63;
    const bool     valid = qi < nq * (uint64_t) L.n;
    int            l     = 0;
    uint32_t       gp    = 0;
    uint8_t        ls    = LS_SKIPPED;
    if (valid) {
        l  = (int) (qi / nq);
        gp = lists[(size_t) l * lstride + (qi - (uint64_t) l * nq)];
        ls = lstat[(size_t) l * npix + gp];
        /* a light after one that discarded the fragment does not count (its
         * ray may have been traced: the lights share one launch) */
        for (int j = 0; j < l; j++) ls = lstat[(size_t) j * npix + gp] == LS_DISCARD ? (uint8_t) LS_SKIPPED : ls;
    }
    /* one slot reservation per wave (a per-sample atomic on one counter
     * would queue every sample behind the others) */
    const bool     keep = ls == LS_LIT || ls == LS_OCCLUDED;
    const uint64_t m    = __ballot(keep);
    if (m == 0ull) return; /* uniform over the wave */
    const int          leader = __ffsll((unsigned long long) m) - 1;
    unsigned long long base   = 0;
    if (lane == leader) base = atomicAdd(&ctr[0], (unsigned long long) __popcll(m));
    base                          = __shfl(base, leader, 64);
    const unsigned long long slot = base + (unsigned long long) __popcll(m & ((1ull << lane) - 1ull));
    const uint64_t           lit  = __ballot(keep && ls == LS_LIT && slot < cap);
    if (lane == leader && lit) atomicAdd(&ctr[1], (unsigned long long) __popcll(lit));
    if (!keep || slot >= cap) return;
    RawSample    rs;
    const float4 ip = isp[gp];
    rs.isp[0] = ip.x, rs.isp[1] = ip.y, rs.isp[2] = ip.z;
    float col[4], n4[4];
    fetch_attr(s.astat, ms[gp], col, n4);
    if (DUAL && md[gp] > 0) fetch_attr(s.adyn, md[gp], col, n4);
    rs.nrm[0] = n4[0], rs.nrm[1] = n4[1], rs.nrm[2] = n4[2];
    rs.light[0] = L.p[l][0], rs.light[1] = L.p[l][1], rs.light[2] = L.p[l][2];
    rs.label    = ls == LS_LIT ? 1.0f : 0.0f;
    out[slot]   = rs;
}

__global__ void k_unpack_samples(const RawSample* __restrict__ S, size_t start, size_t n, float* __restrict__ out)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const RawSample r = S[start + i];
    float*          o = out + 10 * i;
    for (int k = 0; k < 3; k++) o[k] = r.isp[k], o[3 + k] = r.nrm[k], o[6 + k] = r.light[k];
    o[9] = r.label;
}

} // namespace

/* ------------------------------------------------------------------------ */
/* host side                                                                */
/* ------------------------------------------------------------------------ */

void qbt_ctx::mlp_free()
{
    if (!mlp) return;
    MlpState* m = mlp;
    for (DevBuf* b : {&m->params, &m->m, &m->v, &m->packed, &m->ctr, &m->samples, &m->perm, &m->keys,
                      &m->vals, &m->sort_tmp, &m->X, &m->gpart, &m->lossbuf, &m->io_x, &m->io_p, &m->io_y,
                      &m->io_a, &m->io_c, &m->flat})
        dev_free(*b);
    delete mlp;
    mlp = nullptr;
}

bool qbt_surrogate_ready(const qbt_ctx* c) { return c && c->mlp && c->mlp->ready; }

static int mlp_state(qbt_ctx* c, MlpState** out)
{
    if (!c->mlp) {
        c->mlp = new (std::nothrow) MlpState();
        if (!c->mlp) return QBT_ENOMEM;
        MlpState* m = c->mlp;
        int       rc;
        if ((rc = c->dev_alloc(m->params, kMlpParams * 4)) || (rc = c->dev_alloc(m->m, kMlpParams * 4)) ||
            (rc = c->dev_alloc(m->v, kMlpParams * 4)) || (rc = c->dev_alloc(m->packed, kPackAll * 2)) || (rc = c->dev_alloc(m->lossbuf, 64)) ||
            (rc = c->dev_alloc(m->ctr, 16)) || (rc = c->dev_alloc(m->flat, kMlpParams * 4))) {
            c->mlp_free();
            return rc;
        }
        k_fill_u64<<<1, 64, 0, c->stream>>>((unsigned long long*) m->ctr.p, 2);
        HIPCHK(hipGetLastError());
    }
    *out = c->mlp;
    return QBT_OK;
}

static int mlp_repack(qbt_ctx* c)
{
    k_mlp_pack<<<nblk(kPackAll), 256, 0, c->stream>>>((const float*) c->mlp->params.p, (uint16_t*) c->mlp->packed.p);
    HIPCHK(hipGetLastError());
    return QBT_OK;
}

static int mlp_reset_adam(qbt_ctx* c)
{
    MlpState* m = c->mlp;
    k_fill_f32<<<nblk(kMlpParams), 256, 0, c->stream>>>((float*) m->m.p, kMlpParams, 0.0f);
    k_fill_f32<<<nblk(kMlpParams), 256, 0, c->stream>>>((float*) m->v.p, kMlpParams, 0.0f);
    HIPCHK(hipGetLastError());
    m->t = 0;
    return QBT_OK;
}

extern "C" int qbt_surrogate_init(qbt_ctx* c, uint64_t seed)
{
    if (!c) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m;
    int       rc = mlp_state(c, &m);
    if (rc) return rc;
    k_mlp_init<<<nblk(kMlpParams), 256, 0, c->stream>>>((float*) m->params.p, seed);
    HIPCHK(hipGetLastError());
    if ((rc = mlp_reset_adam(c)) || (rc = mlp_repack(c))) return rc;
    m->ready = true;
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

extern "C" int qbt_surrogate_set_params(qbt_ctx* c, const float* params, size_t n)
{
    if (!c || !params || n != (size_t) kMlpParams) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m;
    int       rc = mlp_state(c, &m);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(m->params.p, params, kMlpParams * 4, hipMemcpyHostToDevice, c->stream));
    if ((rc = mlp_reset_adam(c)) || (rc = mlp_repack(c))) return rc;
    m->ready = true;
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

extern "C" int qbt_surrogate_get_params(qbt_ctx* c, float* params, size_t n)
{
    if (!c || !params || n != (size_t) kMlpParams || !qbt_surrogate_ready(c)) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemcpyAsync(params, c->mlp->params.p, kMlpParams * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

extern "C" int qbt_surrogate_set_band(qbt_ctx* c, float lo, float hi)
{
    if (!c || !(lo > 0.0f) || !(hi < 1.0f) || !(lo <= hi)) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m;
    int       rc = mlp_state(c, &m);
    if (rc) return rc;
    m->band_lo = lo;
    m->band_hi = hi;
    return QBT_OK;
}

extern "C" int qbt_surrogate_reserve(qbt_ctx* c, size_t nsamples, uint32_t stride)
{
    if (!c || nsamples == 0 || nsamples > ((size_t) 1 << 31) || stride == 0) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m;
    int       rc = mlp_state(c, &m);
    if (rc) return rc;
    if ((rc = c->dev_alloc(m->samples, nsamples * sizeof(RawSample)))) return rc;
    m->cap    = nsamples;
    m->stride = stride;
    m->phase  = 0;
    m->perm_n = 0;
    k_fill_u64<<<1, 64, 0, c->stream>>>((unsigned long long*) m->ctr.p, 2);
    HIPCHK(hipGetLastError());
    return QBT_OK;
}

static int mlp_counts(qbt_ctx* c, size_t* n, size_t* lit)
{
    unsigned long long h[2] = {0ull, 0ull};
    MlpState*          m    = c->mlp;
    if (m && m->cap) {
        HIPCHK(hipMemcpyAsync(h, m->ctr.p, 16, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
    }
    if (n) *n = m ? (size_t) (h[0] < m->cap ? h[0] : m->cap) : 0;
    if (lit) *lit = (size_t) h[1];
    return QBT_OK;
}

extern "C" int qbt_surrogate_samples(qbt_ctx* c, size_t* n, size_t* lit)
{
    if (!c || !n) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    return mlp_counts(c, n, lit);
}

extern "C" int qbt_surrogate_read_samples(qbt_ctx* c, size_t start, size_t n, float* out)
{
    if (!c || (n && !out)) return QBT_EINVAL;
    if (n == 0) return QBT_OK;
    HIPCHK(hipSetDevice(c->device));
    size_t held = 0;
    int    rc   = mlp_counts(c, &held, nullptr);
    if (rc) return rc;
    if (start > held || n > held - start) return QBT_ERANGE;
    MlpState* m = c->mlp;
    if ((rc = c->dev_alloc(m->io_c, n * 40))) return rc;
    k_unpack_samples<<<nblk(n), 256, 0, c->stream>>>((const RawSample*) m->samples.p, start, n, (float*) m->io_c.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, m->io_c.p, n * 40, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

constexpr int kTrainBlocks = 256; /* blocks of k_mlp_train, rows of partial gradients, at most */

static int train_rows(int B) { return std::min((B + kChunk - 1) / kChunk, kTrainBlocks); }

/* the partial gradients of a batch of width B */
static int mlp_grad_buf(qbt_ctx* c, int B) { return c->dev_alloc(c->mlp->gpart, (size_t) train_rows(B) * kGradN * 4); }

/* Forward and backward of a minibatch: the partial gradients into gpart and,
 * if asked for, the summed loss into lossbuf. */
static int mlp_fwd_bwd(qbt_ctx* c, const TrainBatch& T, bool want_loss)
{
    MlpState*       m    = c->mlp;
    const int       rows = train_rows(T.B);
    double*         loss = want_loss ? (double*) m->lossbuf.p : nullptr;
    const uint16_t* W    = (const uint16_t*) m->packed.p;
    if (loss) k_fill_f32<<<1, 64, 0, c->stream>>>((float*) m->lossbuf.p, 2, 0.0f);
    if (T.S) k_mlp_train<true><<<rows, 256, 0, c->stream>>>(W, (const float*) m->params.p, T, (float*) m->gpart.p, loss);
    else k_mlp_train<false><<<rows, 256, 0, c->stream>>>(W, (const float*) m->params.p, T, (float*) m->gpart.p, loss);
    HIPCHK(hipGetLastError());
    return QBT_OK;
}

/* mean loss of the last mlp_fwd_bwd that was asked for it (synchronises) */
static int mlp_read_loss(qbt_ctx* c, int n, double* out)
{
    double l = 0.0;
    HIPCHK(hipMemcpyAsync(&l, c->mlp->lossbuf.p, 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    *out = l / (n > 0 ? n : 1);
    return QBT_OK;
}

/* an Adam step with the gradient of the last mlp_fwd_bwd (batch width B) */
static int mlp_adam_step(qbt_ctx* c, int B, float lr)
{
    MlpState* m = c->mlp;
    m->t++;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f - powf(b1, (float) m->t), c2 = 1.0f - powf(b2, (float) m->t);
    k_mlp_step<<<kGradN / 64, 256, 0, c->stream>>>((const float*) m->gpart.p, train_rows(B), nullptr, (float*) m->params.p,
                                                   (float*) m->m.p, (float*) m->v.p, (uint16_t*) m->packed.p,
                                                   AdamArgs{lr, b1, b2, eps, c1, c2});
    HIPCHK(hipGetLastError());
    return QBT_OK;
}

/* host feature rows (n x 42) -> X, labels -> io_y; B = n rounded up to 16 */
static int mlp_load_host(qbt_ctx* c, const float* x, const float* y, size_t n, int* Bout)
{
    MlpState* m = c->mlp;
    const int    B = (int) ((n + 15) / 16) * 16;
    const size_t b = (size_t) B;
    int          rc;
    if ((rc = c->dev_alloc(m->X, kMlpInPad * b * 2)) || (rc = c->dev_alloc(m->io_y, b * 4)) ||
        (rc = c->dev_alloc(m->io_p, b * 4)) || (rc = c->dev_alloc(m->io_x, n * kMlpIn * 4)) ||
        (rc = c->dev_alloc(m->io_a, n * 4)))
        return rc;
    HIPCHK(hipMemcpyAsync(m->io_x.p, x, n * kMlpIn * 4, hipMemcpyHostToDevice, c->stream));
    if (y) HIPCHK(hipMemcpyAsync(m->io_a.p, y, n * 4, hipMemcpyHostToDevice, c->stream));
    k_copy_features<<<nblk(B), 256, 0, c->stream>>>((const float*) m->io_x.p, B, (int) n, (uint16_t*) m->X.p,
                                                    y ? (const float*) m->io_a.p : nullptr, (float*) m->io_y.p);
    HIPCHK(hipGetLastError());
    *Bout = B;
    return QBT_OK;
}

static unsigned infer_grid(const qbt_ctx* c, size_t n)
{
    const size_t groups = (n + 15) / 16; /* one group of 16 queries per wave, 4 waves per block */
    const size_t blocks = (groups + 3) / 4;
    const size_t maxb   = (size_t) c->num_cus * 4;
    return (unsigned) (blocks < maxb ? (blocks ? blocks : 1) : maxb);
}

extern "C" int qbt_surrogate_forward(qbt_ctx* c, const float* x, size_t n, float* p)
{
    if (!c || (n && (!x || !p)) || n > ((size_t) 1 << 24) || !qbt_surrogate_ready(c)) return QBT_EINVAL;
    if (n == 0) return QBT_OK;
    HIPCHK(hipSetDevice(c->device));
    int B, rc;
    if ((rc = mlp_load_host(c, x, nullptr, n, &B))) return rc;
    MlpState* m = c->mlp;
    InferArgs ia{(const uint16_t*) m->packed.p, (const float*) m->params.p, 0.f, 0.f, 0.f, 1.f};
    k_mlp_infer<false><<<infer_grid(c, n), 256, 0, c->stream>>>(ia, (const uint16_t*) m->X.p, B, nullptr, nullptr,
                                                                 nullptr, (int) n, (float*) m->io_p.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(p, m->io_p.p, n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

extern "C" int qbt_surrogate_predict(qbt_ctx* c, const float* isp, const float* nrm, const float* light, size_t n,
                                     const float basecube[4], float* p)
{
    if (!c || (n && (!isp || !nrm || !light || !p)) || !basecube || !(basecube[3] > 0.0f) ||
        n > ((size_t) 1 << 24) || !qbt_surrogate_ready(c))
        return QBT_EINVAL;
    if (n == 0) return QBT_OK;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m = c->mlp;
    int       rc;
    if ((rc = c->dev_alloc(m->io_x, n * 12 * 3)) || (rc = c->dev_alloc(m->io_a, n * 4))) return rc;
    float* d = (float*) m->io_x.p;
    HIPCHK(hipMemcpyAsync(d, isp, n * 12, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d + 3 * n, nrm, n * 12, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d + 6 * n, light, n * 12, hipMemcpyHostToDevice, c->stream));
    InferArgs ia{(const uint16_t*) m->packed.p, (const float*) m->params.p, basecube[0], basecube[1], basecube[2],
                 basecube[3]};
    k_mlp_infer<true><<<infer_grid(c, n), 256, 0, c->stream>>>(ia, nullptr, 0, d, d + 3 * n, d + 6 * n, (int) n,
                                                                (float*) m->io_a.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(p, m->io_a.p, n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

/* forward and backward of n labelled host rows; *B the padded batch width */
static int mlp_host_batch(qbt_ctx* c, const float* x, const float* y, size_t n, float* loss, int* B)
{
    if (!c || !x || !y || n == 0 || n > ((size_t) 1 << 22) || !qbt_surrogate_ready(c)) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    int rc;
    if ((rc = mlp_load_host(c, x, y, n, B)) || (rc = mlp_grad_buf(c, *B))) return rc;
    TrainBatch T{};
    T.X = (const uint16_t*) c->mlp->X.p, T.Y = (const float*) c->mlp->io_y.p, T.B = *B, T.n = (int) n;
    if ((rc = mlp_fwd_bwd(c, T, true))) return rc;
    double l = 0.0;
    if ((rc = mlp_read_loss(c, (int) n, &l))) return rc;
    if (loss) *loss = (float) l;
    return QBT_OK;
}

extern "C" int qbt_surrogate_grad(qbt_ctx* c, const float* x, const float* y, size_t n, float* grads, float* loss)
{
    int B, rc;
    if ((rc = mlp_host_batch(c, x, y, n, loss, &B))) return rc;
    if (!grads) return QBT_OK;
    MlpState* m = c->mlp;
    k_mlp_step<<<kGradN / 64, 256, 0, c->stream>>>((const float*) m->gpart.p, train_rows(B), (float*) m->flat.p, nullptr,
                                                   nullptr, nullptr, nullptr, AdamArgs{});
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(grads, m->flat.p, kMlpParams * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

extern "C" int qbt_surrogate_step(qbt_ctx* c, const float* x, const float* y, size_t n, float lr, float* loss)
{
    if (!(lr >= 0.0f)) return QBT_EINVAL;
    int B, rc;
    if ((rc = mlp_host_batch(c, x, y, n, loss, &B)) || (rc = mlp_adam_step(c, B, lr))) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    return QBT_OK;
}

int qbt_collect_batch(qbt_ctx* c, const SceneDev& s, bool dual, const LightsDev& L, const uint32_t* lists,
                      size_t list_stride, const unsigned* nsel, size_t npix)
{
    MlpState* m = c->mlp;
    if (!m || !m->cap) return QBT_OK;
    const uint32_t stride = m->stride, phase = m->phase;
    m->phase = (m->phase + 1) % stride; /* successive renders sample different queries */
    const size_t threads = (npix * (size_t) L.n) / stride + 1;
    auto         go      = [&](auto kern) {
        kern<<<nblk(threads), 256, 0, c->stream>>>(s, L, lists, list_stride, nsel, (const float4*) c->wb_isp.p,
                                                   (const int*) c->wb_ms.p, (const int*) c->wb_md.p,
                                                   (const uint8_t*) c->wb_lstat.p, npix, stride, phase,
                                                   (RawSample*) m->samples.p, m->cap, (unsigned long long*) m->ctr.p);
    };
    if (dual) go(k_collect<true>);
    else go(k_collect<false>);
    HIPCHK(hipGetLastError());
    return QBT_OK;
}

extern "C" int qbt_surrogate_train(qbt_ctx* c, const float basecube[4], int steps, int batch, float lr,
                                   uint64_t seed, float* loss_out)
{
    if (!c || !basecube || steps <= 0 || batch < 16 || batch % 16 || batch > (1 << 20) || !(lr >= 0.0f) ||
        !(basecube[3] > 0.0f) || !qbt_surrogate_ready(c))
        return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    MlpState* m = c->mlp;
    size_t    n = 0;
    int       rc;
    if ((rc = mlp_counts(c, &n, nullptr))) return rc;
    if (n < (size_t) batch) return QBT_EINVAL;
    if ((rc = mlp_grad_buf(c, batch)) || (rc = c->dev_alloc(m->perm, n * 4)) || (rc = c->dev_alloc(m->keys, n * 8)) ||
        (rc = c->dev_alloc(m->vals, n * 4)))
        return rc;
    size_t tb = 0;
    HIPCHK(rocprim::radix_sort_pairs(nullptr, tb, (uint32_t*) m->keys.p, (uint32_t*) m->keys.p + n,
                                     (uint32_t*) m->vals.p, (uint32_t*) m->perm.p, n, 0, 32, c->stream));
    if ((rc = c->dev_alloc(m->sort_tmp, tb ? tb : 16))) return rc;
    auto shuffle = [&]() -> int {
        k_perm_keys<<<nblk(n), 256, 0, c->stream>>>((uint32_t*) m->keys.p, (uint32_t*) m->vals.p, n,
                                                    seed + 0x51ED270Bull * ++m->epoch);
        size_t b2 = tb;
        HIPCHK(rocprim::radix_sort_pairs(m->sort_tmp.p, b2, (uint32_t*) m->keys.p, (uint32_t*) m->keys.p + n,
                                         (uint32_t*) m->vals.p, (uint32_t*) m->perm.p, n, 0, 32, c->stream));
        m->pos    = 0;
        m->perm_n = n;
        return QBT_OK;
    };
    /* a new shuffle when the store changed size or the permutation is used up */
    if (m->perm_n != n && (rc = shuffle())) return rc;
    for (int it = 0; it < steps; it++) {
        if (m->pos + (size_t) batch > n && (rc = shuffle())) return rc;
        TrainBatch T{};
        T.S = (const RawSample*) m->samples.p, T.perm = (const uint32_t*) m->perm.p, T.off = m->pos;
        T.bx = basecube[0], T.by = basecube[1], T.bz = basecube[2], T.bw = basecube[3];
        T.B = T.n = batch;
        m->pos += (size_t) batch;
        if ((rc = mlp_fwd_bwd(c, T, it == steps - 1)) || (rc = mlp_adam_step(c, batch, lr))) return rc;
    }
    double last = 0.0;
    if ((rc = mlp_read_loss(c, batch, &last))) return rc;
    if (loss_out) *loss_out = (float) last;
    return QBT_OK;
}

void qbt_surrogate_band(const qbt_ctx* c, float* lo, float* hi)
{
    *lo = c->mlp ? c->mlp->band_lo : 0.0f;
    *hi = c->mlp ? c->mlp->band_hi : 0.0f;
}

int qbt_surrogate_decide(qbt_ctx* c, const SceneDev& s, bool dual, const LightsDev& L, const uint32_t* lists,
                         size_t list_stride, const unsigned* nsel, size_t npix)
{
    MlpState* m = c->mlp;
    if (!m || !m->ready) return QBT_EINVAL;
    InferArgs ia{(const uint16_t*) m->packed.p, (const float*) m->params.p, s.bx, s.by, s.bz, s.bw};
    /* band edges as logits: p < lo  <=>  logit < log(lo / (1 - lo)) */
    const float lo   = logf(m->band_lo / (1.0f - m->band_lo));
    const float hi   = logf(m->band_hi / (1.0f - m->band_hi));
    const int   grid = c->num_cus * 2; /* two 4-wave blocks per CU: the occupancy at ~220 VGPRs */
    auto        go   = [&](auto kern) {
        kern<<<grid, 256, 0, c->stream>>>(ia, s, L, lists, list_stride, nsel, (const float4*) c->wb_isp.p,
                                          (const int*) c->wb_ms.p, (const int*) c->wb_md.p, (uint8_t*) c->wb_lstat.p,
                                          npix, lo, hi, (unsigned long long*) c->counters.p);
    };
    c->prof_mark_begin(QBT_PROF_SURROGATE);
    if (dual) go(k_mlp_shadow<true>);
    else go(k_mlp_shadow<false>);
    c->prof_mark_end();
    return QBT_OK;
}
