// Learned SGS closure kernels: training (gradient, reduction, Adam), inference
// with the network staged in LDS, the fused per-point closure of the solver
// step, its DSM fallback merge, and training-pair sampling from a DSM state.
//
// Matrix products use v_mfma_f32_16x16x32_bf16 (gfx950).  Operand layout of
// one 16x16x32 product D = A B on a 64-lane wave, lane l, g = l / 16:
//   A[i][k]: lane holds i = l % 16, k = 8 g + e (e = 0..7)
//   B[k][j]: lane holds j = l % 16, k = 8 g + e
//   D[i][j]: lane holds j = l % 16, i = 4 g + r (r = 0..3)
// Compiled with -ffp-contract=off: the FP32 and FP64 scalar arithmetic is
// rounded once per operation, except for the fused step in the GELU's exponent;
// biases enter a product as its accumulator.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "closure.h"

namespace mc3d {

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(const s16x8 &a, const s16x8 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
}

// the biases of the four neurons 16t + 4g + r of an output tile
__device__ __forceinline__ f32x4 bias4(const float *b, int t, int g) {
    return *reinterpret_cast<const f32x4 *>(b + 16 * t + 4 * g);
}

constexpr float kG0 = 0.7978845608028654f;  // sqrt(2 / pi)
constexpr float kG1 = 0.044715f;

// tanh-form GELU 0.5 z (1 + tanh u), u = k0 (z + k1 z^3), written as z s with
// s = 1 / (1 + exp(-2u)) = (1 + tanh u) / 2 and exp(-2u) = 2^(z (c1 + c2 z^2)),
// c1 = -2 k0 log2(e), c2 = c1 k1: two products and a fused one, the hardware 2^x
// and reciprocal (the network's evaluation is bound by these vector operations:
// the biases enter as the products' accumulator for the same reason)
constexpr float kGc1 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634);
constexpr float kGc2 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634 * 0.044715);
__device__ __forceinline__ float gelu_s(float z) {
    const float z2 = z * z;
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * __builtin_fmaf(kGc2, z2, kGc1)));
}
__device__ __forceinline__ float gelu(float z) { return z * gelu_s(z); }
// d/dz, s = gelu_s(z): s + z 2 s (1 - s) k0 (1 + 3 k1 z^2)
__device__ __forceinline__ float gelu_grad(float z, float s) {
    return s + z * (2.0f * s * (1.0f - s)) * (kG0 * (1.0f + 3.0f * kG1 * z * z));
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

// FP32 -> BF16 by the hardware conversion (round to nearest even)
__device__ __forceinline__ short bf16_bits(float v) { return __builtin_bit_cast(short, (__bf16)v); }

__device__ __forceinline__ int kappa(int b, int g, int e) { return 16 * (2 * b + (e >> 2)) + 4 * g + (e & 3); }

// ---------------------------------------------------------------------------
// training: one workgroup = 4 waves = 64 samples; wave w carries samples
// 16w .. 16w+15 forward and backward in registers, then forms row tile w of
// every weight gradient.
//
// Products of the passes are computed transposed as in the inference below:
// D = W h^T (rows = neurons, columns = the wave's 16 samples), so a layer's
// output tiles are the next layer's B operand once the contraction index is
// permuted by kappa, forward (W) and backward (W^T) alike, and z, h and dz
// never leave the registers that form them.  LDS holds what lanes share: the
// weights as operands (16 bytes per lane and product, converted once per
// workgroup), and h^T and dz^T as BF16 rows of 64 samples, from which the
// weight gradients dW = dz^T h read their operands as 16-byte loads.
//
// What bounds it: a batch of 8192 is 128 workgroups, one per CU, so the chain
// of one wave (staging, 60 products, 192 GELUs and their gradients per
// sample), not the matrix units.  The earlier form staged every operand
// element by element through 16-bit LDS reads and recomputed z in the backward
// pass: 56.0 us per batch of 8192, now 13.4.
// ---------------------------------------------------------------------------
constexpr int kT = kMlpTile;
constexpr int kTLd = kT + 8;              // samples per LDS row, padded (16-byte rows, no bank conflicts)
constexpr int kFwdOps = 4 + 8 + 8 + 2;    // W1 t; W2 t,b; W3 t,b; W4 b
constexpr int kTrainOps = kFwdOps + 4 + 8 + 8;  // then W4^T t; W3^T t,b; W2^T t,b

struct TrainLds {
    s16x8 w[kTrainOps][64];                  // operands, entry [op][lane]
    unsigned short a0[16 * kTLd];            // inputs^T (7 features, zero rows above)
    unsigned short act[3][kMlpHid * kTLd];   // GELU outputs^T
    unsigned short dz[3][kMlpHid * kTLd];    // deltas^T of the pre-activations
    unsigned short dy[kMlpOut * kTLd];       // dL/dy^T
    float b[3][kMlpHid];
    float red[4][3 * kMlpHid + kMlpOut + 1]; // per-wave sums: three bias gradients, db4, squares
};

// the operands of wave w (row tile w of every matrix; TRAIN: column tiles too, for
// the backward products) for the lane (i = lane % 16, g = lane / 16), converted
// from the FP32 parameters; the four waves' shares are equal and straight-line, so
// every load is in flight before the first conversion
template <bool TRAIN>
__device__ __forceinline__ void stage_operands(const float *__restrict__ P, s16x8 (*ops)[64], int w, int l) {
    const int i = l & 15, g = l >> 4;
    float r1[8], c4[2], c3[2][8], c2[2][8];
    f32x4 r[3][2][2];
#pragma unroll
    for (int e = 0; e < kMlpIn; ++e) r1[e] = P[kMlpOffW1 + (16 * w + i) * kMlpIn + e];
    r1[7] = 0.0f;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            const int col = 32 * b + 16 * hi + 4 * g;
            r[0][b][hi] = *reinterpret_cast<const f32x4 *>(P + kMlpOffW2 + (16 * w + i) * kMlpHid + col);
            r[1][b][hi] = *reinterpret_cast<const f32x4 *>(P + kMlpOffW3 + (16 * w + i) * kMlpHid + col);
            r[2][b][hi] = *reinterpret_cast<const f32x4 *>(P + kMlpOffW4 + (i < kMlpOut ? i : 0) * kMlpHid + col);
        }
    if constexpr (TRAIN) {
#pragma unroll
        for (int o = 0; o < kMlpOut; ++o) c4[o] = P[kMlpOffW4 + o * kMlpHid + 16 * w + i];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                c3[b][e] = P[kMlpOffW3 + kappa(b, g, e) * kMlpHid + 16 * w + i];
                c2[b][e] = P[kMlpOffW2 + kappa(b, g, e) * kMlpHid + 16 * w + i];
            }
    }
    s16x8 o1, o4;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        o1[e] = g == 0 ? bf16_bits(r1[e]) : (short)0;
        if constexpr (TRAIN) o4[e] = g == 0 && e < kMlpOut ? bf16_bits(c4[e < kMlpOut ? e : 0]) : (short)0;
    }
    ops[w][l] = o1;
    if constexpr (TRAIN) ops[22 + w][l] = o4;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        s16x8 o2, o3, o2t, o3t, o4r;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o2[e] = bf16_bits(r[0][b][e >> 2][e & 3]);
            o3[e] = bf16_bits(r[1][b][e >> 2][e & 3]);
            o4r[e] = i < kMlpOut ? bf16_bits(r[2][b][e >> 2][e & 3]) : (short)0;
            if constexpr (TRAIN) {
                o3t[e] = bf16_bits(c3[b][e]);
                o2t[e] = bf16_bits(c2[b][e]);
            }
        }
        ops[4 + 2 * w + b][l] = o2;
        ops[12 + 2 * w + b][l] = o3;
        if (w == 0) ops[20 + b][l] = o4r;
        if constexpr (TRAIN) {
            ops[26 + 2 * w + b][l] = o3t;
            ops[34 + 2 * w + b][l] = o2t;
        }
    }
}

// one step of sample_sums: the lane keeps the half of its 2 H values that its
// bit H selects and adds its partner's
template <int H>
__device__ __forceinline__ void fold_samples(float *v, int i) {
    const bool up = i & H;
#pragma unroll
    for (int k = 0; k < H; ++k) {
        const float keep = up ? v[k + H] : v[k], send = up ? v[k] : v[k + H];
        v[k] = keep + __shfl_xor(send, H);
    }
}

// sums over the 16 samples of the wave of the 16 values v[4t + r] (neuron
// 16t + 4g + r): a transposing butterfly, after which lane (g, i) holds the
// sum of value i, neuron 16 (i/4) + 4g + i%4 (fixed order); overwrites v
__device__ __forceinline__ float sample_sums(float *v, int i) {
    fold_samples<8>(v, i);
    fold_samples<4>(v, i);
    fold_samples<2>(v, i);
    fold_samples<1>(v, i);
    return v[0];
}

// h = GELU(z) as the next layer's operand (BF16) and as rows of the transposed
// LDS copy; z becomes GELU'(z), which shares the exponential and the reciprocal
__device__ __forceinline__ void train_activate(f32x4 z[4], s16x8 h[2], unsigned short *rows, int g, int smp) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float zz = z[t][r], sg = gelu_s(zz);
            const short v = bf16_bits(zz * sg);
            z[t][r] = gelu_grad(zz, sg);
            h[t >> 1][4 * (t & 1) + r] = v;
            rows[(16 * t + 4 * g + r) * kTLd + smp] = (unsigned short)v;
        }
}

// dz = dh GELU'(z): FP32 sums over the wave's samples into red, BF16 operand and LDS rows
__device__ __forceinline__ void train_delta(const f32x4 dh[4], const f32x4 gz[4], s16x8 d[2], unsigned short *rows,
                                            float *red, int i, int g, int smp) {
    float v[16];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[4 * t + r] = dh[t][r] * gz[t][r];
            const short q = bf16_bits(v[4 * t + r]);
            d[t >> 1][4 * (t & 1) + r] = q;
            rows[(16 * t + 4 * g + r) * kTLd + smp] = (unsigned short)q;
        }
    red[16 * (i >> 2) + 4 * g + (i & 3)] = sample_sums(v, i);
}

// 16 rows of D = A B over the 64 samples, A rows of dz^T, B rows of h^T
__device__ __forceinline__ f32x4 sample_product(const unsigned short *arow, const unsigned short *brow, int g) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < kT; k0 += 32)
        acc = mfma(*reinterpret_cast<const s16x8 *>(arow + k0 + 8 * g), *reinterpret_cast<const s16x8 *>(brow + k0 + 8 * g),
                   acc);
    return acc;
}

__global__ __launch_bounds__(256) void k_mlp_grad(const float *__restrict__ P, const float *__restrict__ X,
                                                  const float *__restrict__ Tg, const int *__restrict__ idx,
                                                  long n, float scale, float *__restrict__ partial,
                                                  float *__restrict__ lossp) {
    __shared__ __attribute__((aligned(16))) TrainLds s;
    const int tid = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(tid >> 6), i = l & 15, g = l >> 4;
    float *gout = partial + (size_t)blockIdx.x * kMlpParams;

    // ---- this lane's sample (lanes of equal i share it), the operands, the biases ----
    const int smp = 16 * w + i;
    const long q = (long)blockIdx.x * kT + smp;
    const bool ok = q < n;
    const long src = ok ? (idx ? (long)idx[q] : q) : 0;
    s16x8 x;
#pragma unroll
    for (int e = 0; e < 8; ++e)
        x[e] = (g == 0 && ok && e < kMlpIn) ? bf16_bits(X[src * kMlpIn + (e < kMlpIn ? e : 0)]) : (short)0;
    const float t0 = ok ? Tg[src * kMlpOut] : 0.0f, t1 = ok ? Tg[src * kMlpOut + 1] : 0.0f;
    stage_operands<true>(P, s.w, w, l);
    if (tid < 3 * kMlpHid)
        s.b[tid / kMlpHid][tid % kMlpHid] =
            P[(tid < kMlpHid ? kMlpOffB1 : tid < 2 * kMlpHid ? kMlpOffB2 : kMlpOffB3) + tid % kMlpHid];
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // rows 4g .. 4g+3 of the transposed inputs: features of lanes g = 0, zeros above
        const short hi = (short)__shfl((int)x[4 + e], i), lo = (short)__shfl((int)x[e], i);
        s.a0[(4 * g + e) * kTLd + smp] = (unsigned short)(g == 0 ? lo : g == 1 ? hi : (short)0);
    }
    __syncthreads();

    // ---- forward ----
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 z[3][4];
    s16x8 h[2];
#pragma unroll
    for (int t = 0; t < 4; ++t) z[0][t] = mfma(s.w[t][l], x, bias4(s.b[0], t, g));
#pragma unroll
    for (int layer = 0; layer < 3; ++layer) {
        if (layer > 0) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                z[layer][t] = mfma(s.w[8 * layer - 4 + 2 * t + 1][l], h[1],
                                   mfma(s.w[8 * layer - 4 + 2 * t][l], h[0], bias4(s.b[layer], t, g)));
        }
        train_activate(z[layer], h, s.act[layer], g, smp);
    }
    // ---- output layer, loss, dL/dy (lanes g = 0 hold the two outputs of their sample) ----
    const f32x4 y = mfma(s.w[21][l], h[1], mfma(s.w[20][l], h[0], zero));
    const bool real = g == 0 && ok;
    const float d0 = real ? (y[0] + P[kMlpOffB4]) - t0 : 0.0f, d1 = real ? (y[1] + P[kMlpOffB4 + 1]) - t1 : 0.0f;
    const float e0 = scale * d0, e1 = scale * d1;
    s16x8 d[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) d[0][e] = e == 0 ? bf16_bits(e0) : e == 1 ? bf16_bits(e1) : (short)0;
    if (g == 0) {
        s.dy[smp] = (unsigned short)d[0][0];
        s.dy[kTLd + smp] = (unsigned short)d[0][1];
    }
    {
        float sq = d0 * d0 + d1 * d1, s0 = e0, s1 = e1;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
            sq = sq + __shfl_xor(sq, off);
            s0 = s0 + __shfl_xor(s0, off);
            s1 = s1 + __shfl_xor(s1, off);
        }
        if (l == 0) {
            s.red[w][3 * kMlpHid] = s0;
            s.red[w][3 * kMlpHid + 1] = s1;
            s.red[w][3 * kMlpHid + 2] = sq;
        }
    }
    // ---- backward ----
    f32x4 dh[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) dh[t] = mfma(s.w[22 + t][l], d[0], zero);
#pragma unroll
    for (int layer = 2; layer >= 0; --layer) {
        train_delta(dh, z[layer], d, s.dz[layer], s.red[w] + layer * kMlpHid, i, g, smp);
        if (layer == 0) break;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int op = (layer == 2 ? 26 : 34) + 2 * t;
            dh[t] = mfma(s.w[op + 1][l], d[1], mfma(s.w[op][l], d[0], zero));
        }
    }
    __syncthreads();

    // ---- gradients: wave w forms rows 16w .. 16w+15 (columns of W4) ----
#pragma unroll
    for (int layer = 1; layer < 3; ++layer) {
        const unsigned short *a = s.dz[layer] + (16 * w + i) * kTLd, *in = s.act[layer - 1];
        float *o = gout + (layer == 1 ? kMlpOffW2 : kMlpOffW3) + (16 * w + 4 * g) * kMlpHid + i;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const f32x4 acc = sample_product(a, in + (16 * kt + i) * kTLd, g);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r * kMlpHid + 16 * kt] = acc[r];
        }
    }
    {
        const f32x4 acc = sample_product(s.dz[0] + (16 * w + i) * kTLd, s.a0 + i * kTLd, g);
        if (i < kMlpIn) {
#pragma unroll
            for (int r = 0; r < 4; ++r) gout[kMlpOffW1 + (16 * w + 4 * g + r) * kMlpIn + i] = acc[r];
        }
        // rows 2.. of this product repeat row 1 and are not stored
        const f32x4 acc4 = sample_product(s.dy + (i < kMlpOut ? i : kMlpOut - 1) * kTLd, s.act[2] + (16 * w + i) * kTLd, g);
        if (g == 0) {
#pragma unroll
            for (int r = 0; r < kMlpOut; ++r) gout[kMlpOffW4 + r * kMlpHid + 16 * w + i] = acc4[r];
        }
    }
    if (tid < 3 * kMlpHid + kMlpOut + 1) {
        const float v = ((s.red[0][tid] + s.red[1][tid]) + s.red[2][tid]) + s.red[3][tid];
        const int layer = tid / kMlpHid;
        if (layer < 3) gout[(layer == 0 ? kMlpOffB1 : layer == 1 ? kMlpOffB2 : kMlpOffB3) + tid % kMlpHid] = v;
        else if (tid < 3 * kMlpHid + kMlpOut) gout[kMlpOffB4 + tid - 3 * kMlpHid] = v;
        else lossp[blockIdx.x] = v;
    }
}

__device__ __forceinline__ void adam_update(float *__restrict__ P, float *__restrict__ m, float *__restrict__ v,
                                            int p, float gr, const AdamArgs &a) {
    const float mn = a.b1 * m[p] + (1.0f - a.b1) * gr;
    const float vn = a.b2 * v[p] + (1.0f - a.b2) * (gr * gr);
    m[p] = mn;
    v[p] = vn;
    const float mh = mn / a.c1, vh = vn / a.c2;
    P[p] = P[p] - a.lr * mh / (sqrtf(vh) + a.eps);
}

// Sum of the nb partial gradients of every parameter and of the partial
// losses, in a fixed order (the result does not depend on scheduling): a
// workgroup takes 64 parameters, its eight waves each sum an eighth of the
// partials in order (rows of 64 consecutive floats, 16 loads in flight), and
// the eight sums are added in wave order.  Workgroup 0 also sums the partial
// losses: strided per thread, then a fixed tree.  With ADAM the thread that
// holds a parameter's gradient updates it in the same pass (grad null: not
// written), which saves the training loop a launch per batch.
constexpr int kReduceCols = 64, kReduceWaves = 8;
template <bool ADAM>
__global__ __launch_bounds__(512) void k_mlp_reduce(const float *__restrict__ partial,
                                                    const float *__restrict__ lossp, int nb, float inv_norm,
                                                    float *__restrict__ grad, float *__restrict__ loss,
                                                    float *__restrict__ P, float *__restrict__ m,
                                                    float *__restrict__ v, AdamArgs a) {
    __shared__ float part[kReduceWaves][kReduceCols];
    __shared__ float lsum[512];
    const int t = threadIdx.x % kReduceCols, g = threadIdx.x / kReduceCols;
    const int p = blockIdx.x * kReduceCols + t;
    const int per = (nb + kReduceWaves - 1) / kReduceWaves, b0 = g * per, b1 = b0 + per < nb ? b0 + per : nb;
    float acc = 0.0f;
    if (p < kMlpParams) {
#pragma unroll 16
        for (int b = b0; b < b1; ++b) acc = acc + partial[(size_t)b * kMlpParams + p];
    }
    part[g][t] = acc;
    if (blockIdx.x == 0) {
        float l = 0.0f;
        for (int b = threadIdx.x; b < nb; b += 512) l = l + lossp[b];
        lsum[threadIdx.x] = l;
    }
    __syncthreads();
    if (g == 0 && p < kMlpParams) {
        float gr = part[0][t];
#pragma unroll
        for (int k = 1; k < kReduceWaves; ++k) gr = gr + part[k][t];
        if (grad) grad[p] = gr;
        if (ADAM) adam_update(P, m, v, p, gr, a);
    }
    if (blockIdx.x == 0) {
        for (int h = 256; h > 0; h >>= 1) {
            if (threadIdx.x < h) lsum[threadIdx.x] = lsum[threadIdx.x] + lsum[threadIdx.x + h];
            __syncthreads();
        }
        if (threadIdx.x == 0) loss[0] = lsum[0] * inv_norm;
    }
}

__global__ void k_mlp_adam(float *__restrict__ P, float *__restrict__ m, float *__restrict__ v,
                           const float *__restrict__ grad, AdamArgs a) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kMlpParams) adam_update(P, m, v, p, grad[p], a);
}

// ---------------------------------------------------------------------------
// per-point features (FP64 -> FP32), shared by the solver closure and sampling
// ---------------------------------------------------------------------------
struct GradIn {
    const double *dU[3], *dV[3], *dW[3];
    Metrics m;
};

// d u_i / d x_j from d u_i / d xi_k, src/CurvilinearCSolver_Core.cpp:548-561;
// without metric terms (m.J11 null) the inputs are the Cartesian gradient itself
__device__ __forceinline__ void cart_grad(const GradIn &a, long p, double A[3][3]) {
    if (!a.m.J11) {
        const double *const *d[3] = {a.dU, a.dV, a.dW};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) A[i][j] = d[i][j][p];
        return;
    }
    const double J11 = a.m.J11[p], J12 = a.m.J12[p], J13 = a.m.J13[p];
    const double J21 = a.m.J21[p], J22 = a.m.J22[p], J23 = a.m.J23[p];
    const double J31 = a.m.J31[p], J32 = a.m.J32[p], J33 = a.m.J33[p];
    const double *const *d[3] = {a.dU, a.dV, a.dW};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double d0 = d[i][0][p], d1 = d[i][1][p], d2 = d[i][2][p];
        A[i][0] = J11 * d0 + J21 * d1 + J31 * d2;
        A[i][1] = J12 * d0 + J22 * d1 + J32 * d2;
        A[i][2] = J13 * d0 + J23 * d1 + J33 * d2;
    }
}

// raw features and |S| = sqrt(2 S_ij S_ij):
// theta/a, (s2 - w2)/a^2, s3/a^3, sw2/a^3, s2w2/a^4, log a, log(vol/J)/3
__device__ __forceinline__ void features(const double A[3][3], double vol_J, float f[kMlpIn], double &Smag) {
    double S[3][3], Wm[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            S[i][j] = 0.5 * (A[i][j] + A[j][i]);
            Wm[i][j] = 0.5 * (A[i][j] - A[j][i]);
        }
    double s2 = 0.0, w2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            s2 = s2 + S[i][j] * S[i][j];
            w2 = w2 + Wm[i][j] * Wm[i][j];
        }
    double SS[3][3], WW[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            SS[i][j] = (S[i][0] * S[0][j] + S[i][1] * S[1][j]) + S[i][2] * S[2][j];
            WW[i][j] = (Wm[i][0] * Wm[0][j] + Wm[i][1] * Wm[1][j]) + Wm[i][2] * Wm[2][j];
        }
    double s3 = 0.0, sw2 = 0.0, s2w2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            s3 = s3 + SS[i][j] * S[j][i];
            sw2 = sw2 + S[i][j] * WW[j][i];
            s2w2 = s2w2 + SS[i][j] * WW[j][i];
        }
    const double theta = (A[0][0] + A[1][1]) + A[2][2];
    const double a2 = s2 + w2;
    Smag = sqrt(2.0 * s2);
    if (a2 > 0.0) {
        const double a = sqrt(a2), inv = 1.0 / a;
        const double inv2 = inv * inv, inv3 = inv2 * inv;
        f[0] = (float)(theta * inv);
        f[1] = (float)((s2 - w2) * inv2);
        f[2] = (float)(s3 * inv3);
        f[3] = (float)(sw2 * inv3);
        f[4] = (float)(s2w2 * (inv2 * inv2));
        f[5] = (float)log(a);
    } else {
        f[0] = f[1] = f[2] = f[3] = f[4] = 0.0f;
        f[5] = (float)log(1e-300);
    }
    f[6] = (float)(log(vol_J) / 3.0);
}

// ---------------------------------------------------------------------------
// inference: products are computed transposed, D = W h^T (rows = neurons,
// columns = 16 samples), so a layer's output D tiles are already the next
// layer's B operand once the contraction index is permuted: for k-block b, lane
// group g, element e the neuron is kappa(b, g, e) = 16 (2b + e/4) + 4g + e%4,
// which is exactly what the lane holds in its output tiles 2b and 2b+1.
//
// The network stays in LDS and a wave's weight operands are loaded into
// registers only around the products of each 64-point group: the FP64 feature
// phase and the network phase then do not hold their registers at the same
// time (3 waves per SIMD instead of 1).  Per-lane
// operands are stored [operand][lane] as 16-byte entries (w1 t = 0..3, w2 t,b,
// w3 t,b, w4 b), biases by neuron.
// ---------------------------------------------------------------------------
struct InferLds {
    s16x8 w[kFwdOps][64];
    float b[3][kMlpHid];
    float b4[4];  // zero beyond the two outputs
};

// the operands and biases, by a workgroup of four waves.  (Entry by entry, 44
// loads and conversions a thread one after another, k_mlp_infer of up to 60000
// samples, at most one group a wave, took 16.4-18.0 us; 9.2 so, 300000 samples
// 39.5 -> 24.9, k_learned_sgs of 160^3 points 332 -> 307.)
__device__ void stage_infer(const float *__restrict__ P, InferLds &s) {
    stage_operands<false>(P, s.w, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane_id());
    for (int k = threadIdx.x; k < 3 * kMlpHid; k += blockDim.x) {
        const int layer = k / kMlpHid, j = k % kMlpHid;
        s.b[layer][j] = P[(layer == 0 ? kMlpOffB1 : layer == 1 ? kMlpOffB2 : kMlpOffB3) + j];
    }
    if (threadIdx.x < 4) s.b4[threadIdx.x] = threadIdx.x < kMlpOut ? P[kMlpOffB4 + threadIdx.x] : 0.0f;
    __syncthreads();
}

__device__ __forceinline__ void activate(const f32x4 z[4], s16x8 h[2]) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int t = 2 * b + (e >> 2), r = e & 3;
            h[b][e] = bf16_bits(gelu(z[t][r]));
        }
}

// The network on the 64 points of a wave (lane L: standardised inputs x[7]),
// layer by layer over the wave's four 16-point blocks: only one layer's weight
// operands are in registers at a time, loaded from LDS right before its
// products.  Returns this lane's two outputs.
__device__ __forceinline__ void infer64_lds(const InferLds &s, const float x[kMlpIn], float &y0, float &y1) {
    const int l = lane_id(), g = l >> 4;
    // compiler-only barrier: the operand loads below stay here instead of being
    // hoisted out of the caller's loop (which would keep them live through the
    // feature phase)
    __asm__ volatile("" ::: "memory");
    s16x8 h[4][2];
    {  // layer 1: block b's inputs are the features of points 16 b .. 16 b + 15
        s16x8 w[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) w[t] = s.w[t][l];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            s16x8 op;
            const int src = 16 * b + (l & 15);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = e < kMlpIn ? __shfl(x[e < kMlpIn ? e : 0], src) : 0.0f;
                op[e] = (g == 0 && e < kMlpIn) ? bf16_bits(v) : (short)0;
            }
            f32x4 acc[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = mfma(w[t], op, bias4(s.b[0], t, g));
            activate(acc, h[b]);
        }
    }
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {  // layers 2 and 3
        s16x8 w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = s.w[4 + 8 * layer + k][l];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f32x4 acc[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[t] = mfma(w[2 * t + 1], h[b][1], mfma(w[2 * t], h[b][0], bias4(s.b[1 + layer], t, g)));
            activate(acc, h[b]);
        }
    }
    const s16x8 w40 = s.w[20][l], w41 = s.w[21][l];
    const f32x4 b4 = *reinterpret_cast<const f32x4 *>(s.b4);  // (the rows of lanes g > 0 are not read)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const f32x4 y = mfma(w41, h[b][1], mfma(w40, h[b][0], b4));
        const float o0 = __shfl(y[0], l & 15), o1 = __shfl(y[1], l & 15);
        if (g == b) { y0 = o0; y1 = o1; }
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_mlp_infer(
    const float *__restrict__ P, const float *__restrict__ X, float *__restrict__ Y, long n) {
    __shared__ __attribute__((aligned(16))) InferLds net;
    stage_infer(P, net);
    const long nwaves = (long)gridDim.x * (blockDim.x >> 6);
    const long wave = (long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const long ngroups = (n + 63) / 64;
    for (long grp = wave; grp < ngroups; grp += nwaves) {
        const long q = grp * 64 + lane_id();
        float x[kMlpIn];
#pragma unroll
        for (int k = 0; k < kMlpIn; ++k) x[k] = q < n ? X[q * kMlpIn + k] : 0.0f;
        float y0 = 0.0f, y1 = 0.0f;
        infer64_lds(net, x, y0, y1);
        if (q < n) {
            Y[q * kMlpOut] = y0;
            Y[q * kMlpOut + 1] = y1;
        }
    }
}

__global__ __launch_bounds__(256) void k_closure_features(FeatureArgs a, long n) {
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const GradIn gi{{a.dU[0], a.dU[1], a.dU[2]}, {a.dV[0], a.dV[1], a.dV[2]}, {a.dW[0], a.dW[1], a.dW[2]}, a.m};
    double A[3][3];
    cart_grad(gi, p, A);
    float f[kMlpIn];
    double Smag;
    const double vol_J = a.vol / a.m.J[p];
    features(A, vol_J, f, Smag);
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) __builtin_nontemporal_store((double)f[k], a.feat[k] + p);
    if (a.smag) {
        const double d = cbrt(vol_J);
        __builtin_nontemporal_store(Smag, a.smag + p);
        __builtin_nontemporal_store(d * d, a.delta2 + p);
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_learned_sgs(ClosureArgs a, long n) {
    __shared__ __attribute__((aligned(16))) InferLds net;
    // the input range and standardisation in LDS: read per group instead of
    // held in scalar registers, which spilled to vector-register lanes
    __shared__ MlpScaling sc;
    if (threadIdx.x < sizeof(MlpScaling) / sizeof(float))
        reinterpret_cast<float *>(&sc)[threadIdx.x] = reinterpret_cast<const float *>(&a.sc)[threadIdx.x];
    stage_infer(a.params, net);
    __shared__ int wcount[4];
    const int l = lane_id(), w = threadIdx.x >> 6;
    const long nwaves = (long)gridDim.x * 4;
    const long ngroups = (n + 63) / 64;
    const GradIn gi{{a.dU[0], a.dU[1], a.dU[2]}, {a.dV[0], a.dV[1], a.dV[2]}, {a.dW[0], a.dW[1], a.dW[2]}, a.m};
    int count = 0;
    for (long grp = (long)blockIdx.x * 4 + w; grp < ngroups; grp += nwaves) {
        const long p = grp * 64 + l;
        const bool live = p < n;
        float x[kMlpIn];
        double base = 0.0;
        bool out = false;
        if (live) {
            float f[kMlpIn];
            double Smag, d2;
            if (a.feat[0]) {  // averaged inputs; |S| and Delta^2 of the point from the feature pass
#pragma unroll
                for (int k = 0; k < kMlpIn; ++k) f[k] = (float)a.feat[k][p];
                Smag = a.smag[p];
                d2 = a.delta2[p];
            } else {
                double A[3][3];
                cart_grad(gi, p, A);
                const double vol_J = a.vol / a.m.J[p];
                features(A, vol_J, f, Smag);
                const double d = cbrt(vol_J);
                d2 = d * d;
            }
#pragma unroll
            for (int k = 0; k < kMlpIn; ++k) {
                const bool in = f[k] >= sc.lo[k] && f[k] <= sc.hi[k];
                out = out || !in;
                // outside the trusted range the input is clamped to it
                const float fc = in ? f[k] : (f[k] < sc.lo[k] ? sc.lo[k] : sc.hi[k]);
                x[k] = (fc - sc.in_mean[k]) / sc.in_std[k];
            }
            base = (a.rho[p] * d2) * Smag;
        } else {
#pragma unroll
            for (int k = 0; k < kMlpIn; ++k) x[k] = 0.0f;
        }
        float y0 = 0.0f, y1 = 0.0f;
        infer64_lds(net, x, y0, y1);
        if (live) {
            const float C = y0 * sc.out_std[0] + sc.out_mean[0];
            const float D = y1 * sc.out_std[1] + sc.out_mean[1];
            a.mu_sgs[p] = base * (double)C;
            a.k_sgs[p] = (a.cp * base) * (double)D;
            a.flag[p] = out ? 1 : 0;
        }
        count += __popcll(__ballot(live && out));
    }
    if (l == 0) wcount[w] = count;
    __syncthreads();
    if (threadIdx.x == 0) a.blockcount[blockIdx.x] = ((wcount[0] + wcount[1]) + wcount[2]) + wcount[3];
}

// the network on lines (LineClosureArgs); the clamp, standardisation and
// de-standardisation of k_learned_sgs
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_line_closure(LineClosureArgs a) {
    __shared__ __attribute__((aligned(16))) InferLds net;
    stage_infer(a.params, net);
    __shared__ int wcount[4];
    const int l = lane_id(), w = threadIdx.x >> 6;
    const long nwaves = (long)gridDim.x * 4;
    const long ngroups = (a.nlines + 63) / 64;
    int count = 0;
    for (long grp = (long)blockIdx.x * 4 + w; grp < ngroups; grp += nwaves) {
        const long q = grp * 64 + l;
        const bool live = q < a.nlines;
        float x[kMlpIn];
        bool out = false;
#pragma unroll
        for (int k = 0; k < kMlpIn; ++k) {
            const float f = live ? (float)a.feat[k][q] : 0.0f;
            const bool in = f >= a.sc.lo[k] && f <= a.sc.hi[k];
            out = out || !in;
            const float fc = in ? f : (f < a.sc.lo[k] ? a.sc.lo[k] : a.sc.hi[k]);
            x[k] = live ? (fc - a.sc.in_mean[k]) / a.sc.in_std[k] : 0.0f;
        }
        float y0 = 0.0f, y1 = 0.0f;
        infer64_lds(net, x, y0, y1);
        if (live) {
            a.C[q] = y0 * a.sc.out_std[0] + a.sc.out_mean[0];
            a.D[q] = y1 * a.sc.out_std[1] + a.sc.out_mean[1];
            a.lflag[q] = out ? 1 : 0;
        }
        count += __popcll(__ballot(live && out));
    }
    if (l == 0) wcount[w] = count;
    __syncthreads();
    if (threadIdx.x == 0) a.blockcount[blockIdx.x] = (((wcount[0] + wcount[1]) + wcount[2]) + wcount[3]) * a.line_len;
}

__global__ __launch_bounds__(256) void k_closure_apply(ClosureApplyArgs a, long n) {
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const long q = xi_line_of(p, a.dir, a.Nx, a.Ny);
    const double base = (ldnt(a.rho, p) * ldnt(a.delta2, p)) * ldnt(a.smag, p);
    stnt(a.mu_sgs, p, base * (double)a.C[q]);
    stnt(a.k_sgs, p, (a.cp * base) * (double)a.D[q]);
    a.flag[p] = a.lflag[q];
}

__global__ void k_count_sum(const int *__restrict__ bc, int nb, int *__restrict__ count) {
    __shared__ int part[256];
    int acc = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) acc += bc[b];
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) count[0] = part[0];
}

__global__ void k_closure_fallback(FallbackArgs a, long n) {
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || !a.flag[p]) return;
    a.mu_sgs[p] = a.mu_dsm[p];
    a.k_sgs[p] = a.k_dsm[p];
}

__global__ void k_closure_samples(SampleArgs a) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.count) return;
    const long p = a.offset + i * a.stride;
    const GradIn gi{{a.dU[0], a.dU[1], a.dU[2]}, {a.dV[0], a.dV[1], a.dV[2]}, {a.dW[0], a.dW[1], a.dW[2]}, a.m};
    float f[kMlpIn];
    if (a.feat[0]) {
#pragma unroll
        for (int k = 0; k < kMlpIn; ++k) f[k] = (float)a.feat[k][p];
    } else {
        double A[3][3];
        cart_grad(gi, p, A);
        double Smag;
        features(A, a.vol / a.m.J[p], f, Smag);
    }
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) a.X[i * kMlpIn + k] = f[k];
    const double C = a.C[p];
    a.T[i * kMlpOut] = (float)C;
    a.T[i * kMlpOut + 1] = (float)(C / a.Prt[p]);
}

}  // namespace

hipError_t launch_closure_features(const FeatureArgs &a, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_closure_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, n);
    return hipGetLastError();
}

hipError_t launch_mlp_grad_partials(const float *params, const float *X, const float *T, const int *idx, long n,
                                    long n_total, float *partial, float *lossp, hipStream_t st) {
    if (n <= 0) return hipErrorInvalidValue;
    const unsigned nb = (unsigned)((n + kT - 1) / kT);
    const float scale = (float)(2.0 / ((double)n_total * kMlpOut));
    hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(256), 0, st, params, X, T, idx, n, scale, partial, lossp);
    return hipGetLastError();
}

hipError_t launch_mlp_reduce(const float *partial, const float *lossp, int nblocks, long n_total, float *grad,
                             float *loss, hipStream_t st) {
    const float inv_norm = (float)(1.0 / ((double)n_total * kMlpOut));
    hipLaunchKernelGGL(k_mlp_reduce<false>, dim3((kMlpParams + kReduceCols - 1) / kReduceCols), dim3(512), 0, st,
                       partial, lossp, nblocks, inv_norm, grad, loss, nullptr, nullptr, nullptr, AdamArgs{});
    return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(const float *partial, const float *lossp, int nblocks, long n_total, float *loss,
                                  float *params, float *m, float *v, AdamArgs a, hipStream_t st) {
    const float inv_norm = (float)(1.0 / ((double)n_total * kMlpOut));
    hipLaunchKernelGGL(k_mlp_reduce<true>, dim3((kMlpParams + kReduceCols - 1) / kReduceCols), dim3(512), 0, st,
                       partial, lossp, nblocks, inv_norm, nullptr, loss, params, m, v, a);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float *params, float *m, float *v, const float *grad, AdamArgs a, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + 255) / 256), dim3(256), 0, st, params, m, v, grad, a);
    return hipGetLastError();
}

hipError_t launch_mlp_infer(const float *params, const float *X, float *Y, long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const long groups = (n + 63) / 64;
    const unsigned nb = (unsigned)std::min<long>((groups + 3) / 4, 2048);
    hipLaunchKernelGGL(k_mlp_infer, dim3(nb), dim3(256), 0, st, params, X, Y, n);
    return hipGetLastError();
}

int closure_blocks(long n) {
    const long groups = (n + 63) / 64;
    return (int)std::max<long>(1, std::min<long>((groups + 3) / 4, 2048));
}

int line_closure_blocks(long nlines) { return closure_blocks(nlines); }

hipError_t launch_line_closure(const LineClosureArgs &a, hipStream_t st) {
    if (a.nlines < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_line_closure, dim3((unsigned)line_closure_blocks(a.nlines)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_closure_apply(const ClosureApplyArgs &a, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_closure_apply, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, n);
    return hipGetLastError();
}

hipError_t launch_learned_sgs(const ClosureArgs &a, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_learned_sgs, dim3((unsigned)closure_blocks(n)), dim3(256), 0, st, a, n);
    return hipGetLastError();
}

hipError_t launch_count_sum(const int *blockcount, int nb, int *count, hipStream_t st) {
    hipLaunchKernelGGL(k_count_sum, dim3(1), dim3(256), 0, st, blockcount, nb, count);
    return hipGetLastError();
}

hipError_t launch_closure_fallback(const FallbackArgs &a, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_closure_fallback, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, n);
    return hipGetLastError();
}

hipError_t launch_closure_samples(const SampleArgs &a, hipStream_t st) {
    if (a.count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_closure_samples, dim3((unsigned)((a.count + 255) / 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace mc3d
