// muca_mlp.hip -- the weight surrogate: an MLP 4 -> 128 -> 128 -> 128 -> 1
// (SiLU) that predicts ln W(D)/N from (D/N, 1/L, beta, Delta) features, trained
// on converged weights and used to seed new weight runs (the init-weight
// boundary of multigpu_weight's `continuing` mode, muca_delta_multigpu.cu:223-235).
//
// Arithmetic: FP32 master parameters; every product uses BF16-rounded
// weights; the two 128 x 128 layers (forward, input-gradient and weight-
// gradient products) run on MFMA (v_mfma_f32_32x32x16_bf16) with BF16
// operands (activations and weights) and FP32 accumulation.  The 4-wide input
// layer and the 128 -> 1 output layer are VALU work in FP32 with BF16-rounded
// weights.  Adam on the FP32 masters.
//
// Training: one workgroup (1024 lanes = 16 wavefronts) owns a tile of 64 samples
// and runs the forward and the backward pass entirely in LDS; its parameter
// gradients go to its own slot of a partial-gradient buffer, which a second
// kernel sums in a fixed order (deterministic) before the Adam step.
// Prediction: 256 lanes own 32 samples.
#include "../../include/muca.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

namespace {

constexpr int kH = 128;           // hidden width
constexpr int kIn = 4;            // input features
constexpr int kTile = 64;         // samples per training workgroup
constexpr int kTrainThreads = 1024;
constexpr int kPredTile = 32;     // samples per prediction workgroup
constexpr int kPredThreads = 256;
// LDS row strides: 16-byte reads of 32 rows, and float accesses of four rows
// apart, fall on different banks
constexpr int kP = kH + 8;        // bf16
constexpr int kF = kH + 4;        // float

// parameter vector layout (FP32 masters, gradients, Adam moments)
constexpr int oW1 = 0;                       // [128][4]
constexpr int oB1 = oW1 + kH * kIn;          // [128]
constexpr int oW2 = oB1 + kH;                // [128][128], W2[o][k]
constexpr int oB2 = oW2 + kH * kH;
constexpr int oW3 = oB2 + kH;
constexpr int oB3 = oW3 + kH * kH;
constexpr int oW4 = oB3 + kH;                // [128]
constexpr int oB4 = oW4 + kH;                // [1]
constexpr int kParams = oB4 + 1;             // 33793

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// float -> bf16 bits, round to nearest even (inputs are finite)
__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t b)
{
    const uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

__device__ inline float silu(float z)
{
    return z / (1.0f + expf(-z));
}

// a = silu(z) = z / q and d = silu'(z) = s (1 + z (1 - s)), s = 1 / q, with
// q = 1 + exp(-z).  Both quotients come from one reciprocal, refined once, and
// a residual correction each; for 1e-30 < |z| < 80 they equal the divisions'
// results (correctly rounded) for every float z, in 8 instructions instead of
// about 20 (division by a refined reciprocal and the residual's correction:
// P. W. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", IBM J. Res. Develop. 34 (1990) 111); k_silu_check
// compares every float.  Outside, they are divided.
__device__ inline void silu_both(float z, float &a, float &d)
{
    const float q = 1.0f + expf(-z);
    float y = __builtin_amdgcn_rcpf(q);
    y = __builtin_fmaf(__builtin_fmaf(-q, y, 1.0f), y, y);
    float s = __builtin_fmaf(__builtin_fmaf(-q, y, 1.0f), y, y);
    const float t = z * y;
    a = __builtin_fmaf(__builtin_fmaf(-q, t, z), y, t);
    const bool plain = fabsf(z) > 1e-30f && fabsf(z) < 80.0f;
    if (__builtin_amdgcn_ballot_w64(!plain)) {
        if (!plain) {
            a = z / q;
            s = 1.0f / q;
        }
    }
    d = s * (1.0f + z * (1.0f - s));
}

// differing[0] counts the floats z = bits 0 .. 2^32 - 1 at which silu_both is not
// what divisions give (bits compared, any NaN equal to any), differing[1] keeps
// one of them
__global__ __launch_bounds__(256) void k_silu_check(uint64_t *differing)
{
    const uint64_t step = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < 1ull << 32; i += step) {
        const float z = __uint_as_float((uint32_t)i);
        float a, d;
        silu_both(z, a, d);
        const float s = 1.0f / (1.0f + expf(-z));
        const float ra = z / (1.0f + expf(-z)), rd = s * (1.0f + z * (1.0f - s));
        const bool same_a = __float_as_uint(a) == __float_as_uint(ra) || (a != a && ra != ra);
        const bool same_d = __float_as_uint(d) == __float_as_uint(rd) || (d != d && rd != rd);
        if (!same_a || !same_d) {
            atomicAdd((unsigned long long *)&differing[0], 1ull);
            differing[1] = i;
        }
    }
}

// BF16 copies of the weights used by the products.  The square ones are kept as
// the B operands of a product's output tiles (frag_at): w2 and w3 for columns
// o summed over k (forward), w2t and w3t for columns k summed over o.
struct MlpBf16 {
    uint16_t *w1;    // [128][4]
    uint16_t *w2, *w2t;
    uint16_t *w3, *w3t;
    uint16_t *w4;    // [128]
};

// place of B(k, c): tile c / 32, step k / 16, lane 32 ((k / 8) % 2) + c % 32,
// element k % 8, so that a wavefront reads a step's operands as one kilobyte
__device__ inline int frag_at(int c, int k)
{
    return (((c >> 5) * (kH / 16) + (k >> 4)) * 64 + ((k >> 3) & 1) * 32 + (c & 31)) * 8 + (k & 7);
}

// the BF16 copies of parameter i
__device__ inline void put_bf16(const MlpBf16 &wb, int i, float v)
{
    const uint16_t h = f2bf(v);
    if (i < oB1) {
        wb.w1[i - oW1] = h;
    } else if (i >= oW2 && i < oB2) {
        const int o = (i - oW2) / kH, k = (i - oW2) % kH;
        wb.w2[frag_at(o, k)] = h;
        wb.w2t[frag_at(k, o)] = h;
    } else if (i >= oW3 && i < oB3) {
        const int o = (i - oW3) / kH, k = (i - oW3) % kH;
        wb.w3[frag_at(o, k)] = h;
        wb.w3t[frag_at(k, o)] = h;
    } else if (i >= oW4 && i < oB4) {
        wb.w4[i - oW4] = h;
    }
}

struct TileArgs {
    const float *x;        // [n][4]
    const float *t;        // [n] targets (training)
    const float *w;        // [n] sample weights of the squared error (nullable: 1)
    float *y;              // [n] predictions (nullable)
    const float *p;        // FP32 parameters (biases are read from here)
    MlpBf16 wb;
    float *part;           // [tiles][kParams + 1] partial gradients and loss
    uint32_t n;            // samples
    float dy_scale;        // 2 / batch
};

// 32 x 32 output tiles of a wavefront, C(r, c) = sum_k A(r, k) B(k, c) in steps
// of 16.  Lane l supplies A(r0 + l % 32, k0 + 8 (l / 32) + 0..7) and
// B(k0 + 8 (l / 32) + 0..7, c0 + l % 32); it receives C rows
// 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32, for i = 0..15.
__device__ inline int tile_row(int i)
{
    return 8 * (i >> 2) + 4 * ((threadIdx.x & 63) >> 5) + (i & 3);
}

__device__ inline int tile_col()
{
    return threadIdx.x & 31;
}

__device__ inline f32x16 mma_step(f32x16 acc, u16x8 a, u16x8 b)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

__device__ inline f32x16 zero16()
{
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.0f;
    return z;
}

// the B operands of output tile c0 / 32
struct WFrag {
    u16x8 v[kH / 16];
};

__device__ inline WFrag load_w(const uint16_t *w, int c0)
{
    const uint16_t *q = w + ((c0 >> 5) * (kH / 16) * 64 + (threadIdx.x & 63)) * 8;
    WFrag f;
#pragma unroll
    for (int i = 0; i < kH / 16; i++) f.v[i] = *(const u16x8 *)(q + i * 64 * 8);
    return f;
}

// rows r0.. of x (LDS, stride kP) times the weights f
__device__ inline f32x16 mma_rows(const uint16_t *x, int r0, const WFrag &f)
{
    const int lane = threadIdx.x & 63;
    const uint16_t *q = x + (r0 + (lane & 31)) * kP + (lane >> 5) * 8;
    f32x16 acc = zero16();
#pragma unroll
    for (int i = 0; i < kH / 16; i++) acc = mma_step(acc, *(const u16x8 *)(q + 16 * i), f.v[i]);
    return acc;
}

// 64 x 32 sums over the tile's samples s of p[s][o0 + .] q[s][k0 + .] (LDS,
// stride kP), to out[o][k] (stride kH).  Two product tiles, of the even and
// odd columns of p: a lane reads two columns of a sample at once.
__device__ inline void mma_samples(const uint16_t *p, int o0, const uint16_t *q, int k0,
                                   float *out)
{
    const int lane = threadIdx.x & 63, rc = lane & 31, kg = (lane >> 5) * 8;
    f32x16 acc[2] = {zero16(), zero16()};
#pragma unroll
    for (int s0 = 0; s0 < kTile; s0 += 16) {
        u16x8 a[2], b;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t av = *(const uint32_t *)(p + (s0 + kg + j) * kP + o0 + 2 * rc);
            a[0][j] = (uint16_t)av;
            a[1][j] = (uint16_t)(av >> 16);
            b[j] = q[(s0 + kg + j) * kP + k0 + rc];
        }
        acc[0] = mma_step(acc[0], a[0], b);
        acc[1] = mma_step(acc[1], a[1], b);
    }
#pragma unroll
    for (int e = 0; e < 2; e++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            out[(o0 + 2 * tile_row(i) + e) * kH + k0 + rc] = acc[e][i];
}

// z1 of unit k in the order j = 0..3
__device__ inline float layer1(float b1, const float *w1, const float *x)
{
    float z = b1;
#pragma unroll
    for (int j = 0; j < kIn; j++) z = z + w1[j] * x[j];
    return z;
}

// One tile of training: forward and backward.  Bound by the activations'
// VALU work (an exponential and two divisions per unit, sample and layer) on
// the compute unit that owns the tile, so it is spread over sixteen
// wavefronts: lane t works unit t % 128 of samples t / 128 + 8 i, each
// derivative is made together with its activation, and the products (eight
// wavefronts each, weights loaded a phase ahead) run beside the sums over
// samples.  Every sum keeps one order: products over k, or over the tile's
// samples, in steps of 16; sums over samples one by one.  Batch 4096: 20.6
// us for a step's tiles against 43.4 us with four wavefronts, whose lanes made
// the sums over samples and their activations serially; the Adam kernel's
// sums with sixteen loads in flight 4.7 against 17.6 us.
__global__ __launch_bounds__(kTrainThreads) void k_mlp_tile(TileArgs g)
{
    __shared__ __attribute__((aligned(16))) uint16_t a1[kTile * kP];     // bf16 silu(z1)
    __shared__ __attribute__((aligned(16))) uint16_t a2[kTile * kP];     // bf16 silu(z2)
    __shared__ __attribute__((aligned(16))) uint16_t dz3b[kTile * kP];   // bf16 dz3
    __shared__ float f2[kTile * kF];     // z2, then silu'(z2), then dz2
    __shared__ float f3[kTile * kF];     // z3, then silu'(z3), then dz3, then dz1
    __shared__ __attribute__((aligned(16))) float a3[kTile * kF];   // silu(z3); then bf16 dz2
    __shared__ float xs[kTile][kIn];
    __shared__ float ts[kTile], dys[kTile];
    __shared__ float red[4 * kTile];
    __shared__ float sq[kTile];          // squared errors
    __shared__ float w4s[kH];
    uint16_t *const dz2b = (uint16_t *)a3;

    const int tid = threadIdx.x, wave = tid >> 6;
    const uint32_t s0 = blockIdx.x * kTile;
    const float *P = g.p;
    const int k = tid & (kH - 1), sr = tid >> 7;   // this lane's unit and first sample
    constexpr int kS = kTrainThreads / kH;         // its samples' distance
    // product tile of wavefronts 0..7 and 8..15
    const int r0 = 32 * (wave & 1), c0 = 32 * ((wave >> 1) & 3);
    const bool lower = wave < 8;

    // everything the phases read from memory, loaded before the first one
    // (the step before has just written it: the loads miss the L2)
    const int cc = c0 + tile_col();   // this lane's column of a product tile
    const float b1 = P[oB1 + k], b23 = P[(lower ? oB2 : oB3) + cc], b4 = P[oB4];
    const float w4 = bf2f(g.wb.w4[k]);
    float w1[kIn];
#pragma unroll
    for (int j = 0; j < kIn; j++) w1[j] = bf2f(g.wb.w1[k * kIn + j]);
    WFrag wf = load_w(lower ? g.wb.w2 : g.wb.w3, c0);
    const bool valid = tid < kTile && s0 + tid < g.n;
    const float wt = (valid && g.w) ? g.w[s0 + tid] : 1.0f;
    if (tid < kTile * kIn) {
        const int s = tid / kIn, j = tid % kIn;
        xs[s][j] = (s0 + s < g.n) ? g.x[(uint64_t)(s0 + s) * kIn + j] : 0.0f;
    }
    if (tid < kTile) ts[tid] = valid ? g.t[s0 + tid] : 0.0f;
    if (sr == 0) w4s[k] = w4;
    __syncthreads();

    // layer 1 (VALU)
    constexpr int kN = kTile / kS;   // samples per lane
    float d1[kN];                    // silu'(z1)
#pragma unroll
    for (int i = 0; i < kN; i++) {
        const int s = sr + kS * i;
        float a;
        silu_both(layer1(b1, w1, xs[s]), a, d1[i]);
        a1[s * kP + k] = f2bf(a);
    }
    __syncthreads();
    // layer 2 (MFMA)
    if (lower) {
        const f32x16 acc = mma_rows(a1, r0, wf);
#pragma unroll
        for (int i = 0; i < 16; i++) f2[(r0 + tile_row(i)) * kF + cc] = acc[i] + b23;
        wf = load_w(g.wb.w3t, c0);   // for da2
    }
    __syncthreads();
#pragma unroll 2
    for (int s = sr; s < kTile; s += kS) {
        float a, d;
        silu_both(f2[s * kF + k], a, d);
        a2[s * kP + k] = f2bf(a);
        f2[s * kF + k] = d;
    }
    __syncthreads();
    // layer 3 (MFMA)
    if (!lower) {
        const f32x16 acc = mma_rows(a2, r0, wf);
#pragma unroll
        for (int i = 0; i < 16; i++) f3[(r0 + tile_row(i)) * kF + cc] = acc[i] + b23;
        wf = load_w(g.wb.w2t, c0);   // for da1
    }
    __syncthreads();
#pragma unroll 2
    for (int s = sr; s < kTile; s += kS) {
        float a, d;
        silu_both(f3[s * kF + k], a, d);
        a3[s * kF + k] = a;
        f3[s * kF + k] = d;
    }
    __syncthreads();
    // output layer (VALU): y = b4 + sum_k w4[k] silu(z3[k]); four lanes per
    // sample each sum 32 consecutive k, then the four partials in order
    if (tid < 4 * kTile) {
        const int s = tid >> 2, q = tid & 3;
        float acc = 0.0f;
#pragma unroll 8
        for (int i = 32 * q; i < 32 * q + 32; i++) acc = acc + w4s[i] * a3[s * kF + i];
        red[tid] = acc;
    }
    __syncthreads();
    if (tid < kTile) {
        const float y = b4 + (((red[4 * tid] + red[4 * tid + 1]) + red[4 * tid + 2]) +
                              red[4 * tid + 3]);
        const float d = y - ts[tid];
        dys[tid] = valid ? g.dy_scale * (wt * d) : 0.0f;
        sq[tid] = valid ? wt * (d * d) : 0.0f;
    }
    __syncthreads();
    // dz3 = dy w4 silu'(z3)
#pragma unroll
    for (int s = sr; s < kTile; s += kS) {
        const float dz = (dys[s] * w4) * f3[s * kF + k];
        f3[s * kF + k] = dz;
        dz3b[s * kP + k] = f2bf(dz);
    }
    __syncthreads();
    float *part = g.part + (uint64_t)blockIdx.x * (kParams + 1);
    // sums over the tile's samples, in order
    auto column = [&](const float *f, int c) {
        float v = 0.0f;
#pragma unroll 16
        for (int s = 0; s < kTile; s++) v = v + f[s * kF + c];
        return v;
    };
    if (lower) {
        // da2[s][k] = sum_o dz3[s][o] W3[o][k]; dz2 = da2 silu'(z2)
        const f32x16 acc = mma_rows(dz3b, r0, wf);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float *q = f2 + (r0 + tile_row(i)) * kF + cc;
            *q = acc[i] * *q;
        }
        if (wave < 2) {           // db3[k] = sum_s dz3
            part[oB3 + k] = column(f3, k);
        } else if (wave < 4) {    // dw4[k] = sum_s dy[s] silu(z3[s][k])
            float dw = 0.0f;
#pragma unroll 16
            for (int s = 0; s < kTile; s++) dw = dw + dys[s] * a3[s * kF + k];
            part[oW4 + k] = dw;
        }
    } else {   // dW3[o][k] = sum_s dz3[s][o] a2[s][k]
        mma_samples(dz3b, 64 * ((wave >> 2) & 1), a2, 32 * (wave & 3), part + oW3);
    }
    __syncthreads();
#pragma unroll
    for (int s = sr; s < kTile; s += kS) dz2b[s * kP + k] = f2bf(f2[s * kF + k]);
    __syncthreads();
    if (lower) {   // dW2[o][k] = sum_s dz2[s][o] a1[s][k]
        mma_samples(dz2b, 64 * (wave >> 2), a1, 32 * (wave & 3), part + oW2);
    } else {
        // da1[s][k] = sum_o dz2[s][o] W2[o][k]
        const f32x16 acc = mma_rows(dz2b, r0, wf);
#pragma unroll
        for (int i = 0; i < 16; i++) f3[(r0 + tile_row(i)) * kF + cc] = acc[i];
        if (wave < 10) {
            part[oB2 + k] = column(f2, k);   // db2
        } else if (tid == 10 * 64) {         // loss and db4
            float l = 0.0f, db = 0.0f;
#pragma unroll 16
            for (int s = 0; s < kTile; s++) {
                l = l + sq[s];
                db = db + dys[s];
            }
            part[kParams] = l;
            part[oB4] = db;
        }
    }
    __syncthreads();
    // dz1 = da1 silu'(z1)
#pragma unroll
    for (int i = 0; i < kN; i++) {
        float *q = f3 + (sr + kS * i) * kF + k;
        *q = *q * d1[i];
    }
    __syncthreads();
    // db1[k] = sum_s dz1[s][k]; dW1[k][j] = sum_s dz1[s][k] x[s][j]
    if (sr == 4) {
        part[oB1 + k] = column(f3, k);
    } else if (sr < kIn) {
        float dw = 0.0f;
#pragma unroll 16
        for (int s = 0; s < kTile; s++) dw = dw + f3[s * kF + k] * xs[s][sr];
        part[oW1 + k * kIn + sr] = dw;
    }
}

// Predictions of 32 samples per workgroup: the forward pass above, with the
// same operations in the same order for each sample.  Small tiles so that
// several workgroups share a compute unit and a few thousand samples reach
// all of them: 16 385 samples 13.7 us against 22.0 with the training tile.
__global__ __launch_bounds__(kPredThreads) void k_mlp_predict(TileArgs g)
{
    __shared__ __attribute__((aligned(16))) uint16_t a1[kPredTile * kP];
    __shared__ __attribute__((aligned(16))) uint16_t a2[kPredTile * kP];
    __shared__ float a3[kPredTile * kF];
    __shared__ float xs[kPredTile][kIn];
    __shared__ float w4s[kH];
    const int tid = threadIdx.x, wave = tid >> 6;
    const uint32_t s0 = blockIdx.x * kPredTile;
    const float *P = g.p;
    const int c = 32 * wave + tile_col();   // this lane's column of a product tile
    const int k = tid & (kH - 1);
    const float b1 = P[oB1 + k], b2 = P[oB2 + c], b3 = P[oB3 + c], b4 = P[oB4];
    float w1[kIn];
#pragma unroll
    for (int j = 0; j < kIn; j++) w1[j] = bf2f(g.wb.w1[k * kIn + j]);
    const WFrag w2 = load_w(g.wb.w2, 32 * wave), w3 = load_w(g.wb.w3, 32 * wave);
    if (tid < kH) w4s[tid] = bf2f(g.wb.w4[tid]);
    if (tid < kPredTile * kIn) {
        const int s = tid / kIn, j = tid % kIn;
        xs[s][j] = (s0 + s < g.n) ? g.x[(uint64_t)(s0 + s) * kIn + j] : 0.0f;
    }
    __syncthreads();
#pragma unroll 4
    for (int s = tid >> 7; s < kPredTile; s += kPredThreads / kH)
        a1[s * kP + k] = f2bf(silu(layer1(b1, w1, xs[s])));
    __syncthreads();
    {
        const f32x16 acc = mma_rows(a1, 0, w2);
#pragma unroll
        for (int i = 0; i < 16; i++) a2[tile_row(i) * kP + c] = f2bf(silu(acc[i] + b2));
    }
    __syncthreads();
    {
        const f32x16 acc = mma_rows(a2, 0, w3);
#pragma unroll
        for (int i = 0; i < 16; i++) a3[tile_row(i) * kF + c] = silu(acc[i] + b3);
    }
    __syncthreads();
    if (tid < 4 * kPredTile) {
        const int s = tid >> 2, q = tid & 3;
        float acc = 0.0f;
#pragma unroll 8
        for (int i = 32 * q; i < 32 * q + 32; i++) acc = acc + w4s[i] * a3[s * kF + i];
        // the four partials of a sample in order
        const float p1 = __shfl_down(acc, 1, 4), p2 = __shfl_down(acc, 2, 4),
                    p3 = __shfl_down(acc, 3, 4);
        if (q == 0 && s0 + s < g.n) g.y[s0 + s] = b4 + (((acc + p1) + p2) + p3);
    }
}

// Sums the tiles' partial gradients in tile order; optionally takes one Adam
// step and refreshes the BF16 copies.
__global__ __launch_bounds__(256) void k_mlp_reduce(const float *part, uint32_t tiles, float *grad,
                                                   float *loss, float *p, float *m, float *v,
                                                   MlpBf16 wb, int adam, float lr, float b1,
                                                   float b2, float eps, float c1, float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > kParams) return;
    // sixteen loads in flight, added in tile order
    float gsum = 0.0f;
    const float *q = part + i;
    uint32_t t = 0;
    for (; t + 16 <= tiles; t += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = q[(uint64_t)(t + u) * (kParams + 1)];
#pragma unroll
        for (int u = 0; u < 16; u++) gsum = gsum + v[u];
    }
    for (; t < tiles; t++) gsum = gsum + q[(uint64_t)t * (kParams + 1)];
    if (i == kParams) {
        if (loss) *loss = gsum;
        return;
    }
    if (grad) grad[i] = gsum;
    if (!adam) return;
    const float mi = b1 * m[i] + (1.0f - b1) * gsum;
    const float vi = b2 * v[i] + (1.0f - b2) * gsum * gsum;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    put_bf16(wb, i, pi);
}

__global__ void k_mlp_refresh_bf16(const float *p, MlpBf16 wb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kParams) return;
    put_bf16(wb, i, p[i]);
}

thread_local std::string g_merr;

int mfail(int code, const std::string &m)
{
    g_merr = m;
    return code;
}

#define MHIP(expr)                                                                      \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess)                                                           \
            return mfail(MUCA_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

}  // namespace

struct muca_mlp {
    int device = 0;
    hipStream_t st = nullptr;
    float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr, *loss = nullptr;
    float *part = nullptr;
    uint32_t part_tiles = 0;
    uint16_t *bf = nullptr;   // all BF16 copies in one allocation
    MlpBf16 wb{};
    float *x = nullptr, *t = nullptr, *y = nullptr;   // resident training data / scratch
    float *w = nullptr;                               // resident sample weights
    bool weighted = false;
    uint32_t n = 0, cap = 0;
    uint64_t step = 0;
};

namespace {

void mlp_free(muca_mlp *g)
{
    if (!g) return;
    (void)hipSetDevice(g->device);
    void *bufs[] = {g->p, g->m, g->v, g->grad, g->loss, g->part, g->bf, g->x, g->t, g->y, g->w};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    if (g->st) (void)hipStreamDestroy(g->st);
    delete g;
}

hipError_t ensure_part(muca_mlp *g, uint32_t tiles)
{
    if (tiles <= g->part_tiles) return hipSuccess;
    if (g->part) (void)hipFree(g->part);
    g->part = nullptr;
    g->part_tiles = 0;
    hipError_t e = hipMalloc((void **)&g->part, (size_t)tiles * (kParams + 1) * sizeof(float));
    if (e == hipSuccess) g->part_tiles = tiles;
    return e;
}

hipError_t ensure_data(muca_mlp *g, uint32_t n)
{
    if (n <= g->cap) return hipSuccess;
    for (float **b : {&g->x, &g->t, &g->y, &g->w})
        if (*b) {
            (void)hipFree(*b);
            *b = nullptr;
        }
    g->cap = 0;
    hipError_t e = hipMalloc((void **)&g->x, (size_t)n * kIn * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->t, (size_t)n * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->y, (size_t)n * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->w, (size_t)n * sizeof(float));
    if (e == hipSuccess) g->cap = n;
    return e;
}

TileArgs tile_args(muca_mlp *g, const float *x, const float *t, const float *w, float *y,
                   uint32_t n, float dy_scale)
{
    TileArgs a{};
    a.x = x;
    a.t = t;
    a.w = w;
    a.y = y;
    a.p = g->p;
    a.wb = g->wb;
    a.part = g->part;
    a.n = n;
    a.dy_scale = dy_scale;
    return a;
}

}  // namespace

extern "C" {

const char *muca_mlp_last_error(void)
{
    return g_merr.c_str();
}

uint32_t muca_mlp_param_count(void)
{
    return kParams;
}

int muca_mlp_create(int32_t device, muca_mlp **out)
{
    if (!out) return mfail(MUCA_E_ARG, "NULL output");
    *out = nullptr;
    int ndev = 0;
    MHIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return mfail(MUCA_E_ARG, "device not present");
    MHIP(hipSetDevice(device));
    muca_mlp *g = new muca_mlp();
    g->device = device;
    hipError_t e = hipStreamCreateWithFlags(&g->st, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc((void **)&g->p, kParams * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->m, kParams * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->v, kParams * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->grad, kParams * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&g->loss, sizeof(float));
    const size_t nbf = kH * kIn + 4 * kH * kH + kH;
    if (e == hipSuccess) e = hipMalloc((void **)&g->bf, nbf * sizeof(uint16_t));
    if (e != hipSuccess) {
        mlp_free(g);
        return mfail(MUCA_E_NOMEM, std::string("mlp setup: ") + hipGetErrorString(e));
    }
    g->wb.w1 = g->bf;
    g->wb.w2 = g->wb.w1 + kH * kIn;
    g->wb.w2t = g->wb.w2 + kH * kH;
    g->wb.w3 = g->wb.w2t + kH * kH;
    g->wb.w3t = g->wb.w3 + kH * kH;
    g->wb.w4 = g->wb.w3t + kH * kH;
    *out = g;
    return MUCA_OK;
}

int muca_mlp_silu_check(int32_t device, uint64_t *differing, uint32_t *example)
{
    if (!differing || !example) return mfail(MUCA_E_ARG, "NULL argument");
    MHIP(hipSetDevice(device));
    struct Buf {
        uint64_t *p = nullptr;
        ~Buf()
        {
            if (p) (void)hipFree(p);
        }
    } d;
    uint64_t h[2] = {0, 0};
    MHIP(hipMalloc((void **)&d.p, sizeof(h)));
    MHIP(hipMemcpy(d.p, h, sizeof(h), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_silu_check, dim3(8192), dim3(256), 0, nullptr, d.p);
    MHIP(hipGetLastError());
    MHIP(hipMemcpy(h, d.p, sizeof(h), hipMemcpyDeviceToHost));
    *differing = h[0];
    *example = (uint32_t)h[1];
    return MUCA_OK;
}

int muca_mlp_destroy(muca_mlp *g)
{
    mlp_free(g);
    return MUCA_OK;
}

int muca_mlp_set_params(muca_mlp *g, const float *params, uint32_t n)
{
    if (!g || !params || n != (uint32_t)kParams) return mfail(MUCA_E_ARG, "need kParams values");
    for (uint32_t i = 0; i < n; i++)
        if (!std::isfinite(params[i])) return mfail(MUCA_E_ARG, "parameters must be finite");
    MHIP(hipSetDevice(g->device));
    MHIP(hipMemcpy(g->p, params, kParams * sizeof(float), hipMemcpyHostToDevice));
    MHIP(hipMemsetAsync(g->m, 0, kParams * sizeof(float), g->st));
    MHIP(hipMemsetAsync(g->v, 0, kParams * sizeof(float), g->st));
    g->step = 0;
    hipLaunchKernelGGL(k_mlp_refresh_bf16, dim3((kParams + 255) / 256), dim3(256), 0, g->st, g->p,
                       g->wb);
    MHIP(hipGetLastError());
    MHIP(hipStreamSynchronize(g->st));
    return MUCA_OK;
}

int muca_mlp_get_params(muca_mlp *g, float *params, uint32_t n)
{
    if (!g || !params || n != (uint32_t)kParams) return mfail(MUCA_E_ARG, "need kParams values");
    MHIP(hipSetDevice(g->device));
    MHIP(hipStreamSynchronize(g->st));
    MHIP(hipMemcpy(params, g->p, kParams * sizeof(float), hipMemcpyDeviceToHost));
    return MUCA_OK;
}

int muca_mlp_predict(muca_mlp *g, const float *x, uint32_t n, float *y)
{
    if (!g || !x || !y || n == 0) return mfail(MUCA_E_ARG, "bad arguments");
    MHIP(hipSetDevice(g->device));
    MHIP(ensure_data(g, n));
    MHIP(hipMemcpy(g->x, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice));
    const uint32_t tiles = (n + kPredTile - 1) / kPredTile;
    hipLaunchKernelGGL(k_mlp_predict, dim3(tiles), dim3(kPredThreads), 0, g->st,
                       tile_args(g, g->x, nullptr, nullptr, g->y, n, 0.0f));
    MHIP(hipGetLastError());
    MHIP(hipStreamSynchronize(g->st));
    MHIP(hipMemcpy(y, g->y, (size_t)n * sizeof(float), hipMemcpyDeviceToHost));
    return MUCA_OK;
}

int muca_mlp_gradient(muca_mlp *g, const float *x, const float *t, uint32_t n, float *grad,
                      float *loss)
{
    if (!g || !x || !t || n == 0) return mfail(MUCA_E_ARG, "bad arguments");
    MHIP(hipSetDevice(g->device));
    MHIP(ensure_data(g, n));
    const uint32_t tiles = (n + kTile - 1) / kTile;
    MHIP(ensure_part(g, tiles));
    MHIP(hipMemcpy(g->x, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice));
    MHIP(hipMemcpy(g->t, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_mlp_tile, dim3(tiles), dim3(kTrainThreads), 0, g->st,
                       tile_args(g, g->x, g->t, nullptr, nullptr, n, 2.0f / (float)n));
    MHIP(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_reduce, dim3((kParams + 1 + 255) / 256), dim3(256), 0, g->st, g->part,
                       tiles, g->grad, g->loss, g->p, g->m, g->v, g->wb, 0, 0.0f, 0.0f, 0.0f, 0.0f,
                       1.0f, 1.0f);
    MHIP(hipGetLastError());
    MHIP(hipStreamSynchronize(g->st));
    if (grad) MHIP(hipMemcpy(grad, g->grad, kParams * sizeof(float), hipMemcpyDeviceToHost));
    if (loss) {
        float l = 0;
        MHIP(hipMemcpy(&l, g->loss, sizeof(float), hipMemcpyDeviceToHost));
        *loss = l / (float)n;
    }
    return MUCA_OK;
}

int muca_mlp_set_data(muca_mlp *g, const float *x, const float *t, const float *w, uint32_t n)
{
    if (!g || !x || !t || n == 0) return mfail(MUCA_E_ARG, "bad arguments");
    if (w)
        for (uint32_t i = 0; i < n; i++)
            if (!(w[i] >= 0.0f) || !std::isfinite(w[i]))
                return mfail(MUCA_E_ARG, "sample weights must be finite and >= 0");
    MHIP(hipSetDevice(g->device));
    MHIP(ensure_data(g, n));
    MHIP(hipMemcpy(g->x, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice));
    MHIP(hipMemcpy(g->t, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
    if (w) MHIP(hipMemcpy(g->w, w, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
    g->weighted = w != nullptr;
    g->n = n;
    return MUCA_OK;
}

int muca_mlp_train(muca_mlp *g, uint32_t steps, uint32_t batch, float lr, float lr_final,
                   float *loss_out, float *gpu_ms)
{
    if (!g || steps == 0 || batch == 0 || batch % kTile != 0)
        return mfail(MUCA_E_ARG, "batch must be a positive multiple of 64");
    if (g->n < batch) return mfail(MUCA_E_STATE, "set at least `batch` samples first");
    MHIP(hipSetDevice(g->device));
    const uint32_t tiles = batch / kTile;
    MHIP(ensure_part(g, tiles));
    struct Events {   // destroyed on every return path
        hipEvent_t e[2] = {nullptr, nullptr};
        ~Events()
        {
            for (hipEvent_t x : e)
                if (x) (void)hipEventDestroy(x);
        }
    } ev;
    MHIP(hipEventCreate(&ev.e[0]));
    MHIP(hipEventCreate(&ev.e[1]));
    hipEvent_t e0 = ev.e[0], e1 = ev.e[1];
    MHIP(hipEventRecord(e0, g->st));
    const uint32_t nbatches = g->n / batch;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (uint32_t s = 0; s < steps; s++) {
        // minibatches walk the resident samples in order (shuffled by the caller)
        const uint64_t off = (uint64_t)(s % nbatches) * batch;
        // cosine schedule from lr to lr_final
        const float lr_s =
            lr_final + 0.5f * (lr - lr_final) * (1.0f + cosf(3.14159265f * (float)s / (float)steps));
        g->step++;
        const float c1 = 1.0f - powf(b1, (float)g->step), c2 = 1.0f - powf(b2, (float)g->step);
        hipLaunchKernelGGL(k_mlp_tile, dim3(tiles), dim3(kTrainThreads), 0, g->st,
                           tile_args(g, g->x + off * kIn, g->t + off,
                                     g->weighted ? g->w + off : nullptr, nullptr, batch,
                                     2.0f / (float)batch));
        MHIP(hipGetLastError());
        hipLaunchKernelGGL(k_mlp_reduce, dim3((kParams + 1 + 255) / 256), dim3(256), 0, g->st,
                           g->part, tiles, nullptr, g->loss, g->p, g->m, g->v, g->wb, 1, lr_s, b1,
                           b2, eps, c1, c2);
        MHIP(hipGetLastError());
    }
    MHIP(hipEventRecord(e1, g->st));
    MHIP(hipEventSynchronize(e1));
    float ms = 0;
    MHIP(hipEventElapsedTime(&ms, e0, e1));
    if (gpu_ms) *gpu_ms = ms;
    if (loss_out) {
        float l = 0;
        MHIP(hipMemcpy(&l, g->loss, sizeof(float), hipMemcpyDeviceToHost));
        *loss_out = l / (float)batch;
    }
    return MUCA_OK;
}

}  // extern "C"
