// Learned Newton warm start (include/cmg.h, cmg_mlp_*): a per-node MLP
// 8 -> H -> H -> 3 (tanh hidden layers) that maps nodal features of the next
// Newmark step (the two previous increments, the pressure rate and the activation
// phase) to that step's displacement increment.  Hand-written gfx950 kernels for
// inference, the training pass (forward, backward and all weight gradients in one
// kernel, partial sums added in a fixed order) and Adam.  The step only uses the
// proposed guess when its residual is below the predictor's (the predictor is both
// the fallback and the yardstick).
//
// Weight layout (FP32, flat): W1[8][H] b1[H] W2[H][H] b2[H] W3[H][3] b3[3]
// (W[k][c]: input k -> output c).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "cmg_ctx.h"

using namespace cmg;

namespace {

constexpr int kH = 128;         // hidden width of the kernels
constexpr int kIn = 8;
constexpr int kOut = 3;
constexpr int kThr = 256;       // threads per workgroup
constexpr int kWaveRows = 16;   // rows of one wave's tile
constexpr int kTile = 64;       // rows of a training workgroup's tile (four waves)
constexpr int kTrainBlocks = 256;   // partial gradients: one training workgroup per CU

constexpr int64_t n_weights() { return kIn * kH + kH + kH * kH + kH + kH * kOut + kOut; }
constexpr int64_t off_b1 = kIn * kH;
constexpr int64_t off_W2 = off_b1 + kH;
constexpr int64_t off_b2 = off_W2 + kH * kH;
constexpr int64_t off_W3 = off_b2 + kH;
constexpr int64_t off_b3 = off_W3 + kH * kOut;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// All kernels hold activations transposed, H^T[c][row], in the output layout of the
// 16x16 matrix instructions: lane 16 g + i has row i and columns 16 b + 4 g + s in
// component s of register b.  Read as the second operand of the next product, that
// register s of block b is one k-step over the columns 16 b + 4 g + s of the four lane
// groups g, so the layers of a row follow each other in one wave's registers, and only
// the weights come from LDS.  Operand layouts (i, j < 16):
//   16x16x4 f32    A[i][k] lane i + 16 k,  B[k][j] lane j + 16 k
//   16x16x16 bf16  A[i][k] lane i + 16 (k / 4), B alike, item k % 4
//   16x16x32 bf16  A[i][k] lane i + 16 (k / 8), B alike, item k % 8
//   result         D[i][j] lane j + 16 (i / 4), item i % 4
// ---------------------------------------------------------------------------

// tanh for activations that are rounded to bfloat16: 1 - 2 / (e^2x + 1), and below 1/4, where
// that cancels, x + x^3 (c0 + c1 x^2) (least-squares fit of (tanh x - x) / x^3, reweighted to
// equal ripple).  Relative error at most 5.3e-7 over all single-precision numbers, against
// the rounding's 2e-3, without branches and in 17 vector operations' time; tanhf (1.5e-7)
// takes about three times that.
__device__ __forceinline__ float tanh_bf16(float x) {
    const float z = x * x;
    const float t = fmaf(-2.f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * 2.8853900817779268f) + 1.f), 1.f);
    const float p = fmaf(z, 0.12876420190194154f, -0.33324571367681377f);
    return fabsf(x) < 0.25f ? fmaf(x * z, p, x) : t;
}

// W3[c..c+3][0..2] (12 floats, 16-byte aligned)
__device__ __forceinline__ void load_w3(const float* sW3, int c, float* w3) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(sW3 + kOut * c + 4 * q);
#pragma unroll
        for (int s = 0; s < 4; s++) w3[4 * q + s] = v[s];
    }
}

// sums over the four lane groups of a row, in every one of them
__device__ __forceinline__ void sum_groups(float* y) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1)
#pragma unroll
        for (int j = 0; j < kOut; j++) y[j] += __shfl_xor(y[j], o, 64);
}

// ---------------------------------------------------------------------------
// FP32 layers of one wave's 16 rows (FP32 matrix instructions: FP32 products and sums)
// ---------------------------------------------------------------------------
constexpr int kW2Pitch = kH + 4;   // floats per LDS row of W2: W2^T reads one value per lane, W2 four, no conflicts

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// this lane's W1 operands, kept for all tiles
__device__ __forceinline__ void load_w1(const float* w, int i, int g, float (*w1)[2]) {
#pragma unroll
    for (int b = 0; b < kH / 16; b++)
#pragma unroll
        for (int k = 0; k < 2; k++) w1[b][k] = w[(4 * k + g) * kH + 16 * b + i];
}

// a1 = tanh(W1^T x + b1); x0, x1: inputs g and 4 + g of the lane's row
__device__ __forceinline__ void layer1(const float (*w1)[2], const float* sb1, int g, float x0, float x1, f32x4* a1) {
#pragma unroll
    for (int b = 0; b < kH / 16; b++) {
        f32x4 acc = *reinterpret_cast<const f32x4*>(sb1 + 16 * b + 4 * g);
        acc = mfma4(w1[b][0], x0, acc);
        acc = mfma4(w1[b][1], x1, acc);
#pragma unroll
        for (int s = 0; s < 4; s++) a1[b][s] = tanhf(acc[s]);
    }
}

// a2 = tanh(W2^T a1 + b2).  The lane's offset is hidden from the compiler, which would
// otherwise keep W2 in registers across a workgroup's tiles and spill them.
__device__ __forceinline__ void layer2(const float* sW2, const float* sb2, int i, int g, const f32x4* a1, f32x4* a2) {
    int lane = 4 * g * kW2Pitch + i;
    asm volatile("" : "+v"(lane));
#pragma unroll
    for (int n = 0; n < kH / 16; n++) a2[n] = *reinterpret_cast<const f32x4*>(sb2 + 16 * n + 4 * g);
    // the next k-step's weights are requested before this one's products (the barrier keeps the
    // compiler from moving the loads back to their use, where every pair of products waits)
    float wk[2][kH / 16];
    auto load = [&](int k) {
#pragma unroll
        for (int n = 0; n < kH / 16; n++)
            wk[k % 2][n] = sW2[lane + (16 * (k / 4) + k % 4) * kW2Pitch + 16 * n];
    };
    load(0);
#pragma unroll
    for (int k = 0; k < kH / 4; k++) {
        if (k + 1 < kH / 4) load(k + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < kH / 16; n++) a2[n] = mfma4(wk[k % 2][n], a1[k / 4][k % 4], a2[n]);
    }
#pragma unroll
    for (int n = 0; n < kH / 16; n++)
#pragma unroll
        for (int s = 0; s < 4; s++) a2[n][s] = tanhf(a2[n][s]);
}

// y = W3^T a2 of the lane's row (without the bias), in all four lane groups
__device__ __forceinline__ void layer3(const float* sW3, int g, const f32x4* a2, float* y) {
    y[0] = y[1] = y[2] = 0.f;
#pragma unroll
    for (int b = 0; b < kH / 16; b++) {
        float w3[12];
        load_w3(sW3, 16 * b + 4 * g, w3);
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int o = 0; o < kOut; o++) y[o] = fmaf(a2[b][s], w3[3 * s + o], y[o]);
    }
    sum_groups(y);
}

// ---------------------------------------------------------------------------
// forward (FP32): W2 in LDS for all tiles of a workgroup, 16 rows per wave.
// Bound by the FP32 matrix rate (2 x 128 x 128 flops per row) and the two tanh layers on the
// vector ALUs, which four waves per SIMD overlap.  290,927 rows: 139 us,
// 430 with 4 x 8 outputs per thread on the vector ALUs.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(4 * kThr) void k_mlp_forward(const float* __restrict__ w, const float* __restrict__ X,
                                                          int64_t rows, float* __restrict__ Y) {
    __shared__ __align__(16) float sW2[kH * kW2Pitch];
    __shared__ __align__(16) float sb1[kH], sb2[kH], sW3[kH * kOut];
    const int t = threadIdx.x, nt = blockDim.x;
    for (int e = 4 * t; e < kH * kH; e += 4 * nt)
        *reinterpret_cast<f32x4*>(sW2 + (e / kH) * kW2Pitch + e % kH) = *reinterpret_cast<const f32x4*>(w + off_W2 + e);
    for (int e = t; e < kH * kOut; e += nt) sW3[e] = w[off_W3 + e];
    if (t < kH) {
        sb1[t] = w[off_b1 + t];
        sb2[t] = w[off_b2 + t];
    }
    const int i = t % 16, g = (t % 64) / 16;
    float w1[kH / 16][2];
    load_w1(w, i, g, w1);
    const float b3 = g < kOut ? w[off_b3 + g] : 0.f;
    __syncthreads();
    const int64_t ntiles = (rows + kWaveRows - 1) / kWaveRows, step = (int64_t)gridDim.x * (nt / 64);
    for (int64_t tile = (int64_t)blockIdx.x * (nt / 64) + t / 64; tile < ntiles; tile += step) {
        const int64_t r = tile * kWaveRows + i;
        const bool in = r < rows;
        f32x4 a1[kH / 16], a2[kH / 16];
        float y[kOut];
        layer1(w1, sb1, g, in ? X[r * kIn + g] : 0.f, in ? X[r * kIn + 4 + g] : 0.f, a1);
        layer2(sW2, sb2, i, g, a1, a2);
        layer3(sW3, g, a2, y);
        if (in && g < kOut) Y[r * kOut + g] = (g == 0 ? y[0] : g == 1 ? y[1] : y[2]) + b3;
    }
}

// ---------------------------------------------------------------------------
// bfloat16 inference: inputs, weights and both hidden activations rounded to bfloat16,
// products and sums in FP32 on the matrix cores (layers 1 and 2) and the vector ALUs
// (layer 3).  Layer 1 has k = 8, the instruction 16: the two upper lane groups hold zeros.
// W2^T is stored in LDS with k permuted so that a lane's eight values of a 16x16x32 step,
// columns 32 p + 4 g + s and 32 p + 16 + 4 g + s, are 16 contiguous bytes.
// Bound by the 256 tanh per row (17 of the about 25 vector operations per activation).
// 290,927 rows: 40 us, 89 with layer 1 on the vector ALUs, tanhf and one k = 16 step per
// instruction.
// ---------------------------------------------------------------------------
constexpr int kW2tPitch = kH + 8;   // bf16 per row of the transposed W2 (spreads the lanes over banks)

__global__ __launch_bounds__(4 * kThr) void k_mlp_forward_bf16(const float* __restrict__ w,
                                                               const float* __restrict__ X, int64_t rows,
                                                               float* __restrict__ Y) {
    __shared__ __align__(16) __bf16 sW2t[kH * kW2tPitch];
    __shared__ __align__(16) float sb1[kH], sb2[kH], sW3[kH * kOut];
    const int t = threadIdx.x, nt = blockDim.x;
    for (int e = t; e < kH * kH / 4; e += nt) {
        const int n = e % kH, k = 4 * (e / kH);   // four values of column n
        bf16x4 v;
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = (__bf16)w[off_W2 + (k + s) * kH + n];
        const int kp = (k & ~31) + 8 * ((k % 16) / 4) + 4 * ((k / 16) % 2);
        *reinterpret_cast<bf16x4*>(sW2t + n * kW2tPitch + kp) = v;
    }
    for (int e = t; e < kH * kOut; e += nt) sW3[e] = (float)(__bf16)w[off_W3 + e];
    if (t < kH) {
        sb1[t] = w[off_b1 + t];
        sb2[t] = w[off_b2 + t];
    }
    const int i = t % 16, g = (t % 64) / 16;
    bf16x4 w1[kH / 16];
#pragma unroll
    for (int b = 0; b < kH / 16; b++)
#pragma unroll
        for (int s = 0; s < 4; s++) w1[b][s] = (__bf16)(g < 2 ? w[(4 * g + s) * kH + 16 * b + i] : 0.f);
    const float b3 = g < kOut ? w[off_b3 + g] : 0.f;
    __syncthreads();
    const int64_t ntiles = (rows + kWaveRows - 1) / kWaveRows, step = (int64_t)gridDim.x * (nt / 64);
    for (int64_t tile = (int64_t)blockIdx.x * (nt / 64) + t / 64; tile < ntiles; tile += step) {
        const int64_t r = tile * kWaveRows + i;
        const bool in = r < rows;
        bf16x4 x;
#pragma unroll
        for (int s = 0; s < 4; s++) x[s] = (__bf16)(in && g < 2 ? X[r * kIn + 4 * g + s] : 0.f);
        bf16x8 a1[kH / 32];
#pragma unroll
        for (int p = 0; p < kH / 32; p++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int b = 2 * p + h;
                f32x4 acc = *reinterpret_cast<const f32x4*>(sb1 + 16 * b + 4 * g);
                acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, w1[b]),
                                                                __builtin_bit_cast(s16x4, x), acc, 0, 0, 0);
#pragma unroll
                for (int s = 0; s < 4; s++) a1[p][4 * h + s] = (__bf16)tanh_bf16(acc[s]);
            }
        float y[kOut] = {0.f, 0.f, 0.f};
#pragma unroll 2
        for (int n = 0; n < kH / 16; n++) {
            f32x4 acc = *reinterpret_cast<const f32x4*>(sb2 + 16 * n + 4 * g);
#pragma unroll
            for (int p = 0; p < kH / 32; p++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(sW2t + (16 * n + i) * kW2tPitch + 32 * p + 8 * g);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, a1[p], acc, 0, 0, 0);
            }
            float w3[12];
            load_w3(sW3, 16 * n + 4 * g, w3);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float h = (float)(__bf16)tanh_bf16(acc[s]);
#pragma unroll
                for (int o = 0; o < kOut; o++) y[o] = fmaf(h, w3[3 * s + o], y[o]);
            }
        }
        sum_groups(y);
        if (in && g < kOut) Y[r * kOut + g] = (g == 0 ? y[0] : g == 1 ? y[1] : y[2]) + b3;
    }
}

// ---------------------------------------------------------------------------
// training pass: forward, dY = 2 (Y - T) / (3 rows), dZ2 = (dY W3^T) (1 - A2^2),
// dZ1 = (dZ2 W2^T) (1 - A1^2), and the workgroup's partial of every gradient and of the
// squared error, in one kernel.  A workgroup of four waves runs over 64-row tiles; a wave
// keeps its 16 rows' activations and their gradients in registers and passes them through
// LDS only as operands of the gradients' contractions over the rows:
//   W2: A1^T dZ2, each wave 32 x 128 of it in accumulators for all tiles
//   W1, b1: dZ1^T [X 1],  W3: A2^T dY,  b2: dZ2^T 1   with [X 1 dY] as one 16-column operand
// Bound by the FP32 matrix rate (6 x 128 x 128 flops per row; one wave per SIMD, since the
// LDS holds one workgroup) and the tanh between the products.  The activations that seven
// kernels wrote and read (2 KB per row, up to three times) stay on the chip.
// 31,000 rows: 67 us and 5 for the sum of the partials; the seven kernels took 606.
// ---------------------------------------------------------------------------
constexpr int kActPitch = kH + 16;   // floats per row of the activations in LDS: column reads without conflicts
constexpr int64_t kPartPitch = (n_weights() + 63) / 64 * 64;

__global__ __launch_bounds__(kThr) void k_mlp_train(const float* __restrict__ w, const float* __restrict__ X,
                                                    const float* __restrict__ T, int64_t rows,
                                                    float* __restrict__ part, double* __restrict__ loss_part) {
    __shared__ __align__(16) float sW2[kH * kW2Pitch];
    __shared__ __align__(16) float sA[kTile * kActPitch], sZ[kTile * kActPitch];
    __shared__ __align__(16) float sB[kTile * 16];   // columns 0..7 X, 8 one, 9..11 dY
    __shared__ __align__(16) float sb1[kH], sb2[kH], sW3[kH * kOut];
    __shared__ double sl[kThr / 64];
    __shared__ float sg[kThr / 64][kOut];
    const int t = threadIdx.x;
    for (int e = 4 * t; e < kH * kH; e += 4 * kThr)
        *reinterpret_cast<f32x4*>(sW2 + (e / kH) * kW2Pitch + e % kH) = *reinterpret_cast<const f32x4*>(w + off_W2 + e);
    for (int e = t; e < kH * kOut; e += kThr) sW3[e] = w[off_W3 + e];
    if (t < kH) {
        sb1[t] = w[off_b1 + t];
        sb2[t] = w[off_b2 + t];
    }
    const int wv = t / 64, i = t % 16, g = (t % 64) / 16;
    float w1[kH / 16][2], b3[kOut];
    load_w1(w, i, g, w1);
#pragma unroll
    for (int o = 0; o < kOut; o++) b3[o] = w[off_b3 + o];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 gW2[2][kH / 16], gb2[2], gW3[2], gW1[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        gb2[h] = gW3[h] = gW1[h] = zero;
#pragma unroll
        for (int n = 0; n < kH / 16; n++) gW2[h][n] = zero;
    }
    float gb3[kOut] = {0.f, 0.f, 0.f};
    double lsum = 0.0;
    const float scale = 2.0f / (float)(3 * rows);
    __syncthreads();
    const int64_t ntiles = (rows + kTile - 1) / kTile;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int lr = kWaveRows * wv + i;   // the lane's row in the tile
        const int64_t r = tile * kTile + lr;
        const bool in = r < rows;
        const float x0 = in ? X[r * kIn + g] : 0.f, x1 = in ? X[r * kIn + 4 + g] : 0.f;
        f32x4 a1[kH / 16], a2[kH / 16], z2[kH / 16], z1[kH / 16];
        float y[kOut], d[kOut];
        layer1(w1, sb1, g, x0, x1, a1);
        layer2(sW2, sb2, i, g, a1, a2);
        layer3(sW3, g, a2, y);
#pragma unroll
        for (int o = 0; o < kOut; o++) {
            const float e = in ? (y[o] + b3[o]) - T[r * kOut + o] : 0.f;
            d[o] = scale * e;
            if (g == 0) {
                lsum += (double)e * (double)e;
                gb3[o] += d[o];
            }
        }
#pragma unroll
        for (int b = 0; b < kH / 16; b++) {
            float w3[12];
            load_w3(sW3, 16 * b + 4 * g, w3);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float da = d[0] * w3[3 * s] + d[1] * w3[3 * s + 1] + d[2] * w3[3 * s + 2];
                z2[b][s] = da * (1.f - a2[b][s] * a2[b][s]);
            }
        }
        // dA1^T[c][row] = sum_k W2[c][k] dZ2^T[k][row]
#pragma unroll
        for (int n = 0; n < kH / 16; n++) z1[n] = zero;
        {
            f32x4 wk[2][kH / 16];
            int lane = i * kW2Pitch + 4 * g;
            asm volatile("" : "+v"(lane));   // as in layer2
            auto load = [&](int b) {
#pragma unroll
                for (int n = 0; n < kH / 16; n++)
                    wk[b % 2][n] = *reinterpret_cast<const f32x4*>(sW2 + lane + 16 * n * kW2Pitch + 16 * b);
            };
            load(0);
#pragma unroll
            for (int b = 0; b < kH / 16; b++) {
                if (b + 1 < kH / 16) load(b + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int n = 0; n < kH / 16; n++) z1[n] = mfma4(wk[b % 2][n][s], z2[b][s], z1[n]);
            }
        }
#pragma unroll
        for (int b = 0; b < kH / 16; b++)
#pragma unroll
            for (int s = 0; s < 4; s++) z1[b][s] *= 1.f - a1[b][s] * a1[b][s];
        __syncthreads();   // the last tile's operands are consumed
        sB[16 * lr + g] = x0;
        sB[16 * lr + 4 + g] = x1;
        sB[16 * lr + 8 + g] = g == 0 ? 1.f : g == 1 ? d[0] : g == 2 ? d[1] : d[2];
        sB[16 * lr + 12 + g] = 0.f;
#pragma unroll
        for (int b = 0; b < kH / 16; b++) {
            *reinterpret_cast<f32x4*>(sA + lr * kActPitch + 16 * b + 4 * g) = a1[b];
            *reinterpret_cast<f32x4*>(sZ + lr * kActPitch + 16 * b + 4 * g) = z2[b];
        }
        __syncthreads();
        {
            float va[2][2], vz[2][kH / 16], vb[2][2], v1[2];
            auto load = [&](int j) {
                const float* ra = sA + (4 * j + g) * kActPitch + i;
                const float* rz = sZ + (4 * j + g) * kActPitch + i;
                const int u = j % 2;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    va[u][h] = ra[32 * wv + 16 * h];
                    vb[u][h] = rz[32 * wv + 16 * h];
                }
#pragma unroll
                for (int n = 0; n < kH / 16; n++) vz[u][n] = rz[16 * n];
                v1[u] = sB[16 * (4 * j + g) + i];
            };
            load(0);
#pragma unroll
            for (int j = 0; j < kTile / 4; j++) {
                const int u = j % 2;
                if (j + 1 < kTile / 4) load(j + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int n = 0; n < kH / 16; n++) gW2[h][n] = mfma4(va[u][h], vz[u][n], gW2[h][n]);
                    gb2[h] = mfma4(vb[u][h], v1[u], gb2[h]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < kH / 16; b++) {
            *reinterpret_cast<f32x4*>(sA + lr * kActPitch + 16 * b + 4 * g) = a2[b];
            *reinterpret_cast<f32x4*>(sZ + lr * kActPitch + 16 * b + 4 * g) = z1[b];
        }
        __syncthreads();
        {
            constexpr int kAhead = 4;   // k-steps loaded together: each has only four products
            float v[2][kAhead], x[2][kAhead][2], z[2][kAhead][2];
            auto load = [&](int j) {
#pragma unroll
                for (int q = 0; q < kAhead; q++) {
                    const int row = 4 * (kAhead * j + q) + g;
                    v[j % 2][q] = sB[16 * row + i];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        x[j % 2][q][h] = sA[row * kActPitch + 32 * wv + 16 * h + i];
                        z[j % 2][q][h] = sZ[row * kActPitch + 32 * wv + 16 * h + i];
                    }
                }
            };
            load(0);
#pragma unroll
            for (int j = 0; j < kTile / 4 / kAhead; j++) {
                if (j + 1 < kTile / 4 / kAhead) load(j + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < kAhead; q++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        gW3[h] = mfma4(x[j % 2][q][h], v[j % 2][q], gW3[h]);
                        gW1[h] = mfma4(z[j % 2][q][h], v[j % 2][q], gW1[h]);
                    }
            }
        }
    }
    // partials, laid out like the weights
    float* out = part + (int64_t)blockIdx.x * kPartPitch;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int c = 32 * wv + 16 * h + 4 * g + s;
#pragma unroll
            for (int n = 0; n < kH / 16; n++) out[off_W2 + c * kH + 16 * n + i] = gW2[h][n][s];
            if (i < kIn) out[i * kH + c] = gW1[h][s];
            if (i == kIn) {
                out[off_b1 + c] = gW1[h][s];
                out[off_b2 + c] = gb2[h][s];
            }
            if (i > kIn && i <= kIn + kOut) out[off_W3 + c * kOut + i - kIn - 1] = gW3[h][s];
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lsum += __shfl_xor(lsum, o, 64);
#pragma unroll
        for (int j = 0; j < kOut; j++) gb3[j] += __shfl_xor(gb3[j], o, 64);
    }
    if (t % 64 == 0) {
        sl[wv] = lsum;
#pragma unroll
        for (int j = 0; j < kOut; j++) sg[wv][j] = gb3[j];
    }
    __syncthreads();
    if (t < kOut) out[off_b3 + t] = sg[0][t] + sg[1][t] + sg[2][t] + sg[3][t];
    if (t == 0) loss_part[blockIdx.x] = sl[0] + sl[1] + sl[2] + sl[3];
}

// sum of the workgroups' partial gradients: 32 weights per workgroup, eight threads each over
// every eighth partial, then the eight in order
__global__ __launch_bounds__(kThr) void k_mlp_grad_reduce(const float* __restrict__ part, int nblk,
                                                          float* __restrict__ grad) {
    __shared__ float sh[kThr / 32][32];
    const int t = threadIdx.x % 32, seg = threadIdx.x / 32;
    const int e = blockIdx.x * 32 + t;   // < kPartPitch
    float s = 0.f;
#pragma unroll 8
    for (int b = seg; b < nblk; b += kThr / 32) s += part[(int64_t)b * kPartPitch + e];
    sh[seg][t] = s;
    __syncthreads();
    if (seg == 0 && e < n_weights()) {
#pragma unroll
        for (int q = 1; q < kThr / 32; q++) s += sh[q][t];
        grad[e] = s;
    }
}

__global__ __launch_bounds__(kThr) void k_adam(int64_t P, float* __restrict__ w, const float* __restrict__ g,
                                               float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                               float b2, float eps, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * kThr + threadIdx.x;
    if (i >= P) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---- features / targets / guesses on the context's state ----
__global__ __launch_bounds__(kThr) void k_mlp_features(int64_t N, const double* __restrict__ inc1,
                                                       const double* __restrict__ inc2,
                                                       const double* __restrict__ tact_node, double time,
                                                       double prate, double s_inc, double s_p, double s_t,
                                                       float* __restrict__ X) {
    const int64_t i = (int64_t)blockIdx.x * kThr + threadIdx.x;
    if (i >= N) return;
    float* x = X + i * kIn;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        x[c] = (float)(inc1[3 * i + c] * s_inc);
        x[3 + c] = (float)(inc2[3 * i + c] * s_inc);
    }
    x[6] = (float)(prate * s_p);
    x[7] = (float)((time - tact_node[i]) * s_t);
}

__global__ __launch_bounds__(kThr) void k_mlp_targets(int64_t n, const double* __restrict__ d, double s_inc,
                                                      float* __restrict__ T) {
    const int64_t i = (int64_t)blockIdx.x * kThr + threadIdx.x;
    if (i >= n) return;
    T[i] = (float)(d[i] * s_inc);
}

__global__ __launch_bounds__(kThr) void k_mlp_guess(int64_t N, const float* __restrict__ Y, double inv_s_inc,
                                                    const uint8_t* __restrict__ bcmask, double* __restrict__ g) {
    const int64_t i = (int64_t)blockIdx.x * kThr + threadIdx.x;
    if (i >= N) return;
    const uint8_t m = bcmask[i];
#pragma unroll
    for (int c = 0; c < 3; c++) g[3 * i + c] = ((m >> c) & 1) ? 0.0 : (double)Y[3 * i + c] * inv_s_inc;
}

// mean activation time of the elements incident to each node
__global__ __launch_bounds__(kThr) void k_node_activation(int64_t N, const int64_t* __restrict__ inc_ptr,
                                                          const int32_t* __restrict__ inc, int npe,
                                                          const double* __restrict__ tact, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kThr + threadIdx.x;
    if (i >= N) return;
    double s = 0.0;
    const int64_t b = inc_ptr[i], e = inc_ptr[i + 1];
    for (int64_t k = b; k < e; k++) s += tact[inc[k] / npe];
    out[i] = (e > b) ? s / (double)(e - b) : 0.0;
}

unsigned grid_for(int64_t n) { return (unsigned)((n + kThr - 1) / kThr); }

}  // namespace

struct cmg_mlp {
    cmg_ctx* c = nullptr;
    int device = 0;
    DevBuf w, g, m, v, part, loss_part, tact_node;
    int adam_t = 0;
    double s_inc = 1.0, s_p = 1.0, s_t = 1.0;
    double* h_pin = nullptr;
    ~cmg_mlp() {
        if (h_pin) (void)hipHostFree(h_pin);
    }
};

namespace {

// one 16-row tile per wave up to a wave on every SIMD, then sixteen per workgroup, so that
// a workgroup's copy of the weights serves more rows, in at most one workgroup per CU
struct ForwardShape {
    unsigned blocks, threads;
};
ForwardShape forward_shape(int64_t rows) {
    const int64_t tiles = (rows + kWaveRows - 1) / kWaveRows;
    const int per = tiles > 4 * 256 ? 16 : 4;
    return {(unsigned)std::min<int64_t>((tiles + per - 1) / per, 256), (unsigned)(64 * per)};
}

}  // namespace

extern "C" {

int32_t cmg_mlp_num_weights(int32_t hidden) { return hidden == kH ? (int32_t)n_weights() : -1; }

int cmg_mlp_create(cmg_ctx* c, int32_t hidden, uint64_t seed, cmg_mlp** out) {
    if (!c || !out) return fail("cmg_mlp_create: null argument");
    if (hidden != kH) return fail("cmg_mlp_create: the kernels are built for 128 hidden units");
    CMG_HIP_CHECK(hipSetDevice(c->device));
    std::unique_ptr<cmg_mlp> m(new cmg_mlp());
    m->c = c;
    m->device = c->device;
    const int64_t P = n_weights();
    for (DevBuf* b : {&m->w, &m->g, &m->m, &m->v}) CMG_TRY(alloc(*b, P * sizeof(float)));
    CMG_TRY(alloc(m->part, (size_t)kTrainBlocks * kPartPitch * sizeof(float)));
    CMG_TRY(alloc(m->loss_part, kTrainBlocks * sizeof(double)));
    CMG_TRY(alloc(m->tact_node, c->N * sizeof(double)));
    CMG_HIP_CHECK(hipHostMalloc((void**)&m->h_pin, kTrainBlocks * sizeof(double), hipHostMallocDefault));
    // Glorot-uniform weights, zero biases (seeded host generator)
    std::vector<float> w(P, 0.f);
    std::mt19937_64 gen(seed);
    auto fill = [&](int64_t off, int fan_in, int fan_out) {
        const double a = std::sqrt(6.0 / (fan_in + fan_out));
        std::uniform_real_distribution<double> u(-a, a);
        for (int64_t i = 0; i < (int64_t)fan_in * fan_out; i++) w[off + i] = (float)u(gen);
    };
    fill(0, kIn, kH);
    fill(off_W2, kH, kH);
    fill(off_W3, kH, kOut);
    hipStream_t s = c->stream;
    CMG_HIP_CHECK(hipMemcpyAsync(m->w.p, w.data(), P * sizeof(float), hipMemcpyHostToDevice, s));
    CMG_HIP_CHECK(hipMemsetAsync(m->m.p, 0, P * sizeof(float), s));
    CMG_HIP_CHECK(hipMemsetAsync(m->v.p, 0, P * sizeof(float), s));
    CMG_HIP_CHECK(hipMemsetAsync(m->g.p, 0, P * sizeof(float), s));
    hipLaunchKernelGGL(k_node_activation, dim3(grid_for(c->N)), dim3(kThr), 0, s, c->N, c->inc_ptr.as<int64_t>(),
                       c->inc.as<int32_t>(), c->npe, c->tact.as<double>(), m->tact_node.as<double>());
    CMG_HIP_CHECK(hipGetLastError());
    CMG_HIP_CHECK(hipStreamSynchronize(s));
    *out = m.release();
    return CMG_SUCCESS;
}

int cmg_mlp_destroy(cmg_mlp* m) {
    if (!m) return CMG_SUCCESS;
    (void)hipSetDevice(m->device);   // the context may already be gone: do not touch it
    (void)hipDeviceSynchronize();
    delete m;
    return CMG_SUCCESS;
}

int cmg_mlp_get_weights(cmg_mlp* m, float* w) {
    if (!m || !w) return fail("cmg_mlp_get_weights: null argument");
    CMG_HIP_CHECK(hipMemcpyAsync(w, m->w.p, n_weights() * sizeof(float), hipMemcpyDeviceToHost, m->c->stream));
    CMG_HIP_CHECK(hipStreamSynchronize(m->c->stream));
    return CMG_SUCCESS;
}

int cmg_mlp_set_weights(cmg_mlp* m, const float* w) {
    if (!m || !w) return fail("cmg_mlp_set_weights: null argument");
    CMG_HIP_CHECK(hipMemcpyAsync(m->w.p, w, n_weights() * sizeof(float), hipMemcpyHostToDevice, m->c->stream));
    CMG_HIP_CHECK(hipStreamSynchronize(m->c->stream));
    m->adam_t = 0;
    CMG_HIP_CHECK(hipMemsetAsync(m->m.p, 0, n_weights() * sizeof(float), m->c->stream));
    CMG_HIP_CHECK(hipMemsetAsync(m->v.p, 0, n_weights() * sizeof(float), m->c->stream));
    CMG_HIP_CHECK(hipStreamSynchronize(m->c->stream));
    return CMG_SUCCESS;
}

int cmg_mlp_set_scales(cmg_mlp* m, double inc_scale, double pressure_rate_scale, double phase_scale) {
    if (!m) return fail("null network");
    if (!(inc_scale > 0.0)) return fail("cmg_mlp_set_scales: inc_scale must be positive");
    m->s_inc = inc_scale;
    m->s_p = pressure_rate_scale;
    m->s_t = phase_scale;
    return CMG_SUCCESS;
}

int cmg_mlp_features(cmg_mlp* m, double time, double pressure_rate, float* X) {
    if (!m || !X) return fail("cmg_mlp_features: null argument");
    cmg_ctx* c = m->c;
    CMG_HIP_CHECK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_mlp_features, dim3(grid_for(c->N)), dim3(kThr), 0, c->stream, c->N, c->inc1.as<double>(),
                       c->inc2.as<double>(), m->tact_node.as<double>(), time, pressure_rate, m->s_inc, m->s_p,
                       m->s_t, X);
    CMG_HIP_CHECK(hipGetLastError());
    return CMG_SUCCESS;
}

int cmg_mlp_targets(cmg_mlp* m, float* T) {
    if (!m || !T) return fail("cmg_mlp_targets: null argument");
    cmg_ctx* c = m->c;
    CMG_HIP_CHECK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_mlp_targets, dim3(grid_for(c->n)), dim3(kThr), 0, c->stream, c->n, c->inc1.as<double>(),
                       m->s_inc, T);
    CMG_HIP_CHECK(hipGetLastError());
    return CMG_SUCCESS;
}

int cmg_mlp_forward(cmg_mlp* m, const float* X, int64_t rows, int32_t bf16, float* Y) {
    if (!m || !X || !Y) return fail("cmg_mlp_forward: null argument");
    if (rows <= 0) return CMG_SUCCESS;
    CMG_HIP_CHECK(hipSetDevice(m->c->device));
    hipStream_t s = m->c->stream;
    const ForwardShape sh = forward_shape(rows);
    if (bf16)
        hipLaunchKernelGGL(k_mlp_forward_bf16, dim3(sh.blocks), dim3(sh.threads), 0, s, m->w.as<float>(), X, rows, Y);
    else
        hipLaunchKernelGGL(k_mlp_forward, dim3(sh.blocks), dim3(sh.threads), 0, s, m->w.as<float>(), X, rows, Y);
    CMG_HIP_CHECK(hipGetLastError());
    return CMG_SUCCESS;
}

int cmg_mlp_loss_grad(cmg_mlp* m, const float* X, const float* T, int64_t rows, double* loss, float* grad_host) {
    if (!m || !X || !T) return fail("cmg_mlp_loss_grad: null argument");
    if (rows <= 0) return fail("cmg_mlp_loss_grad: no rows");
    cmg_ctx* c = m->c;
    CMG_HIP_CHECK(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    float* g = m->g.as<float>();
    const unsigned nb = (unsigned)std::min<int64_t>((rows + kTile - 1) / kTile, kTrainBlocks);
    hipLaunchKernelGGL(k_mlp_train, dim3(nb), dim3(kThr), 0, s, m->w.as<float>(), X, T, rows, m->part.as<float>(),
                       m->loss_part.as<double>());
    hipLaunchKernelGGL(k_mlp_grad_reduce, dim3((unsigned)(kPartPitch / 32)), dim3(kThr), 0, s, m->part.as<float>(),
                       (int)nb, g);
    CMG_HIP_CHECK(hipGetLastError());
    CMG_HIP_CHECK(hipMemcpyAsync(m->h_pin, m->loss_part.p, nb * sizeof(double), hipMemcpyDeviceToHost, s));
    if (grad_host) CMG_HIP_CHECK(hipMemcpyAsync(grad_host, g, n_weights() * sizeof(float), hipMemcpyDeviceToHost, s));
    CMG_HIP_CHECK(hipStreamSynchronize(s));
    if (loss) {
        double l = 0.0;
        for (unsigned b = 0; b < nb; b++) l += m->h_pin[b];
        *loss = l / (3.0 * (double)rows);
    }
    return CMG_SUCCESS;
}

int cmg_mlp_adam_step(cmg_mlp* m, float lr) {
    if (!m) return fail("null network");
    CMG_HIP_CHECK(hipSetDevice(m->c->device));
    m->adam_t++;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.f - std::pow(b1, (float)m->adam_t), c2 = 1.f - std::pow(b2, (float)m->adam_t);
    const int64_t P = n_weights();
    hipLaunchKernelGGL(k_adam, dim3(grid_for(P)), dim3(kThr), 0, m->c->stream, P, m->w.as<float>(), m->g.as<float>(),
                       m->m.as<float>(), m->v.as<float>(), lr, b1, b2, eps, c1, c2);
    CMG_HIP_CHECK(hipGetLastError());
    return CMG_SUCCESS;
}

int cmg_mlp_propose_guess(cmg_mlp* m, const float* Y) {
    if (!m || !Y) return fail("cmg_mlp_propose_guess: null argument");
    cmg_ctx* c = m->c;
    CMG_HIP_CHECK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_mlp_guess, dim3(grid_for(c->N)), dim3(kThr), 0, c->stream, c->N, Y, 1.0 / m->s_inc,
                       c->bcmask.as<uint8_t>(), c->override_guess.as<double>());
    CMG_HIP_CHECK(hipGetLastError());
    c->has_override = true;
    c->override_checked = true;
    return CMG_SUCCESS;
}

}  // extern "C"
