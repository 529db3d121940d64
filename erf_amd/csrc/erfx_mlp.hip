// erfx_mlp.hip -- the learned stand-in for Kessler's cell tendencies: an
// 8 -> 128 -> 128 -> 4 multilayer perceptron with GELU activations, BF16
// weights and activations and FP32 accumulation, trained on the GPU by the
// kernels below (forward, backward, Adam).  It has no counterpart in ERF; the
// plain Kessler scheme (Source/Microphysics/Kessler/ERF_Kessler.cpp:11-250)
// produces its training data and is its fallback and the reference for its error.
//
// Inputs (T, p [mbar], rho, qv, qc, qr, w, dt), normalised per feature;
// outputs the local process tendencies of one step (dqv, dqc, dqr, dtheta,
// sedimentation excluded), scaled per output.
//
// Matrix work runs on the CDNA4 matrix cores: v_mfma_f32_32x32x16_bf16 (one
// wave computes a 32x32 FP32 tile from 32x16 and 16x32 BF16 operands).
// Operand layouts of that instruction for lane l of a 64-wide wave:
//   A (32 x 16): row l % 32, columns 8 (l / 32) .. 8 (l / 32) + 7
//   B (16 x 32): column l % 32, rows 8 (l / 32) .. 8 (l / 32) + 7
//   D (32 x 32): column l % 32, rows 8 (i / 4) + 4 (l / 32) + i % 4, i = 0..15
// The forward pass runs all three layers on the matrix cores (the input and
// output layers zero-padded to the instruction's K = 16 and M = 32); the
// training pass runs the forward layers and the hidden layer's two backward
// products there and the 8-wide and 4-wide gradients on the vector ALUs in FP32.
#include "erfx_common.h"
#include "erfx_internal.h"
#include "erfx_mlp.h"

namespace erfx {
namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// 0.5 erfc(a / sqrt 2), the normal distribution's upper tail, for a >= 0, as
// 2^-(1 + a Q(a)): Q is smooth, and a degree-9 polynomial fitted to
// -(log2 Phi(-a) + 1) / a at 1,000 points of [0, 6.5] (weighted minimax, solved as a
// linear program, the weight that of a gelu's absolute error plus a floor for the
// relative one).  One formula for every lane where erff takes one of two by the
// size of its argument, a dozen instructions with the hardware's 2^x.  Its
// relative error is below 2e-6 up to 6.5, where 1 + erf cancels on the left; beyond,
// Q keeps growing and only the absolute error of a gelu stays small (below 1e-11).
// GELU formed with it is within 2.4e-7 of the 64-bit value on [-9, 9], 4.9e-8 rms;
// with erff 4.5e-7 and 6.4e-8.
__device__ __forceinline__ float upper_tail(float a) {
    float q = 1.30723766e-08f;
    q = fmaf(q, a, -4.47882636e-07f);
    q = fmaf(q, a, 6.49634937e-06f);
    q = fmaf(q, a, -5.01334745e-05f);
    q = fmaf(q, a, 1.88647497e-04f);
    q = fmaf(q, a, 1.87812710e-04f);
    q = fmaf(q, a, -7.17206105e-03f);
    q = fmaf(q, a, 5.25871247e-02f);
    q = fmaf(q, a, 4.59176885e-01f);
    q = fmaf(q, a, 1.15110850e+00f);
    return __builtin_amdgcn_exp2f(fmaf(-a, q, -1.0f));
}
// z Phi(z): z - |z| tail for z > 0, -|z| tail for z < 0.  The factor of the tail
// stops at the largest float above, so that +infinity, whose tail is 0, stays
// +infinity; finite values are not touched, and -infinity and NaN give NaN, as
// 0.5 z (1 + erf(z / sqrt 2)) does.
__device__ __forceinline__ float gelu(float z) {
    // a median of three is a maximum or a clamp in one instruction
    const float f = __builtin_amdgcn_fmed3f(z, -__builtin_inff(), 3.40282347e+38f);
    return fmaf(-fabsf(f), upper_tail(fabsf(z)), __builtin_amdgcn_fmed3f(z, 0.0f, __builtin_inff()));
}
// Phi(z) + z phi(z)
__device__ __forceinline__ float gelu_grad(float z) {
    const float t = upper_tail(fabsf(z));
    const float phi = 0.39894228040143268f * __builtin_amdgcn_exp2f(-0.72134752044448170f * z * z);
    return fmaf(z, phi, z > 0.0f ? 1.0f - t : t);
}
__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }
__device__ __forceinline__ __bf16 f2bf(float v) { return (__bf16)v; }

// LDS row pitch of a 32 x 128 BF16 tile: 8 elements of padding keep the
// 16-byte operand reads of 32 rows on distinct banks
constexpr int TP = NH + 8;

// orders a wave's LDS stores before its later loads of what other lanes stored
// (a wave's LDS operations execute in order; this keeps the compiler's order)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// row of accumulator element i of lane l in a 32 x 32 tile
__device__ __forceinline__ int drow(int l, int i) { return 8 * (i >> 2) + 4 * (l >> 5) + (i & 3); }

// four consecutive accumulator elements as BF16, in the order of their rows
__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
    bf16x4 v;
    v[0] = f2bf(a); v[1] = f2bf(b); v[2] = f2bf(c); v[3] = f2bf(d);
    return v;
}

// Forward pass of 32 samples per wave, WPB waves per block.  x: normalised
// inputs [n][NI]; y: scaled outputs [n][NO].  The products are formed transposed
// (units along the rows of a tile, samples along its columns: A = W^T, B = h^T),
// so a lane holds groups of four consecutive units of one sample, which go to
// LDS as one 8-byte store, and the biases enter as the accumulators' first
// value.  A wave's tile is its own, so no block barriers are needed after the
// weights are staged.  The vector ALUs bound the kernel: two GELUs per unit and
// sample, 256 per sample (1,048,576 samples: 226 us with erff and two-byte
// stores, 135 us now; the products alone would take 19 us).
template <int WPB>
__global__ void __launch_bounds__(64 * WPB, 4) fwd_kernel(const float* __restrict__ x, int n, const Weights W,
                                                        float* __restrict__ y) {
    __shared__ __align__(16) __bf16 tile[WPB][32 * TP];
    __shared__ __align__(16) __bf16 sw1[NH * NI];   // [u][k]
    __shared__ __align__(16) __bf16 sw3[NO * NH];   // [o][u]
    __shared__ __align__(16) float sb1[NH], sb2[NH], sb3[NO];
    for (int e = threadIdx.x; e < NI * NH; e += 64 * WPB) sw1[(e % NH) * NI + e / NH] = W.w1[e];
    for (int e = threadIdx.x; e < NH * NO; e += 64 * WPB) sw3[(e % NO) * NH + e / NO] = W.w3[e];
    for (int e = threadIdx.x; e < NH; e += 64 * WPB) { sb1[e] = W.b1[e]; sb2[e] = W.b2[e]; }
    if (threadIdx.x < NO) sb3[threadIdx.x] = W.b3[threadIdx.x];
    __syncthreads();
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int r = l & 31, half = l >> 5, kh = half * 8;
    const int s = (blockIdx.x * WPB + wv) * 32 + r;
    __bf16* h = tile[wv] + r * TP;      // this lane's sample
    const bool live = s < n;
    const __bf16 zero = f2bf(0.0f);
    // accumulators of 32 units from `b`: rows 8 g + 4 half .. + 3, g = 0..3
    auto start = [&](const float* b) {
        floatx16 a;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 v = *reinterpret_cast<const float4*>(b + 8 * g + 4 * half);
            a[4 * g] = v.x; a[4 * g + 1] = v.y; a[4 * g + 2] = v.z; a[4 * g + 3] = v.w;
        }
        return a;
    };
    // GELU of a tile to the sample's row in LDS
    auto act = [&](const floatx16& a, int t) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<bf16x4*>(h + 32 * t + 8 * g + 4 * half) =
                pack4(gelu(a[4 * g]), gelu(a[4 * g + 1]), gelu(a[4 * g + 2]), gelu(a[4 * g + 3]));
    };
    // ---- input layer: B = x (the 8 inputs in the first half of K, zeros in the second)
    bf16x8 xb;
#pragma unroll
    for (int q = 0; q < 8; ++q) xb[q] = (half == 0 && live) ? f2bf(x[(long)s * NI + q]) : zero;
    floatx16 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        bf16x8 wa = *reinterpret_cast<const bf16x8*>(sw1 + (32 * t + r) * NI);
#pragma unroll
        for (int q = 0; q < 8; ++q) wa[q] = half == 0 ? wa[q] : zero;
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa, xb, start(sb1 + 32 * t), 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) act(acc[t], t);
    wave_lds_fence();
    // ---- hidden layer
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = start(sb2 + 32 * t);
#pragma unroll 2
    for (int c = 0; c < NH / 16; ++c) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(h + 16 * c + kh);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(W.w2t + ((c * 4 + t) * 64 + l) * 8);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
        }
    }
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < 4; ++t) act(acc[t], t);
    wave_lds_fence();
    // ---- output layer: row o of the tile is output o for o < NO
    floatx16 ao;
#pragma unroll
    for (int i = 0; i < 16; ++i) ao[i] = i < NO && half == 0 ? sb3[i < NO ? i : 0] : 0.0f;
    const int oc = r < NO ? r : NO - 1;   // lanes of the padding rows read a valid row, then use 0
#pragma unroll
    for (int c = 0; c < NH / 16; ++c) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(h + 16 * c + kh);
        bf16x8 a = *reinterpret_cast<const bf16x8*>(sw3 + oc * NH + 16 * c + kh);
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = r < NO ? a[q] : zero;
        ao = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, ao, 0, 0, 0);
    }
    if (half == 0 && live) {
#pragma unroll
        for (int o = 0; o < NO; ++o) y[(long)s * NO + o] = ao[o];
    }
}

// One training pass over TS samples per block: forward, mean-squared-error
// gradient and the block's share of every weight gradient, with no activation
// leaving the chip.  A wave takes a group of 32 samples and a quarter of the units.
// Pre-activations stay in the lanes that made them (samples along the rows of a
// tile, a unit per lane column), the activations the products read are in LDS as
// BF16, by sample and, for the product over samples, by unit:
//   h1 = gelu(x W1 + b1), h2 = gelu(h1 W2 + b2), y = h2 W3 + b3,
//   dy = 2 scale (y - t), dz2 = (dy W3^T) gelu'(z2) (BF16), dz1 = (dz2 W2^T) gelu'(z1) (FP32),
//   dW2 = h1^T dz2 (matrix cores), dW1 = x^T dz1, dW3 = h2^T dy and the biases
//   (FP32 sums on the vector ALUs: a lane sums its 16 rows, then the halves of a
//   wave and the two sample groups are added).
// The sums of a block go to `partial`, which the Adam kernel adds over the blocks.
// Latency bound at training batches (8,192 samples are 128 blocks).  The three
// kernels it replaced (forward storing z and h, backward, weight gradients) took
// 26 + 56 + 42 us at 8,192 samples, this 17 us.
constexpr int TS = 64;
constexpr int SP = TS + 8;   // LDS row pitch of the arrays by unit
constexpr int UP = 4;        // parts of the units: a wave per sample group and part
constexpr int NT = 4 / UP;   // tiles of 32 units per wave
constexpr int TW = 64 * 2 * UP;
constexpr int NV = 14 * NT;  // small sums per lane
__global__ void __launch_bounds__(TW) train_kernel(const float* __restrict__ x, const float* __restrict__ tgt, int n,
                                                    const Weights W, float* __restrict__ loss, float scale,
                                                    float* __restrict__ partial) {
    __shared__ __align__(16) __bf16 hb[TS * TP];     // [s][u]: h1, then h2, then dz2
    __shared__ __align__(16) __bf16 h1t[NH * SP];    // [u][s]
    __shared__ __align__(16) __bf16 dzt[NH * SP];    // [u][s]
    __shared__ __align__(16) float sx[TS * NI];      // inputs, rounded to BF16
    __shared__ __align__(16) float sdy[TS * NO];
    __shared__ float red[UP][NV][32];
    __shared__ float red3[2][NO];
    __shared__ __align__(16) __bf16 sw3[NO * NH];    // [o][u]
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const int sg = wv & 1, uh = wv >> 1;
    const int r = l & 31, half = l >> 5, kh = half * 8;
    const int b0 = blockIdx.x * TS, g0 = sg * 32;
    const __bf16 zero = f2bf(0.0f);
    for (int e = tid; e < TS * NI; e += TW) sx[e] = b0 + e / NI < n ? bf2f(f2bf(x[(long)b0 * NI + e])) : 0.0f;
    for (int e = tid; e < NH * NO; e += TW) sw3[(e % NO) * NH + e / NO] = W.w3[e];
    float* out = partial + (long)blockIdx.x * NPARAM;
    int u[NT];
    float bias1[2], bias2[NT];
    bf16x8 w1b[NT];
    bf16x4 w3r[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        u[t] = (uh * NT + t) * 32 + r;
        bias1[t] = W.b1[u[t]];
        bias2[t] = W.b2[u[t]];
        w3r[t] = *reinterpret_cast<const bf16x4*>(W.w3 + u[t] * NO);
#pragma unroll
        for (int q = 0; q < 8; ++q) w1b[t][q] = half == 0 ? W.w1[q * NH + u[t]] : zero;
    }
    __syncthreads();
    // ---- input layer
    bf16x8 xa;
#pragma unroll
    for (int q = 0; q < 8; ++q) xa[q] = half == 0 ? f2bf(sx[(g0 + r) * NI + q]) : zero;
    floatx16 z1[2], z2[NT];
    float h2[NT][16];
    floatx16 z0;
#pragma unroll
    for (int i = 0; i < 16; ++i) z0[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        z1[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, w1b[t], z0, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int row = g0 + 8 * g + 4 * half;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                z1[t][4 * g + e] += bias1[t];
                v[e] = gelu(z1[t][4 * g + e]);
                hb[(row + e) * TP + u[t]] = f2bf(v[e]);
            }
            *reinterpret_cast<bf16x4*>(h1t + u[t] * SP + row) = pack4(v[0], v[1], v[2], v[3]);
        }
    }
    __syncthreads();
    // (rows of hb of the wave's samples) times an operand whose rows are the units (frag order)
    auto gemm = [&](const __bf16* bt, floatx16 (&acc)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = z0;
#pragma unroll
        for (int c = 0; c < NH / 16; ++c) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(hb + (g0 + r) * TP + 16 * c + kh);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(bt + ((c * 4 + NT * uh + t) * 64 + l) * 8);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
            }
        }
    };
    // ---- hidden layer
    gemm(W.w2t, z2);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            z2[t][i] += bias2[t];
            const __bf16 v = f2bf(gelu(z2[t][i]));
            h2[t][i] = bf2f(v);
            hb[(g0 + drow(l, i)) * TP + u[t]] = v;
        }
    __syncthreads();
    // ---- output layer (transposed: row o, a sample per lane) and dy, by the first half's waves
    if (uh == 0) {
        floatx16 ao = z0;
        const int oc = r < NO ? r : NO - 1;
#pragma unroll
        for (int c = 0; c < NH / 16; ++c) {
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(hb + (g0 + r) * TP + 16 * c + kh);
            bf16x8 a = *reinterpret_cast<const bf16x8*>(sw3 + oc * NH + 16 * c + kh);
#pragma unroll
            for (int q = 0; q < 8; ++q) a[q] = r < NO ? a[q] : zero;
            ao = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, ao, 0, 0, 0);
        }
        const int s = b0 + g0 + r;
        const bool live = half == 0 && s < n;
        float se = 0.0f, dy[NO];
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const float d = live ? ao[o] + W.b3[o] - tgt[(long)s * NO + o] : 0.0f;
            se += d * d;
            dy[o] = scale * 2.0f * d;
            if (half == 0) sdy[(g0 + r) * NO + o] = dy[o];
        }
        if (live) loss[s] = se;
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            float a = dy[o];
#pragma unroll
            for (int m = 1; m < 32; m <<= 1) a += __shfl_xor(a, m);
            if (l == 0) red3[sg][o] = a;
        }
    }
    __syncthreads();
    // ---- dz2, dW3, db2
    float gw3[NT][NO] = {}, gb2[NT] = {}, gw1[NT][NI] = {}, gb1[NT] = {};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int row = g0 + 8 * g + 4 * half;
        float4 dy[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) dy[e] = *reinterpret_cast<const float4*>(sdy + (row + e) * NO);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            bf16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 4 * g + e;
                float dh = dy[e].x * bf2f(w3r[t][0]);
                dh += dy[e].y * bf2f(w3r[t][1]);
                dh += dy[e].z * bf2f(w3r[t][2]);
                dh += dy[e].w * bf2f(w3r[t][3]);
                v[e] = f2bf(dh * gelu_grad(z2[t][i]));
                hb[(row + e) * TP + u[t]] = v[e];
                gb2[t] += bf2f(v[e]);
                gw3[t][0] += h2[t][i] * dy[e].x;
                gw3[t][1] += h2[t][i] * dy[e].y;
                gw3[t][2] += h2[t][i] * dy[e].z;
                gw3[t][3] += h2[t][i] * dy[e].w;
            }
            *reinterpret_cast<bf16x4*>(dzt + u[t] * SP + row) = v;
        }
    }
    __syncthreads();
    // ---- dz1, dW1, db1: dh1[s][k] = sum_u dz2[s][u] W2[k][u] (column k of the product is row k of W2)
    floatx16 acc[NT];
    gemm(W.w2, acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float4* xr = reinterpret_cast<const float4*>(sx + (g0 + drow(l, i)) * NI);
        const float4 xl = xr[0], xh = xr[1];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float d = acc[t][i] * gelu_grad(z1[t][i]);
            gb1[t] += d;
            gw1[t][0] += xl.x * d; gw1[t][1] += xl.y * d; gw1[t][2] += xl.z * d; gw1[t][3] += xl.w * d;
            gw1[t][4] += xh.x * d; gw1[t][5] += xh.y * d; gw1[t][6] += xh.z * d; gw1[t][7] += xh.w * d;
        }
    }
    // ---- the block's sums of the small gradients
    float val[NV];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int k = 0; k < NI; ++k) val[14 * t + k] = gw1[t][k];
        val[14 * t + 8] = gb1[t];
        val[14 * t + 9] = gb2[t];
#pragma unroll
        for (int o = 0; o < NO; ++o) val[14 * t + 10 + o] = gw3[t][o];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        val[v] += __shfl_xor(val[v], 32);
        if (sg == 1 && half == 0) red[uh][v][r] = val[v];
    }
    __syncthreads();
    if (sg == 0 && half == 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int k = 0; k < NI; ++k) out[OFF_W1 + k * NH + u[t]] = val[14 * t + k] + red[uh][14 * t + k][r];
            out[OFF_B1 + u[t]] = val[14 * t + 8] + red[uh][14 * t + 8][r];
            out[OFF_B2 + u[t]] = val[14 * t + 9] + red[uh][14 * t + 9][r];
#pragma unroll
            for (int o = 0; o < NO; ++o) out[OFF_W3 + u[t] * NO + o] = val[14 * t + 10 + o] + red[uh][14 * t + 10 + o][r];
        }
    }
    if (tid < NO) out[OFF_B3 + tid] = red3[0][tid] + red3[1][tid];
    // ---- dW2[k][u] = sum_s h1[s][k] dz2[s][u]: 16 tiles of 32 x 32, NT * 2 per wave
    const int tm = wv / (UP / 2);
#pragma unroll
    for (int tt = 0; tt < 2 * NT; ++tt) {
        const int tn = wv % (UP / 2) * 2 * NT + tt;
        floatx16 a2 = z0;
#pragma unroll
        for (int c = 0; c < TS / 16; ++c) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(h1t + (32 * tm + r) * SP + 16 * c + kh);
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(dzt + (32 * tn + r) * SP + 16 * c + kh);
            a2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, a2, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) out[OFF_W2 + (32 * tm + drow(l, i)) * NH + 32 * tn + r] = a2[i];
    }
}

// Sum of the block partials per parameter (four waves per 64 parameters, each
// a quarter of the blocks in order with 8 loads in flight, the quarters added in
// order: the same sum on every run; one lane per parameter waited for one load
// after the other, 32 us at 128 blocks against 4.6 us), then either the
// gradient is written out or Adam updates the FP32 master weights and refreshes
// the BF16 copies used by the kernels.
__global__ void __launch_bounds__(256) adam_kernel(const float* __restrict__ partial, int nblk, Params_ pm,
                                                   float* __restrict__ grad_out, bool update, float lr, float b1c,
                                                   float b2c) {
    __shared__ float part[4][64];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int p = blockIdx.x * 64 + l;
    const int lo = (int)((long)nblk * wv / 4), hi = (int)((long)nblk * (wv + 1) / 4);
    float s = 0.0f;
    if (p < NPARAM) {
        int b = lo;
        for (; b + 8 <= hi; b += 8) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = partial[(long)(b + e) * NPARAM + p];
#pragma unroll
            for (int e = 0; e < 8; ++e) s += v[e];
        }
        for (; b < hi; ++b) s += partial[(long)b * NPARAM + p];
    }
    part[wv][l] = s;
    __syncthreads();
    if (wv != 0 || p >= NPARAM) return;
    const float g = ((part[0][l] + part[1][l]) + part[2][l]) + part[3][l];
    if (grad_out) grad_out[p] = g;
    if (!update) return;
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    float m = beta1 * pm.m[p] + (1.0f - beta1) * g;
    float v = beta2 * pm.v[p] + (1.0f - beta2) * g * g;
    pm.m[p] = m;
    pm.v[p] = v;
    const float mh = m / b1c, vh = v / b2c;
    const float w = pm.w[p] - lr * mh / (sqrtf(vh) + eps);
    pm.w[p] = w;
    write_bf16_copy(pm, p, w);
}

__global__ void refresh_kernel(Params_ pm) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPARAM) write_bf16_copy(pm, p, pm.w[p]);
}

__global__ void loss_kernel(const float* __restrict__ loss, int n, float* __restrict__ out) {
    // one block: fixed-order sum
    __shared__ float sh[256];
    float a = 0.0f;
    for (int s = threadIdx.x; s < n; s += 256) a += loss[s];
    sh[threadIdx.x] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}

}  // namespace mlp

// ---- host side ------------------------------------------------------------------
using namespace mlp;

// Forward launches: 4 waves per block (the weights staged once for 128
// samples) when that still gives every CU several blocks, else one wave per
// block so that a small batch spreads over the 256 CUs.
void mlp_forward(const Net& N, const float* x, float* y, int n, hipStream_t s) {
    if (n <= 0) return;
    if ((n + 127) / 128 >= 1024)
        hipLaunchKernelGGL((fwd_kernel<4>), dim3((n + 127) / 128), dim3(256), 0, s, x, n, N.W, y);
    else
        hipLaunchKernelGGL((fwd_kernel<1>), dim3((n + 31) / 32), dim3(64), 0, s, x, n, N.W, y);
}

void mlp_refresh(const Net& N, hipStream_t s) {
    hipLaunchKernelGGL(refresh_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, s, N.P);
}

// forward + backward + gradient of the mean squared error over n samples
// (n <= N.cap); with `update`, one Adam step at learning rate lr (step count
// N.t incremented by the caller).  With `want_loss` the loss sum lands in
// N.loss_dev[0].
void mlp_train_pass(Net& N, const float* x, const float* tgt, int n, bool update, float lr, float* grad_out,
                    bool want_loss, hipStream_t s) {
    const float scale = 1.0f / (float)(n * NO);
    const int nblk = (n + TS - 1) / TS;
    hipLaunchKernelGGL(train_kernel, dim3(nblk), dim3(TW), 0, s, x, tgt, n, N.W, N.loss, scale, N.partial);
    float b1c = 1.0f, b2c = 1.0f;
    if (update) {
        b1c = 1.0f - powf(0.9f, (float)N.t);
        b2c = 1.0f - powf(0.999f, (float)N.t);
    }
    hipLaunchKernelGGL(adam_kernel, dim3((NPARAM + 63) / 64), dim3(256), 0, s, (const float*)N.partial, nblk, N.P,
                       grad_out, update, lr, b1c, b2c);
    if (want_loss)
        hipLaunchKernelGGL(loss_kernel, dim3(1), dim3(256), 0, s, (const float*)N.loss, n, N.loss_dev);
}

}  // namespace erfx
