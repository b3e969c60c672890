// mlp_device.h — in-kernel inference of the radiance network (hvx_mlp.h):
// the workgroup stages the BF16 weights in LDS, then each wave evaluates 16
// samples per call with the 16x16x32 BF16 MFMA, all activations staying in
// registers. The positional encoding is computed straight into the first
// layer's operand layout; the FP32 output layer is reduced across lanes from
// the last accumulators. Against the training forward pass of mlp.hip: the
// same encoding bits, BF16 operands, instruction, bias and ReLU after the
// FP32 accumulation and output-layer summation order; layers 2 and 3 feed
// each 32-unit K block to the MFMA in a permuted order (mlp_unit).
#pragma once

#include <hip/hip_runtime.h>

#include "hvx_mfma.h"
#include "hvx_mlp.h"

namespace hvx {

// Device view of a network's parameters (owned by hvx_mlp).
struct MlpView {
    const __bf16* W1;  // [64][128]
    const __bf16* W2;  // [64][64]
    const __bf16* W3;  // [64][64]
    const float* P;    // FP32 parameters (biases, W4, b4 are read from here)
    float lod_max;
};

// The weights are kept as the matrix operands: 16-row tile nb and K block s of
// a layer are 64 lanes x 8 values in one piece, so a wave's 16-byte reads meet
// every bank once (as rows of W sixteen lanes met in the same four banks of W1:
// 2 million samples 547 us, so 164). Layers 2 and 3 have K permuted: lane (g, i)'s
// value q of block s is W[16 nb + i][mlp_unit(s, g, q)], the order in which
// each lane holds the previous layer's units.
struct MlpLds {
    __align__(16) __bf16 W1[kMlpHidden * kMlpIn];
    __align__(16) __bf16 W2[kMlpHidden * kMlpHidden];
    __align__(16) __bf16 W3[kMlpHidden * kMlpHidden];
    __align__(16) float b1[kMlpHidden], b2[kMlpHidden], b3[kMlpHidden];
    __align__(16) float W4[kMlpOut * kMlpHidden];
    float b4[4];
};

// Cooperative copy of the weights into LDS (the caller synchronises).
__device__ __forceinline__ void mlp_stage(MlpLds& L, const MlpView& v) {
    const uint32_t t = threadIdx.x, n = blockDim.x;
#pragma unroll 4  // four reads in flight
    for (uint32_t c = t; c < kMlpHidden * kMlpIn / 8; c += n) {
        const uint32_t lane = c & 63, ks = c >> 6 & 3, nb = c >> 8;
        reinterpret_cast<uint4*>(L.W1)[c] = *reinterpret_cast<const uint4*>(
            v.W1 + (16 * nb + (lane & 15)) * kMlpIn + 32 * ks + 8 * (lane >> 4));
    }
#pragma unroll 4
    for (uint32_t c = t; c < 2 * kMlpHidden * kMlpHidden / 8; c += n) {
        const bool third = c >= kMlpHidden * kMlpHidden / 8;
        const uint32_t k = c & (kMlpHidden * kMlpHidden / 8 - 1), lane = k & 63, ks = k >> 6 & 1, nb = k >> 7;
        // units mlp_unit(ks, g, 0..3) and (ks, g, 4..7): four each in a row
        const __bf16* row = (third ? v.W3 : v.W2) + (16 * nb + (lane & 15)) * kMlpHidden + 32 * ks + 4 * (lane >> 4);
        const uint2 a = *reinterpret_cast<const uint2*>(row), b = *reinterpret_cast<const uint2*>(row + 16);
        reinterpret_cast<uint4*>(third ? L.W3 : L.W2)[k] = make_uint4(a.x, a.y, b.x, b.y);
    }
    for (uint32_t i = t; i < kMlpHidden; i += n) {
        L.b1[i] = v.P[kMlpB1 + i];
        L.b2[i] = v.P[kMlpB2 + i];
        L.b3[i] = v.P[kMlpB3 + i];
    }
    for (uint32_t i = t; i < kMlpOut * kMlpHidden; i += n) L.W4[i] = v.P[kMlpW4 + i];
    if (t < kMlpOut) L.b4[t] = v.P[kMlpB4 + t];
}

// ReLU(acc + bias), rounded to BF16, of the accumulators of one layer: lane
// (g, i) holds unit 16 nb + 4 g + r of sample i in acc[nb][r].
template <int T>
__device__ __forceinline__ void mlp_activate(const f32x4 (&acc)[T][4], const float* bias, uint32_t g,
                                             __bf16 (&h)[T][4][4]) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(bias + 16 * nb + 4 * g);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) h[t][nb][r] = (__bf16)fmaxf(acc[t][nb][r] + b[r], 0.0f);
    }
}

// One 64 -> 64 layer: the B operand of K block s is the lane's own units
// h[2 s][0..3], h[2 s + 1][0..3] (K index 8 g + q <-> mlp_unit(s, g, q)).
template <int T>
__device__ __forceinline__ void mlp_hidden_layer(const __bf16* Wp, const __bf16 (&h)[T][4][4], uint32_t lane,
                                                 f32x4 (&acc)[T][4]) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[t][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        bf16x8 b[T];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 8; ++q) b[t][q] = h[t][2 * s + (q >> 2)][q & 3];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(Wp + ((2 * nb + s) * 64 + lane) * 8);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t][nb] = mfma16x16x32(a, b[t], acc[t][nb]);
        }
    }
}

// Forward of T tiles of 16 samples by one wave, entirely in registers (the
// LDS holds only the weights, read once for the T tiles). Lane l holds the
// inputs x[t] = (dir, lod) of sample l & 15 of tile t (the four lanes of a
// sample hold the same values); y[t] is, in lanes with g = l >> 4 < 3, channel
// g of that sample's predicted radiance, in the others 0. Each layer computes
// its outputs transposed (weights as the A operand, samples as the columns),
// so lane (g, i) ends with 16 units of sample i, which are the B operand of
// the next layer as they are.
template <int T>
__device__ __forceinline__ void mlp_forward_tiles(const MlpLds& L, const float (&x)[T][4], float lod_max,
                                                  float (&y)[T]) {
    const uint32_t lane = threadIdx.x & 63, g = lane >> 4;
    f32x4 acc[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[t][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        bf16x8 b[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            // features 32 s + 8 g + 2 q + (0 sin, 1 cos): input s, frequency 4 g + q
            const float xin = s < 3 ? x[t][s] : 2.0f * x[t][3] / lod_max - 1.0f;
            float sv[4], cv[4];
            mlp_sincos_direct(xin, 4 * (int)g, sv[0], cv[0]);
            mlp_sincos_direct(xin, 4 * (int)g + 1, sv[1], cv[1]);
            mlp_sincos_double(sv[0], cv[0], sv[2], cv[2]);
            mlp_sincos_double(sv[1], cv[1], sv[3], cv[3]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                b[t][2 * q] = (__bf16)sv[q];
                b[t][2 * q + 1] = (__bf16)cv[q];
            }
        }
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(L.W1 + ((4 * nb + s) * 64 + lane) * 8);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t][nb] = mfma16x16x32(a, b[t], acc[t][nb]);
        }
        // one K block at a time: without the fence the scheduler hoists every
        // block's weight loads and encoding, past the register budget
        __builtin_amdgcn_sched_barrier(0);
    }
    __bf16 h[T][4][4];
    mlp_activate(acc, L.b1, g, h);
    mlp_hidden_layer(L.W2, h, lane, acc);
    mlp_activate(acc, L.b2, g, h);
    mlp_hidden_layer(L.W3, h, lane, acc);
    mlp_activate(acc, L.b3, g, h);
    // output layer in the order of mlp_output: the lane's 16 units, then
    // across the four lane groups (lanes i, i + 16, i + 32, i + 48)
    float o[T];  // of channel g (lanes with g = 3: of channel 0)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        float v[T];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(L.W4 + c * kMlpHidden + 16 * nb + 4 * g);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = (float)h[t][nb][r] * w[r];
                    v[t] = nb + r == 0 ? p : v[t] + p;
                }
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            v[t] = v[t] + __shfl_xor(v[t], 16, 64);
            v[t] = v[t] + __shfl_xor(v[t], 32, 64);
            v[t] = v[t] + L.b4[c];
            o[t] = c == 0 || g == (uint32_t)c ? v[t] : o[t];
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) y[t] = g < 3 ? expf(o[t]) - (float)kMlpEps : 0.0f;
}
__device__ __forceinline__ float mlp_forward_tile(const MlpLds& L, const float (&x)[4], float lod_max) {
    const float xs[1][4] = {{x[0], x[1], x[2], x[3]}};
    float y[1];
    mlp_forward_tiles(L, xs, lod_max, y);
    return y[0];
}

}  // namespace hvx
