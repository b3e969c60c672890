// mlp.hip — the per-environment radiance network (hvx_mlp_* of
// include/hvx.h), trained with hand-written BF16 MFMA forward and backward
// kernels and FP32 master weights (Adam).
//
// One training step over a batch of B samples (B a multiple of 256):
//   pe            X0 = PE(d, lod)                        bf16 [B][128];
//                 once per training call when the call revisits its samples
//   step          per block of 128 samples, everything in LDS: the three
//                 layers H_l = relu(H_{l-1} W_l^T + b_l), the output layer
//                 y = H3 W4^T + b4 with the loss, dZ3 = (dY W4) * [H3 > 0],
//                 dZ_{l-1} = (dZ_l W_l) * [H_{l-1} > 0], and per slice of the
//                 batch the gradient partials dW_l = dZ_l^T H_{l-1}, db_l, dW4, db4
//   reduce        the slices' partials summed in slice order, with the Adam
//                 update of the FP32 masters and of the BF16 copies of W1..W3
//                 in the same launch
// HVX_OPT_MLP_SEPARATE_LAUNCHES runs the same step as one launch per product
// (gemm FWD x3, out, gemm PART and BWD per layer, reductions, adam), with the
// activations and gradients in memory.
// Every GEMM is C = A Bt^T with both operands row-major along K, so each MFMA
// operand load is one contiguous 16-byte read; the epilogues also write the
// transposed activation that the weight-gradient GEMMs read that way.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "hvx_device.h"
#include "hvx_internal.h"
#include "hvx_contract.h"
#include "hvx_mfma.h"
#include "hvx_mlp.h"
#include "mlp_device.h"

namespace {

using namespace hvx;
typedef __bf16 bf16;

constexpr int kIn = hvx::kMlpIn, kH = hvx::kMlpHidden;
constexpr uint32_t kMaxBatch = 1u << 20;

// ------------------------------------------------------------------- data
__device__ __forceinline__ uint64_t smix(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ __forceinline__ float u01(uint64_t seed, uint64_t stream, uint64_t i) {
    return (float)((double)(smix(seed + (stream << 40) + i) >> 11) * (1.0 / 9007199254740992.0));
}

// textureLod of the prefiltered chain (trilinear, LOD clamped to [0, mips-1])
__device__ __forceinline__ f3 chain_lod(const float4* chain, uint32_t S, uint32_t mips, f3 dir, float lod) {
    const float q = (float)(mips - 1);
    const float lam = gclamp(lod, 0.0f, q);
    const float fl = floorf_(lam);
    const uint32_t l0 = (uint32_t)fl, l1 = min(l0 + 1, mips - 1);
    const float d = lam - fl;
    const int s0 = (int)max(S >> l0, 1u), s1 = (int)max(S >> l1, 1u);
    const f3 c0 = sample_cube(chain + cube_level_offset_floats(S, l0) / 4, s0, dir);
    const f3 c1 = sample_cube(chain + cube_level_offset_floats(S, l1) / 4, s1, dir);
    return {(1.0f - d) * c0.x + d * c1.x, (1.0f - d) * c0.y + d * c1.y, (1.0f - d) * c0.z + d * c1.z};
}

// n samples: direction uniform on the sphere, lod uniform in [0, lod_max];
// target log(textureLod(chain, d, lod) + eps) per channel
__global__ __launch_bounds__(256) void mlp_data_kernel(const float4* __restrict__ chain, uint32_t S, uint32_t mips,
                                                       float lod_max, uint64_t seed, uint32_t n,
                                                       float4* __restrict__ in, float4* __restrict__ tgt) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float z = 2.0f * u01(seed, 0, i) - 1.0f, ph = 6.2831853071795864f * u01(seed, 1, i);
    const float r = sqrtf(fmaxf(1.0f - z * z, 0.0f));
    const f3 d = {r * cosf(ph), r * sinf(ph), z};
    const float lod = lod_max * u01(seed, 2, i);
    const f3 c = chain_lod(chain, S, mips, d, lod);
    const float e = (float)hvx::kMlpEps;
    in[i] = make_float4(d.x, d.y, d.z, lod);
    tgt[i] = make_float4(logf(fmaxf(c.x, 0.0f) + e), logf(fmaxf(c.y, 0.0f) + e), logf(fmaxf(c.z, 0.0f) + e), 0.0f);
}

// ----------------------------------------------------------------- encoding
// Sixteen threads per sample, each one 16-byte store of its row of X (8 of the
// 128 features), so a wave writes 1 KB in one piece; rows >= n are the
// encoding of 0. XT (may be null): the transposed copy the weight-gradient
// GEMM of the separate launches reads.
__global__ __launch_bounds__(256) void mlp_pe_kernel(const float4* __restrict__ in, uint32_t n, uint32_t B,
                                                     float lod_max, bf16* __restrict__ X, bf16* __restrict__ XT) {
    const uint32_t j = threadIdx.x / 4 % 4, g = threadIdx.x % 4;
    for (size_t b = (size_t)blockIdx.x * 16 + threadIdx.x / 16; b < B; b += (size_t)gridDim.x * 16) {
        float x = 0.0f;
        if (b < n) {
            const float4 v = in[b];
            x = j == 0 ? v.x : (j == 1 ? v.y : (j == 2 ? v.z : 2.0f * v.w / lod_max - 1.0f));
        }
        // frequencies 4 g .. 4 g + 3 of input j, as mlp_sincos evaluates them
        float sv[4], cv[4];
        hvx::mlp_sincos_direct(x, (int)(4 * g), sv[0], cv[0]);
        hvx::mlp_sincos_direct(x, (int)(4 * g + 1), sv[1], cv[1]);
        hvx::mlp_sincos_double(sv[0], cv[0], sv[2], cv[2]);
        hvx::mlp_sincos_double(sv[1], cv[1], sv[3], cv[3]);
        bf16x8 pk;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            pk[2 * q] = (bf16)sv[q];
            pk[2 * q + 1] = (bf16)cv[q];
        }
        reinterpret_cast<bf16x8*>(X)[b * (kIn / 8) + 4 * j + g] = pk;
        if (XT)
#pragma unroll
            for (int q = 0; q < 8; ++q) XT[(size_t)(32 * j + 8 * g + q) * B + b] = pk[q];
    }
}

// -------------------------------------------------------------------- GEMM
enum Epi { EPI_FWD = 0, EPI_BWD = 1, EPI_PART = 2 };

struct GemmArgs {
    const bf16* A;   // [M][Kd]
    const bf16* Bt;  // [Nc][Kd]
    uint32_t M, Nc, Kd, splitk;
    uint32_t ldb;       // elements between the rows of Bt
    const float* bias;  // FWD: [Nc]
    const bf16* mask;   // BWD: [M][Nc], zero where <= 0
    bf16* C;            // FWD/BWD: [M][Nc]
    bf16* CT;           // FWD/BWD: [Nc][M]
    float* part;        // PART: per slice [M][Nc] then (colsum) [M], slices pstride apart
    uint32_t pstride;   // PART: floats per slice
    uint32_t colsum;    // PART: also sum A's rows over K (the bias gradient)
};

// A wave computes a 16 x 64 block of C over one K slice.
template <int EPI>
__device__ __forceinline__ void gemm_abt_wave(const GemmArgs& g, uint32_t wave, uint32_t lane) {
    const uint32_t rts = g.M / 16, cgs = g.Nc / 64;
    if (wave >= rts * cgs * g.splitk) return;  // uniform per wave; no barriers below
    const uint32_t slice = wave % g.splitk, t = wave / g.splitk, cg = t % cgs, rt = t / cgs;
    const uint32_t ks = g.Kd / 32;
    const uint32_t kb = slice * ks / g.splitk, ke = (slice + 1) * ks / g.splitk;
    const uint32_t i = lane & 15, gq = lane >> 4;
    const bf16* ap = g.A + (size_t)(rt * 16 + i) * g.Kd + 8 * gq;
    const bf16* bp = g.Bt + (size_t)(cg * 64 + i) * g.ldb + 8 * gq;
    const size_t bstep = (size_t)16 * g.ldb;
    f32x4 acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // PART with colsum: the waves of column group 0 also sum the A elements
    // they load (row rt * 16 + i, this lane's 8 of every 32 K)
    const bool rowsum = EPI == EPI_PART && g.colsum && cg == 0;
    float rs = 0.0f;
    for (uint32_t s = kb; s < ke; ++s) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(ap + 32 * s);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(bp + nb * bstep + 32 * s);
            acc[nb] = hvx::mfma16x16x32(a, b, acc[nb]);
        }
        if (rowsum) {
            float t = 0.0f;
#pragma unroll
            for (int q = 0; q < 8; ++q) t += (float)a[q];
            rs += t;
        }
    }
    if (rowsum) {  // the four lanes of row i hold disjoint K subsets
        rs += __shfl_xor(rs, 16, 64);
        rs += __shfl_xor(rs, 32, 64);
        if (gq == 0) g.part[(size_t)slice * g.pstride + g.M * g.Nc + rt * 16 + i] = rs;
    }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const uint32_t col = cg * 64 + nb * 16 + i;
        bf16 ht[4];  // rows 4 gq .. 4 gq + 3 of column col: one 8-byte store into CT
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t row = rt * 16 + 4 * gq + r;
            float v = acc[nb][r];
            if (EPI == EPI_PART) {
                g.part[(size_t)slice * g.pstride + (size_t)row * g.Nc + col] = v;
            } else {
                if (EPI == EPI_FWD) v = fmaxf(v + g.bias[col], 0.0f);
                else if (!((float)g.mask[(size_t)row * g.Nc + col] > 0.0f)) v = 0.0f;
                const bf16 h = (bf16)v;
                g.C[(size_t)row * g.Nc + col] = h;
                ht[r] = h;
            }
        }
        if (EPI != EPI_PART) {
            typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<bf16x4*>(g.CT + (size_t)col * g.M + rt * 16 + 4 * gq) = bf16x4{ht[0], ht[1], ht[2], ht[3]};
        }
    }
}

template <int EPI>
__global__ __launch_bounds__(256) void gemm_abt_kernel(GemmArgs g) {
    gemm_abt_wave<EPI>(g, blockIdx.x * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
}

// ------------------------------------------------------- output and loss
constexpr int kOutPart = kH * 3 + 3 + 1;  // dW4, db4, loss
// samples per output-layer block: the loss and the output layer's gradient
// are summed per block of this many samples, then over the blocks in order
constexpr uint32_t kOutBlock = 128;

// Training: one thread per sample (B a multiple of kOutBlock). Evaluation
// (TRAIN false): writes radiance exp(y) - eps for samples < n.
template <bool TRAIN>
__global__ __launch_bounds__(kOutBlock) void mlp_out_kernel(const bf16* __restrict__ H3, const float* __restrict__ P,
                                                      const float4* __restrict__ tgt, uint32_t n, uint32_t B,
                                                      float inv_norm, float* __restrict__ Y, bf16* __restrict__ dZ,
                                                      bf16* __restrict__ dZT, float* __restrict__ part) {
    __shared__ float sdY[kOutBlock][3];
    __shared__ float sl[kOutBlock];
    __shared__ bf16 sh3[kH][kOutBlock + 8];  // the block's H3 transposed (padded rows)
    const uint32_t t = threadIdx.x, b = blockIdx.x * kOutBlock + t;
    const float* W4 = P + hvx::kMlpW4;
    const float* b4 = P + hvx::kMlpB4;
    float h[kH];
    const bf16x8* hrow = reinterpret_cast<const bf16x8*>(H3 + (size_t)b * kH);
#pragma unroll
    for (int k8 = 0; k8 < kH / 8; ++k8) {
        const bf16x8 v = hrow[k8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            h[8 * k8 + q] = (float)v[q];
            if (TRAIN) sh3[8 * k8 + q][t] = v[q];
        }
    }
    float y[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) y[c] = hvx::mlp_output(h, W4 + c * kH, b4[c]);
    if (!TRAIN) {
        if (b < n)
            for (int c = 0; c < 3; ++c) Y[(size_t)b * 3 + c] = expf(y[c]) - (float)hvx::kMlpEps;
        return;
    }
    const float4 tv = tgt[b];
    const float e0 = y[0] - tv.x, e1 = y[1] - tv.y, e2 = y[2] - tv.z;
    sdY[t][0] = e0 * inv_norm;
    sdY[t][1] = e1 * inv_norm;
    sdY[t][2] = e2 * inv_norm;
    sl[t] = (e0 * e0 + e1 * e1) + e2 * e2;
#pragma unroll
    for (int k8 = 0; k8 < kH / 8; ++k8) {
        bf16x8 pk;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int k = 8 * k8 + q;
            const float dh = (sdY[t][0] * W4[k] + sdY[t][1] * W4[kH + k]) + sdY[t][2] * W4[2 * kH + k];
            const bf16 v = (bf16)(h[k] > 0.0f ? dh : 0.0f);
            pk[q] = v;
            dZT[(size_t)k * B + b] = v;
        }
        reinterpret_cast<bf16x8*>(dZ + (size_t)b * kH)[k8] = pk;
    }
    __syncthreads();
    float* pp = part + (size_t)blockIdx.x * kOutPart;
    for (uint32_t o = t; o < (uint32_t)kOutPart - 1; o += kOutBlock) {
        float acc = 0.0f;
        if (o < 3 * kH) {
            const uint32_t c = o / kH, k = o % kH;
            for (uint32_t j = 0; j < kOutBlock; ++j) acc += sdY[j][c] * (float)sh3[k][j];
        } else {
            const uint32_t c = o - 3 * kH;
            for (uint32_t j = 0; j < kOutBlock; ++j) acc += sdY[j][c];
        }
        pp[o] = acc;
    }
    for (uint32_t hh = kOutBlock / 2; hh > 0; hh >>= 1) {
        __syncthreads();
        if (t < hh) sl[t] += sl[t + hh];
    }
    if (t == 0) pp[kOutPart - 1] = sl[0];
}


// The output layer's block partials (kOutPart per block: dW4, db4, loss):
// a workgroup takes 64 of them and 16 block ranges (one per wave), each
// summed in block order, then adds the 16 range sums in a fixed tree; dW4
// and db4 into out, the loss (scaled) into *loss when asked for
constexpr uint32_t kOutRedGroups = 16;
__global__ __launch_bounds__(64 * kOutRedGroups) void reduce_out_kernel(const float* __restrict__ part,
                                                                        uint32_t blocks, float* __restrict__ out,
                                                                        float loss_scale, float* __restrict__ loss) {
    __shared__ float sh[kOutRedGroups][64];
    const uint32_t l = threadIdx.x & 63, gq = threadIdx.x >> 6, i = blockIdx.x * 64 + l;
    float acc = 0.0f;
    if (i < (uint32_t)kOutPart) {
        const uint32_t s0 = gq * blocks / kOutRedGroups, s1 = (gq + 1) * blocks / kOutRedGroups;
#pragma unroll 4
        for (uint32_t s = s0; s < s1; ++s) acc += part[(size_t)s * kOutPart + i];
    }
    sh[gq][l] = acc;
    for (uint32_t h = kOutRedGroups / 2; h > 0; h >>= 1) {
        __syncthreads();
        if (gq < h) sh[gq][l] += sh[gq + h][l];
    }
    if (gq != 0 || i >= (uint32_t)kOutPart) return;
    if (i < (uint32_t)kOutPart - 1) out[i] = sh[0][l];
    else if (loss) *loss = sh[0][l] * loss_scale;
}

// ------------------------------------------------ fused per-sample step
// A training step of a slice of the batch, by blocks of kOutBlock samples:
// forward, output layer, backward and the slice's gradient partials, with
// every activation and gradient in LDS (131 KB: one workgroup per CU). Every
// product is the MFMA sequence of gemm_abt_wave over the same BF16 operands,
// and the output part is mlp_out_kernel's, so the results equal those separate
// launches bit for bit.
//
// 128 samples are 0.1 us of matrix work in a chain of eight dependent
// products, so the time is latency and the 17 MB of partials. Every global
// read (the block's encodings, the weights of all five products, one 16-unit
// column per wave) is asked for at the start, and a stage is an LDS round trip
// and a barrier. Wave w computes units 16 (w & 3) .. of rows 64 (w >> 2) ..;
// the products and their derivatives have the same lanes, so the ReLU masks
// are 16 bits of a register. The gradient GEMMs read the row-major activations
// through transposing LDS reads (a second, transposed copy took two-byte
// writes, 7,800 cycles for the encodings alone), and the partials are stored
// past the L2, whose write-back at the end of the launch cost 2.4 us.
//
// A step of 32,768 samples: 53 us (step 29.6, gradient GEMMs over activations
// in memory 14.3, reductions 5.6, Adam 4.8) -> 21.7 us (step 16.0, reductions
// with Adam 5.6). Without the partials' stores the step is 12.7 us, without
// its reads and dW4's serial sums too 9.9: the chain.
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kStepThreads = 512;

// The step's weights as the matrix operands: fragment (16-row tile nb, 32-K
// block s) of a product is 64 lanes x 8 values in one piece, so a wave's load
// is eight whole lines (as rows of W it took half of sixteen: the loads of a
// workgroup took 13,000 cycles, so 7,500).
constexpr uint32_t kWs1 = 0, kWs2 = kH * kIn, kWs3 = kWs2 + kH * kH, kWs3T = kWs3 + kH * kH, kWs2T = kWs3T + kH * kH,
                   kWsLen = kWs2T + kH * kH;
__device__ __forceinline__ uint32_t operand_index(uint32_t row, uint32_t k, uint32_t K) {
    return ((row / 16 * (K / 32) + k / 32) * 64 + (k % 32 / 8) * 16 + row % 16) * 8 + k % 8;
}
// BF16 copies of parameter i: the rows W1..W3, the operands of the step and, if
// set, the transposes of W2 and W3 ([in][out]) for the separate launches
struct WeightCopies {
    bf16 *W1, *W2, *W3, *Ws, *W2T, *W3T;
};
__device__ __forceinline__ void write_copies(const WeightCopies& c, uint32_t i, bf16 h) {
    if (i - (uint32_t)hvx::kMlpW1 < (uint32_t)(kH * kIn)) {
        const uint32_t j = i - hvx::kMlpW1;
        c.W1[j] = h;
        c.Ws[kWs1 + operand_index(j / kIn, j % kIn, kIn)] = h;
    }
    if (i - (uint32_t)hvx::kMlpW2 < (uint32_t)(kH * kH)) {
        const uint32_t j = i - hvx::kMlpW2, o = j / kH, k = j % kH;
        c.W2[j] = h;
        c.Ws[kWs2 + operand_index(o, k, kH)] = h;
        c.Ws[kWs2T + operand_index(k, o, kH)] = h;
        if (c.W2T) c.W2T[k * kH + o] = h;
    }
    if (i - (uint32_t)hvx::kMlpW3 < (uint32_t)(kH * kH)) {
        const uint32_t j = i - hvx::kMlpW3, o = j / kH, k = j % kH;
        c.W3[j] = h;
        c.Ws[kWs3 + operand_index(o, k, kH)] = h;
        c.Ws[kWs3T + operand_index(k, o, kH)] = h;
        if (c.W3T) c.W3T[k * kH + o] = h;
    }
}

// LDS matrices [sample][unit or feature] (and h3t [unit][sample]) without
// padding: the 16-byte chunks of a row are exchanged by a pattern of the row's
// low bits such that the sixteen rows of an operand read, the eight rows x two
// chunks of a transposing read and the rows of a write meet all 64 banks once.
struct StepShared {
    __align__(16) bf16 x[kOutBlock * kIn];
    __align__(16) bf16 h1[kOutBlock * kH], h2[kOutBlock * kH], h3[kOutBlock * kH], z3[kOutBlock * kH],
        z2[kOutBlock * kH], h3t[kH * kOutBlock];
    float dy[3][kOutBlock], loss[kOutBlock];
    float bias[3][kH];
};
// element of chunk c of row r, W elements a row
template <int W> __device__ __forceinline__ uint32_t chunk_at(uint32_t r, uint32_t c) {
    static_assert(W == kH || W == kIn, "8 or 16 chunks");
    const uint32_t x = W == kH ? (r >> 2 & 1) | (r & 2) | (r >> 1 & 4) : (r >> 2 & 1) | (r & 3) << 1 | (r & 8);
    return r * W + ((c ^ x) << 3);
}
// chunk c of row r of h3t
__device__ __forceinline__ uint32_t chunk_t(uint32_t r, uint32_t c) { return r * kOutBlock + ((c ^ (r & 15)) << 3); }

// Row `row`'s 8 values from 32 s + 8 gq as an MFMA operand
template <int W>
__device__ __forceinline__ bf16x8 rows_operand(const bf16* m, uint32_t row, uint32_t s, uint32_t gq) {
    return *reinterpret_cast<const bf16x8*>(m + chunk_at<W>(row, 4 * s + gq));
}
// Column 16 ct + i, rows 32 s + 8 gq .. + 7, as an MFMA operand: two
// transposing reads (each takes 4 rows x 16 columns per 16 lanes, lane j
// addressing 4 columns of row j / 4, and returns column j).
template <int W>
__device__ __forceinline__ bf16x8 cols_operand(const bf16* m, uint32_t s, uint32_t ct, uint32_t i, uint32_t gq) {
    typedef __attribute__((address_space(3))) s16x4* lds;
    const uint32_t r = 32 * s + 8 * gq + (i >> 2), c = 2 * ct + (i >> 1 & 1), e = 4 * (i & 1);
    union {
        s16x4 s[2];
        bf16x8 v;
    } u;
    u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds)(m + chunk_at<W>(r, c) + e));
    u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds)(m + chunk_at<W>(r + 4, c) + e));
    return u.v;
}

// Partial of dW += dZ^T H over the block, for the 16 units of tile ut and NT
// tiles of 16 columns from tile c0: lane (g, i) holds unit 16 ut + i, columns
// 4 g .. of each tile. rs: the unit's sum of dZ over this lane's samples (the bias).
// [lo, hi): the block's steps of 32 samples that are the slice's.
template <int NT, int W>
__device__ __forceinline__ void step_partial(const bf16* z, const bf16* h, uint32_t ut, uint32_t c0, uint32_t i,
                                             uint32_t gq, uint32_t lo, uint32_t hi, f32x4 (&acc)[NT], float& rs) {
    auto step = [&](uint32_t s) {
        const bf16x8 zo = cols_operand<kH>(z, s, ut, i, gq);
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = hvx::mfma16x16x32(cols_operand<W>(h, s, c0 + n, i, gq), zo, acc[n]);
        float t = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += (float)zo[q];
        rs += t;
    };
    if (hi - lo == kOutBlock / 32) {
#pragma unroll
        for (uint32_t s = 0; s < kOutBlock / 32; ++s) step(s);
    } else {
#pragma unroll 1
        for (uint32_t s = lo; s < hi; ++s) step(s);
    }
}
template <int NT>
__device__ __forceinline__ void step_write_partial(float* part, uint32_t K, uint32_t ut, uint32_t c0, uint32_t i,
                                                   uint32_t gq, const f32x4 (&acc)[NT], float rs) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
        __builtin_nontemporal_store(
            acc[n], reinterpret_cast<f32x4*>(part + (size_t)(16 * ut + i) * K + 16 * (c0 + n) + 4 * gq));
    rs += __shfl_xor(rs, 16, 64);
    rs += __shfl_xor(rs, 32, 64);
    if (c0 == 0 && gq == 0) part[(size_t)kH * K + 16 * ut + i] = rs;
}

// X: [blocks * kOutBlock][kIn] encodings; Ws: the weights in operand order;
// slice q of the launch sums steps of 32 samples from q * steps / slices on
// (gemm_abt_wave's slices); a block that two slices share is evaluated for
// both, and its output-layer partials are those of the slice with its first
// step. part: per layer, then slice, [kH][K] and the bias gradient [kH]; opart:
// [blocks][kOutPart]
constexpr uint32_t kLen1 = kH * kIn + kH, kLen23 = kH * kH + kH;  // a layer's partial
// WHOLE: every slice is whole blocks.
template <bool WHOLE>
__global__ __launch_bounds__(kStepThreads) void mlp_step_kernel(const bf16* __restrict__ X, const float* __restrict__ P,
                                                                const bf16* __restrict__ Ws,
                                                                const float4* __restrict__ tgt, uint32_t blocks,
                                                                float inv_norm, float* __restrict__ part,
                                                                float* __restrict__ opart) {
    __shared__ StepShared sh;
    const uint32_t t = threadIdx.x;
    uint32_t lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6), nb = wave & 3, r0 = (wave >> 2) * 64;
    const uint32_t ut = wave >> 1, ch = wave & 1;   // its tile of units and half of the columns in the partials
    const uint32_t tg = wave >> 1;                  // output layer: unit group (as mlp_output's g)

    // the encodings: wave w fetches rows 16 w ..
    bf16x8 x[4];
    float4 tv;
    auto fetch = [&](uint32_t q) {
        const bf16* xp = X + ((size_t)q * kOutBlock + 16 * wave) * kIn;
#pragma unroll
        for (int s = 0; s < 4; ++s) x[s] = *reinterpret_cast<const bf16x8*>(xp + 4 * s * kIn + 8 * lane);
        tv = tgt[(size_t)q * kOutBlock + (wave & 1) * 64 + lane];
    };
    constexpr uint32_t kSteps = kOutBlock / 32;
    const uint32_t k0 = blockIdx.x * (blocks * kSteps) / gridDim.x, k1 = (blockIdx.x + 1) * (blocks * kSteps) / gridDim.x;
    const uint32_t q0 = k0 / kSteps, q1 = (k1 + kSteps - 1) / kSteps;
    if (!WHOLE && k0 == k1) {  // a slice of no steps (uniform over the workgroup)
        const f32x4 none[4] = {};
        const f32x4 none2[2] = {};
        const size_t sl = blockIdx.x, n = gridDim.x;
        const uint32_t i = lane & 15, gq = lane >> 4;
        step_write_partial<2>(part + n * (kLen1 + kLen23) + sl * kLen23, kH, ut, 2 * ch, i, gq, none2, 0.0f);
        step_write_partial<2>(part + n * kLen1 + sl * kLen23, kH, ut, 2 * ch, i, gq, none2, 0.0f);
        step_write_partial<4>(part + sl * kLen1, kIn, ut, 4 * ch, i, gq, none, 0.0f);
        return;
    }
    fetch(q0);
    // this wave's fragment s of a product's weights
    auto weights = [&](uint32_t ofs, uint32_t frags, uint32_t s) {
        return *reinterpret_cast<const bf16x8*>(Ws + ofs + (nb * frags + s) * 512 + 8 * lane);
    };
    bf16x8 w1[4], w2[2], w3[2], w3t[2], w2t[2];
#pragma unroll
    for (uint32_t s = 0; s < 4; ++s) w1[s] = weights(kWs1, 4, s);
#pragma unroll
    for (uint32_t s = 0; s < 2; ++s) {
        w2[s] = weights(kWs2, 2, s);
        w3[s] = weights(kWs3, 2, s);
        w3t[s] = weights(kWs3T, 2, s);
        w2t[s] = weights(kWs2T, 2, s);
    }
    const uint32_t bl = t / kH;  // threads 0 .. 191: the biases
    const float bias = t < 3 * kH ? P[(bl == 0 ? hvx::kMlpB1 : (bl == 1 ? hvx::kMlpB2 : hvx::kMlpB3)) + t % kH] : 0.0f;
    float w4[3][16], b4[3];  // output weights of the thread's 16 units (uniform over the wave)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        b4[c] = P[hvx::kMlpB4 + c];
#pragma unroll
        for (int j = 0; j < 16; ++j) w4[c][j] = P[hvx::kMlpW4 + c * kH + 16 * (j >> 2) + 4 * tg + (j & 3)];
    }
    __builtin_amdgcn_sched_barrier(0);  // every read above is on its way before the first wait
    if (t < 3 * kH) sh.bias[bl][t % kH] = bias;

    const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 p1[4] = {zero, zero, zero, zero}, p2[2] = {zero, zero}, p3[2] = {zero, zero};
    float rs1 = 0.0f, rs2 = 0.0f, rs3 = 0.0f;
#pragma unroll 1
    for (uint32_t q = q0; q < q1; ++q) {
        if (q > q0) __syncthreads();  // the block before has been read
        // the LDS addresses are made anew for every block: hoisted out of the
        // loop they take more registers than there are
        __asm__ volatile("" : "+v"(lane));
        const uint32_t i = lane & 15, gq = lane >> 4, ts = (wave & 1) * 64 + lane;
        const uint32_t un = 16 * nb + 4 * gq;  // this lane's four units in the forward and backward products
#pragma unroll
        for (int s = 0; s < 4; ++s)
            *reinterpret_cast<bf16x8*>(sh.x + chunk_at<kIn>(16 * wave + 4 * s + gq, i)) = x[s];
        const float want[3] = {tv.x, tv.y, tv.z};
        if (q + 1 < q1) fetch(q + 1);
        __syncthreads();
        // 64 rows of a product: units un .. of row r0 + 16 rt + i
        uint32_t m1 = 0, m2 = 0, m3 = 0;
        auto put = [&](bf16x4 h, int rt, bf16* out) {
            *reinterpret_cast<bf16x4*>(out + chunk_at<kH>(r0 + 16 * rt + i, un >> 3) + (un & 4)) = h;
        };
        auto relu = [&](const f32x4 (&acc)[4], int l, uint32_t& mask, bf16* out) {
            const f32x4 b = *reinterpret_cast<const f32x4*>(&sh.bias[l][un]);
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h[r] = (bf16)fmaxf(acc[rt][r] + b[r], 0.0f);
                    mask |= (float)h[r] > 0.0f ? 1u << (4 * rt + r) : 0u;
                }
                put(h, rt, out);
            }
        };
        auto masked = [&](const f32x4 (&acc)[4], uint32_t mask, bf16* out) {
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) h[r] = (bf16)(mask >> (4 * rt + r) & 1u ? acc[rt][r] : 0.0f);
                put(h, rt, out);
            }
        };
        auto product = [&](const bf16* in, const bf16x8 (&w)[2], f32x4 (&acc)[4]) {
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                acc[rt] = zero;
#pragma unroll
                for (uint32_t s = 0; s < 2; ++s)
                    acc[rt] = hvx::mfma16x16x32(w[s], rows_operand<kH>(in, r0 + 16 * rt + i, s, gq), acc[rt]);
            }
        };
        f32x4 acc[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            acc[rt] = zero;
#pragma unroll
            for (uint32_t s = 0; s < 4; ++s)
                acc[rt] = hvx::mfma16x16x32(w1[s], rows_operand<kIn>(sh.x, r0 + 16 * rt + i, s, gq), acc[rt]);
        }
        relu(acc, 0, m1, sh.h1);
        __syncthreads();
        product(sh.h1, w2, acc);
        relu(acc, 1, m2, sh.h2);
        __syncthreads();
        product(sh.h2, w3, acc);
        relu(acc, 2, m3, sh.h3);
        __syncthreads();
        // output layer: a quarter of a sample's units per thread, in the order
        // of mlp_output; the partial sums meet in z2. H3's transpose for dW4.
        float(*py)[3][kOutBlock] = reinterpret_cast<float(*)[3][kOutBlock]>(sh.z2);
        static_assert(sizeof(sh.z2) >= 4 * 3 * kOutBlock * sizeof(float), "partial sums fit");
        float h3[16];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const bf16x4 h = *reinterpret_cast<const bf16x4*>(sh.h3 + chunk_at<kH>(ts, 2 * j + (tg >> 1)) + 4 * (tg & 1));
#pragma unroll
            for (int r = 0; r < 4; ++r) h3[4 * j + r] = (float)h[r];
        }
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s)
            *reinterpret_cast<bf16x8*>(sh.h3t + chunk_t(16 * ut + i, 4 * (2 * ch + s) + gq)) =
                cols_operand<kH>(sh.h3, 2 * ch + s, ut, i, gq);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            float v = h3[0] * w4[c][0];
#pragma unroll
            for (int j = 1; j < 16; ++j) v = v + h3[j] * w4[c][j];
            py[tg][c][ts] = v;
        }
        __syncthreads();
        // the loss and dZ3
        {
            float e[3], dy[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                e[c] = ((py[0][c][ts] + py[1][c][ts]) + (py[2][c][ts] + py[3][c][ts])) + b4[c] - want[c];
                dy[c] = e[c] * inv_norm;
            }
            if (tg == 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) sh.dy[c][ts] = dy[c];
                sh.loss[ts] = (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2];
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                bf16x4 z;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = 4 * j + r;
                    const float dh = (dy[0] * w4[0][k] + dy[1] * w4[1][k]) + dy[2] * w4[2][k];
                    z[r] = (bf16)(h3[k] > 0.0f ? dh : 0.0f);
                }
                *reinterpret_cast<bf16x4*>(sh.z3 + chunk_at<kH>(ts, 2 * j + (tg >> 1)) + 4 * (tg & 1)) = z;
            }
        }
        __syncthreads();
        // dZ2, the partials of layer 3 and of the output layer
        product(sh.z3, w3t, acc);
        masked(acc, m2, sh.z2);
        float* pp = opart + (size_t)q * kOutPart;
        const uint32_t lo = WHOLE ? 0 : max(k0, kSteps * q) - kSteps * q,
                       hi = WHOLE ? kSteps : min(k1 - kSteps * q, kSteps);
        if (!WHOLE && kSteps * q < k0) {
            // the slice before has written them
        } else if (wave < 3) {  // dW4[wave][lane]: the samples in order
            float sum = 0.0f;
#pragma unroll 1
            for (uint32_t c0 = 0; c0 < kOutBlock / 8; c0 += 4) {
                bf16x8 h[4];
                f32x4 d[8];
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) {
                    h[c] = *reinterpret_cast<const bf16x8*>(sh.h3t + chunk_t(lane, c0 + c));
                    d[2 * c] = *reinterpret_cast<const f32x4*>(&sh.dy[wave][8 * (c0 + c)]);
                    d[2 * c + 1] = *reinterpret_cast<const f32x4*>(&sh.dy[wave][8 * (c0 + c) + 4]);
                }
#pragma unroll
                for (uint32_t j = 0; j < 32; ++j) sum += d[j / 4][j % 4] * (float)h[j / 8][j % 8];
            }
            pp[wave * kH + lane] = sum;
        } else if (wave == 3) {
            if (lane < 3) {
                float sum = 0.0f;
#pragma unroll 8
                for (uint32_t j = 0; j < kOutBlock; j += 4) {
                    const f32x4 d = *reinterpret_cast<const f32x4*>(&sh.dy[lane][j]);
                    sum += d[0];
                    sum += d[1];
                    sum += d[2];
                    sum += d[3];
                }
                pp[3 * kH + lane] = sum;
            }
        } else if (wave == 4) {
            float v = sh.loss[lane] + sh.loss[lane + 64];
            for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
            if (lane == 0) pp[kOutPart - 1] = v;
        }
        step_partial<2, kH>(sh.z3, sh.h2, ut, 2 * ch, i, gq, lo, hi, p3, rs3);
        const bool last = q + 1 == q1;
        const size_t sl = blockIdx.x, n = gridDim.x;
        if (last) step_write_partial<2>(part + n * (kLen1 + kLen23) + sl * kLen23, kH, ut, 2 * ch, i, gq, p3, rs3);
        __syncthreads();
        // dZ1 (over dZ3) and the partials of layer 2
        product(sh.z2, w2t, acc);
        masked(acc, m1, sh.z3);
        step_partial<2, kH>(sh.z2, sh.h1, ut, 2 * ch, i, gq, lo, hi, p2, rs2);
        if (last) step_write_partial<2>(part + n * kLen1 + sl * kLen23, kH, ut, 2 * ch, i, gq, p2, rs2);
        __syncthreads();
        step_partial<4, kIn>(sh.z3, sh.x, ut, 4 * ch, i, gq, lo, hi, p1, rs1);
        if (last) step_write_partial<4>(part + sl * kLen1, kIn, ut, 4 * ch, i, gq, p1, rs1);
    }
}

// Sum over the slices of part[s * stride + i] for i < len: a workgroup takes
// 64 outputs and 16 slice ranges (one per wave), each summed in slice order,
// then adds the 16 range sums in a fixed tree. True for the lane that then
// holds output i's sum.
constexpr uint32_t kRedGroups = 16;
__device__ __forceinline__ bool reduce_slices_block(const float* __restrict__ part, uint32_t slices, uint32_t len,
                                                    uint32_t i, float& sum) {
    __shared__ float sh[kRedGroups][64];
    const uint32_t l = threadIdx.x & 63, gq = threadIdx.x >> 6;
    float acc = 0.0f;
    if (i < len) {
        const uint32_t s0 = gq * slices / kRedGroups, s1 = (gq + 1) * slices / kRedGroups;
#pragma unroll 16
        for (uint32_t s = s0; s < s1; ++s) acc += part[(size_t)s * len + i];
    }
    sh[gq][l] = acc;
    __syncthreads();
    if (gq != 0 || i >= len) return false;
    float v[kRedGroups];
#pragma unroll
    for (uint32_t k = 0; k < kRedGroups; ++k) v[k] = sh[k][l];
#pragma unroll
    for (uint32_t h = kRedGroups / 2; h > 0; h >>= 1)
#pragma unroll
        for (uint32_t k = 0; k < h; ++k) v[k] += v[k + h];
    sum = v[0];
    return true;
}
__global__ __launch_bounds__(64 * kRedGroups) void reduce_slices_kernel(const float* __restrict__ part,
                                                                         uint32_t slices, uint32_t len,
                                                                         float* __restrict__ out) {
    const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63);
    float sum;
    if (reduce_slices_block(part, slices, len, i, sum)) out[i] = sum;
}

// Adam step of parameter i; an updated weight also refreshes its BF16 working
// copies, so a step needs no cast launch.
struct AdamArgs {
    float *P, *m, *v;
    float lr, bc1, bc2;
    WeightCopies copies;
};
struct AdamState {
    float p, m, v;
};
__device__ __forceinline__ AdamState adam_load(const AdamArgs& a, uint32_t i) { return {a.P[i], a.m[i], a.v[i]}; }
__device__ __forceinline__ void adam_update(const AdamArgs& a, uint32_t i, const AdamState& s, float g) {
    const float mi = 0.9f * s.m + 0.1f * g, vi = 0.999f * s.v + 0.001f * g * g;
    a.m[i] = mi;
    a.v[i] = vi;
    const float p = s.p - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + 1e-8f);
    a.P[i] = p;
    write_copies(a.copies, i, (bf16)p);
}
__global__ __launch_bounds__(256) void adam_kernel(AdamArgs a, const float* __restrict__ G, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) adam_update(a, i, adam_load(a, i), G[i]);
}

// A step's reductions in one launch: segment k (blocks [b[k], b[k + 1]))
// reduces len[k] outputs over slices[k] partials: the three layers' weight
// and bias gradients and the output layer's block partials, whose last element
// is the loss (scaled by loss_scale into *loss when it is set). The others
// are gradients of the parameters from ofs[k] on: into G or, with ADAM,
// straight into the parameters, which nothing else in this launch reads.
struct ReduceStep {
    const float* part[4];
    uint32_t ofs[4], len[4], slices[4], b[5];
    float *G, *loss;
    float loss_scale;
    AdamArgs adam;
};
template <bool ADAM> __global__ __launch_bounds__(64 * kRedGroups) void reduce_step_kernel(ReduceStep r) {
    const uint32_t blk = blockIdx.x;
    uint32_t k = 0;
    while (k < 3 && blk >= r.b[k + 1]) ++k;
    const uint32_t i = (blk - r.b[k]) * 64 + (threadIdx.x & 63), len = r.len[k], at = r.ofs[k] + i;
    const bool is_loss = k == 3 && i == len - 1;
    // the state is on its way while the partials are summed
    AdamState st{};
    if (ADAM && threadIdx.x < 64 && i < len && !is_loss) st = adam_load(r.adam, at);
    float sum;
    if (!reduce_slices_block(r.part[k], r.slices[k], len, i, sum)) return;
    if (is_loss) {
        if (r.loss) *r.loss = sum * r.loss_scale;
    } else if (ADAM) {
        adam_update(r.adam, at, st, sum);
    } else {
        r.G[at] = sum;
    }
}

// The BF16 working copies of every weight
__global__ __launch_bounds__(256) void mlp_cast_kernel(const float* __restrict__ P, WeightCopies c) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < (uint32_t)hvx::kMlpParams) write_copies(c, i, (bf16)P[i]);
}
// Inference through the in-shading path (mlp_device.h): each workgroup
// stages the weights once, its four waves evaluate kInferTiles x 16 samples
// per call. Bound by its vector instructions, 1,090 per 32 samples (512 of
// them the encoding): 2 million samples 549 -> 123 us, of which those are 110;
// one tile per call reads the weights twice as often (165 against 151 us before
// the encoding's quadrants became sign bits), three and four are no faster.
// Four waves per SIMD asked for: without it the accumulators go through the
// second register file (159 us).
constexpr int kInferTiles = 2;
constexpr uint32_t kInferStep = 64 * kInferTiles;  // samples per workgroup and step
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void mlp_infer_kernel(
    MlpView v, const float4* __restrict__ in, uint32_t n, float* __restrict__ rgb) {
    __shared__ MlpLds L;
    mlp_stage(L, v);
    __syncthreads();
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    for (size_t base = (size_t)blockIdx.x * kInferStep; base < n; base += (size_t)gridDim.x * kInferStep) {
        float x[kInferTiles][4], y[kInferTiles];
        size_t at[kInferTiles];
#pragma unroll
        for (int t = 0; t < kInferTiles; ++t) {
            at[t] = base + (wave * kInferTiles + t) * 16 + i;
            const float4 q = at[t] < n ? in[at[t]] : make_float4(0.0f, 0.0f, 1.0f, 0.0f);
            x[t][0] = q.x;
            x[t][1] = q.y;
            x[t][2] = q.z;
            x[t][3] = q.w;
        }
        mlp_forward_tiles(L, x, v.lod_max, y);
#pragma unroll
        for (int t = 0; t < kInferTiles; ++t)
            if (g < 3 && at[t] < n) rgb[at[t] * 3 + g] = y[t];
    }
}

// Fallback mask cells: (lod bin b, face f, texel y, x) of a mask_face cube.
// Points of a cell: a kMaskGrid x kMaskGrid grid over the texel (corners,
// edge and inner points) at the bin's two ends and middle.
constexpr uint32_t kMaskGrid = 5;
constexpr uint32_t kMaskPoints = kMaskGrid * kMaskGrid * 3;

__device__ __forceinline__ f3 plane_dir_f(int f, double u, double v) {
    double p[3];
    hvx::contract_face_point(f, u, v, p);
    return normalize3(f3{(float)p[0], (float)p[1], (float)p[2]});
}

__global__ __launch_bounds__(256) void mask_points_kernel(uint32_t mf, uint32_t bins, float lod_max,
                                                          float4* __restrict__ pts) {
    const uint32_t cells = bins * 6 * mf * mf;
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= cells * kMaskPoints) return;
    const uint32_t cell = id / kMaskPoints, p = id % kMaskPoints;
    const uint32_t x = cell % mf, y = (cell / mf) % mf, f = (cell / (mf * mf)) % 6, b = cell / (6 * mf * mf);
    const uint32_t gp = p % (kMaskGrid * kMaskGrid), li = p / (kMaskGrid * kMaskGrid);
    const double cx = x + (double)(gp % kMaskGrid) / (kMaskGrid - 1), cy = y + (double)(gp / kMaskGrid) / (kMaskGrid - 1);
    const f3 d = plane_dir_f((int)f, 2.0 * cx / mf - 1.0, 2.0 * cy / mf - 1.0);
    const float lod = lod_max * ((float)b + 0.5f * (float)li) / (float)bins;
    pts[id] = make_float4(d.x, d.y, d.z, lod);
}

// err[cell] = largest relative error (every channel, every point of the
// cell) of the network against the chain's textureLod value; infinity where
// the reference is 0 and the prediction is not. lo[cell] = per channel,
// kCellLowFactor times the smallest prediction over the cell's points: an
// estimate from below of what the network returns anywhere in the cell.
// Shading evaluates the network only where the cell could serve at that
// estimate and decides on the actual output, so the factor trades network
// evaluations against fragments served (3840x2160 frame, 15,000-step
// network: 1.0, 0.75 and 0.5 all serve 24.4 %, learned shading 2.34, 2.36
// and 2.41 ms).
#ifndef HVX_MLP_LO_FACTOR
#define HVX_MLP_LO_FACTOR 1.0f
#endif
constexpr float kCellLowFactor = HVX_MLP_LO_FACTOR;
__global__ __launch_bounds__(256) void cell_error_kernel(const float4* __restrict__ pts, const float* __restrict__ rgb,
                                                         const float4* __restrict__ chain, uint32_t S, uint32_t mips,
                                                         uint32_t cells, float* __restrict__ err,
                                                         float4* __restrict__ lo) {
    const uint32_t cell = blockIdx.x * 256 + threadIdx.x;
    if (cell >= cells) return;
    float e = 0.0f, mn[3] = {INFINITY, INFINITY, INFINITY};
    for (uint32_t p = 0; p < kMaskPoints; ++p) {
        const float4 q = pts[(size_t)cell * kMaskPoints + p];
        const f3 ref = chain_lod(chain, S, mips, f3{q.x, q.y, q.z}, q.w);
        const float* m = rgb + ((size_t)cell * kMaskPoints + p) * 3;
        const float r3[3] = {ref.x, ref.y, ref.z};
        for (int c = 0; c < 3; ++c) {
            const float d = fabsf(m[c] - r3[c]);
            float rel = d == 0.0f ? 0.0f : (r3[c] != 0.0f ? d / fabsf(r3[c]) : INFINITY);
            if (!(rel == rel)) rel = INFINITY;  // a NaN prediction fails every bound
            e = fmaxf(e, rel);
            mn[c] = fminf(mn[c], m[c]);
        }
    }
    err[cell] = e;
    float l3[3];
    for (int c = 0; c < 3; ++c) l3[c] = mn[c] > 0.0f ? kCellLowFactor * mn[c] : 0.0f;
    lo[cell] = make_float4(l3[0], l3[1], l3[2], 0.0f);
}

// The error the fallback decides on: the largest measured error of the cell
// times kCellSafety, a margin for the error between the test points, which
// is not measured.
constexpr float kCellSafety = 2.0f;
__global__ __launch_bounds__(256) void cell_margin_kernel(const float* __restrict__ raw, uint32_t cells,
                                                          float* __restrict__ err) {
    const uint32_t cell = blockIdx.x * 256 + threadIdx.x;
    if (cell < cells) err[cell] = raw[cell] * kCellSafety;
}

}  // namespace

struct hvx_mlp {
    hvx_ctx* ctx = nullptr;
    float lod_max = 1.0f;
    float *P = nullptr, *G = nullptr, *m = nullptr, *v = nullptr;
    bf16 *W1 = nullptr, *W2 = nullptr, *W3 = nullptr, *Ws = nullptr;
    bf16 *W2T = nullptr, *W3T = nullptr;
    bool transposes = false;  // W2T and W3T hold the weights: only the separate launches keep them so
    uint32_t cap = 0;  // batch capacity
    bf16* X0 = nullptr;
    float *part = nullptr, *opart = nullptr;
    uint32_t splitk = 1;
    // HVX_OPT_MLP_SEPARATE_LAUNCHES: the activations and gradients in memory
    uint32_t sep_cap = 0;
    bf16 *X0T = nullptr, *H[3] = {}, *HT[3] = {}, *dZa = nullptr, *dZaT = nullptr, *dZb = nullptr, *dZbT = nullptr;
    uint64_t steps_done = 0;
    // a training call's inputs encoded once: [n][kIn] and, for the separate
    // launches, transposed [kIn][n]
    bf16 *enc = nullptr, *encT = nullptr;
    size_t enc_cap = 0, encT_cap = 0;
    // per-cell estimate from below of the network's output, from the last
    // hvx_mlp_cell_errors call (cell grid lo_face x lo_face x lo_bins)
    float4* cell_lo = nullptr;  // RGB and a pad per cell
    uint32_t lo_face = 0, lo_bins = 0;
    std::vector<void*> batch_allocs, sep_allocs;
    std::vector<void*> allocs;
};

namespace hvx {
MlpView mlp_view(const hvx_mlp* M) { return MlpView{M->W1, M->W2, M->W3, M->P, M->lod_max}; }
const float4* mlp_cell_lower(const hvx_mlp* M, uint32_t cell_face, uint32_t lod_bins) {
    return M->cell_lo && M->lo_face == cell_face && M->lo_bins == lod_bins ? M->cell_lo : nullptr;
}
}  // namespace hvx

namespace {

int mfail(hvx_ctx* ctx, int st, const char* fmt, ...) __attribute__((format(printf, 3, 4)));
int mfail(hvx_ctx* ctx, int st, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (ctx) ctx->last_error = buf;
    return st;
}

template <class T> hipError_t dalloc(std::vector<void*>& list, T** p, size_t count) {
    void* q = nullptr;
    const hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
    if (e == hipSuccess) list.push_back(q);
    *p = static_cast<T*>(q);
    return e;
}

void encode(const float4* in, uint32_t n, uint32_t B, float lod_max, bf16* X, bf16* XT, hipStream_t s) {
    hipLaunchKernelGGL(mlp_pe_kernel, dim3(std::min((B + 15) / 16, 1u << 18)), dim3(256), 0, s, in, n, B, lod_max, X, XT);
}

hipError_t ensure_batch(hvx_mlp* M, uint32_t B) {
    const bool separate = M->ctx->mlp_separate != 0;
    if (B <= M->cap && (!separate || B <= M->sep_cap)) return hipSuccess;
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) return e;
    if (B > M->cap) {
        for (void* p : M->batch_allocs) (void)hipFree(p);
        M->batch_allocs.clear();
        M->cap = 0;
        auto& L = M->batch_allocs;
        // weight gradients are summed in slices of 128 samples of the largest
        // batch, up to 256 of them
        M->splitk = std::max(1u, std::min(256u, B / kOutBlock));
        if ((e = dalloc(L, &M->X0, (size_t)B * kIn)) ||
            (e = dalloc(L, &M->part, (size_t)M->splitk * (kLen1 + 2 * kLen23))) ||
            (e = dalloc(L, &M->opart, (size_t)(B / kOutBlock) * kOutPart)))
            return e;
        M->cap = B;
    }
    if (separate && B > M->sep_cap) {
        for (void* p : M->sep_allocs) (void)hipFree(p);
        M->sep_allocs.clear();
        M->sep_cap = 0;
        auto& L = M->sep_allocs;
        if ((e = dalloc(L, &M->X0T, (size_t)B * kIn))) return e;
        for (int l = 0; l < 3; ++l)
            if ((e = dalloc(L, &M->H[l], (size_t)B * kH)) || (e = dalloc(L, &M->HT[l], (size_t)B * kH))) return e;
        if ((e = dalloc(L, &M->dZa, (size_t)B * kH)) || (e = dalloc(L, &M->dZaT, (size_t)B * kH)) ||
            (e = dalloc(L, &M->dZb, (size_t)B * kH)) || (e = dalloc(L, &M->dZbT, (size_t)B * kH)))
            return e;
        M->sep_cap = B;
    }
    return hipSuccess;
}

template <int EPI> void gemm(const GemmArgs& g, hipStream_t s) {
    const uint32_t waves = (g.M / 16) * (g.Nc / 64) * g.splitk;
    hipLaunchKernelGGL(gemm_abt_kernel<EPI>, dim3((waves + 3) / 4), dim3(256), 0, s, g);
}

void cast(hvx_mlp* M, hipStream_t s) {
    hipLaunchKernelGGL(mlp_cast_kernel, dim3((hvx::kMlpParams + 255) / 256), dim3(256), 0, s, M->P,
                       WeightCopies{M->W1, M->W2, M->W3, M->Ws, M->W2T, M->W3T});
    M->transposes = true;
}

// A batch's encodings: rows X, columns XT (ld elements apart); null: to be made.
struct Encoded {
    const bf16 *X, *XT;
    uint32_t ld;
};

// forward of B samples, as separate launches
void forward(hvx_mlp* M, const float4* in, Encoded& x, uint32_t B, hipStream_t s) {
    if (!x.X) {
        encode(in, B, B, M->lod_max, M->X0, M->X0T, s);
        x = Encoded{M->X0, M->X0T, B};
    }
    const bf16* Ws[3] = {M->W1, M->W2, M->W3};
    const int bias[3] = {hvx::kMlpB1, hvx::kMlpB2, hvx::kMlpB3};
    const bf16* prev = x.X;
    for (int l = 0; l < 3; ++l) {
        GemmArgs g{};
        g.A = prev;
        g.Bt = Ws[l];
        g.M = B;
        g.Nc = kH;
        g.Kd = g.ldb = l == 0 ? kIn : kH;
        g.splitk = 1;
        g.bias = M->P + bias[l];
        g.C = M->H[l];
        g.CT = M->HT[l];
        gemm<EPI_FWD>(g, s);
        prev = M->H[l];
    }
}

// gradient of the mean squared log-radiance error over B samples into G (and
// the loss into *loss) as separate launches
void gradient_separate(hvx_mlp* M, const float4* in, Encoded x, const float4* tgt, uint32_t B, float* G, float* loss,
                       hipStream_t s) {
    if (!M->transposes) cast(M, s);
    forward(M, in, x, B, s);
    const uint32_t nblk = B / kOutBlock;
    hipLaunchKernelGGL(mlp_out_kernel<true>, dim3(nblk), dim3(kOutBlock), 0, s, M->H[2], M->P, tgt, B, B,
                       2.0f / (3.0f * (float)B), nullptr, M->dZa, M->dZaT, M->opart);
    hipLaunchKernelGGL(reduce_out_kernel, dim3((kOutPart + 63) / 64), dim3(64 * kOutRedGroups), 0, s, M->opart, nblk, G + hvx::kMlpW4,
                       1.0f / (3.0f * (float)B), loss);
    const int wofs[3] = {hvx::kMlpW1, hvx::kMlpW2, hvx::kMlpW3};
    const bf16* WT[3] = {nullptr, M->W2T, M->W3T};
    bf16 *dz = M->dZa, *dzT = M->dZaT, *nz = M->dZb, *nzT = M->dZbT;
    for (int l = 2; l >= 0; --l) {
        const uint32_t K = l == 0 ? kIn : kH;
        GemmArgs g{};
        g.A = dzT;
        g.Bt = l == 0 ? x.XT : M->HT[l - 1];
        g.M = kH;
        g.Nc = K;
        g.Kd = B;
        g.ldb = l == 0 ? x.ld : B;
        g.splitk = M->splitk;
        g.part = M->part;
        g.pstride = kH * K + kH;
        g.colsum = 1;
        gemm<EPI_PART>(g, s);
        // W_l and b_l are adjacent in the parameter vector: one reduction
        static_assert(hvx::kMlpB1 == hvx::kMlpW1 + kH * kIn && hvx::kMlpB2 == hvx::kMlpW2 + kH * kH &&
                          hvx::kMlpB3 == hvx::kMlpW3 + kH * kH,
                      "each layer's bias follows its weights");
        hipLaunchKernelGGL(reduce_slices_kernel, dim3((kH * K + kH + 63) / 64), dim3(64 * kRedGroups), 0, s,
                           M->part, M->splitk, (uint32_t)(kH * K + kH), G + wofs[l]);
        if (l > 0) {
            GemmArgs d{};
            d.A = dz;
            d.Bt = WT[l];
            d.M = B;
            d.Nc = kH;
            d.Kd = d.ldb = kH;
            d.splitk = 1;
            d.mask = M->H[l - 1];
            d.C = nz;
            d.CT = nzT;
            gemm<EPI_BWD>(d, s);
            std::swap(dz, nz);
            std::swap(dzT, nzT);
        }
    }
}

// The same gradient in two launches (and the encoding, if x0 does not hold
// it): mlp_step_kernel and the reduction of its partials, into G or, with
// adam set, straight into the parameters.
void gradient_fused(hvx_mlp* M, const float4* in, const bf16* x0, const float4* tgt, uint32_t B, float* G,
                    const AdamArgs* adam, float* loss, hipStream_t s) {
    if (!x0) encode(in, B, B, M->lod_max, M->X0, nullptr, s);
    const uint32_t blocks = B / kOutBlock, slices = M->splitk;
    const int wofs[4] = {hvx::kMlpW1, hvx::kMlpW2, hvx::kMlpW3, hvx::kMlpW4};
    ReduceStep r{};
    float* part = M->part;
    for (int l = 0; l < 4; ++l) {
        const uint32_t len = l == 3 ? kOutPart : (l == 0 ? kLen1 : kLen23);
        r.part[l] = l == 3 ? M->opart : part;
        r.ofs[l] = wofs[l];
        r.len[l] = len;
        r.slices[l] = l == 3 ? blocks : slices;
        r.b[l + 1] = r.b[l] + (len + 63) / 64;
        if (l < 3) part += (size_t)slices * len;
    }
    r.loss = loss;
    r.loss_scale = 1.0f / (3.0f * (float)B);
    r.G = G;
    if (adam) r.adam = *adam;
    hipLaunchKernelGGL(blocks % slices == 0 ? mlp_step_kernel<true> : mlp_step_kernel<false>, dim3(slices), dim3(kStepThreads), 0, s, x0 ? x0 : M->X0, M->P, M->Ws,
                       tgt, blocks, 2.0f / (3.0f * (float)B), M->part, M->opart);
    if (adam) hipLaunchKernelGGL(reduce_step_kernel<true>, dim3(r.b[4]), dim3(64 * kRedGroups), 0, s, r);
    else hipLaunchKernelGGL(reduce_step_kernel<false>, dim3(r.b[4]), dim3(64 * kRedGroups), 0, s, r);
}

int bind(hvx_ctx* ctx) {
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || (cur != ctx->device && hipSetDevice(ctx->device) != hipSuccess))
        return mfail(ctx, HVX_ERR_HIP, "cannot bind device %d", ctx->device);
    return HVX_OK;
}

}  // namespace

extern "C" {

int hvx_mlp_create(hvx_ctx* ctx, float lod_max, uint64_t seed, hvx_mlp** out) {
    if (!ctx || !out) return HVX_ERR_NULL;
    *out = nullptr;
    if (!(lod_max > 0.0f) || lod_max > 64.0f) return mfail(ctx, HVX_ERR_INVALID_ARG, "lod_max must be in (0, 64]");
    int st;
    if ((st = bind(ctx))) return st;
    hvx_mlp* M = new (std::nothrow) hvx_mlp();
    if (!M) return HVX_ERR_HIP;
    M->ctx = ctx;
    M->lod_max = lod_max;
    hipError_t e;
    auto& L = M->allocs;
    const size_t np = hvx::kMlpParams;
    if ((e = dalloc(L, &M->P, np)) || (e = dalloc(L, &M->G, np)) || (e = dalloc(L, &M->m, np)) ||
        (e = dalloc(L, &M->v, np)) || (e = dalloc(L, &M->W1, (size_t)kH * kIn)) ||
        (e = dalloc(L, &M->W2, (size_t)kH * kH)) || (e = dalloc(L, &M->W3, (size_t)kH * kH)) ||
        (e = dalloc(L, &M->Ws, (size_t)kWsLen)) || (e = dalloc(L, &M->W2T, (size_t)kH * kH)) ||
        (e = dalloc(L, &M->W3T, (size_t)kH * kH))) {
        hvx_mlp_destroy(M);
        return mfail(ctx, HVX_ERR_HIP, "hvx_mlp_create: %s", hipGetErrorString(e));
    }
    // uniform He initialisation (bound sqrt(6 / fan_in)), zero biases, from a
    // SplitMix64 stream of the seed
    std::vector<float> h(np, 0.0f);
    uint64_t state = seed;
    auto next = [&]() {
        uint64_t x = (state += 0x9E3779B97F4A7C15ull);
        x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
        x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
        x ^= x >> 31;
        return (double)(x >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int ofs, int count, int fan_in) {
        const double bound = std::sqrt(6.0 / fan_in);
        for (int i = 0; i < count; ++i) h[ofs + i] = (float)((2.0 * next() - 1.0) * bound);
    };
    fill(hvx::kMlpW1, kH * kIn, kIn);
    fill(hvx::kMlpW2, kH * kH, kH);
    fill(hvx::kMlpW3, kH * kH, kH);
    fill(hvx::kMlpW4, 3 * kH, kH);
    if ((e = hipMemcpy(M->P, h.data(), np * 4, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemset(M->m, 0, np * 4)) != hipSuccess || (e = hipMemset(M->v, 0, np * 4)) != hipSuccess) {
        hvx_mlp_destroy(M);
        return mfail(ctx, HVX_ERR_HIP, "hvx_mlp_create: %s", hipGetErrorString(e));
    }
    cast(M, nullptr);
    if ((e = hipDeviceSynchronize()) != hipSuccess) {
        hvx_mlp_destroy(M);
        return mfail(ctx, HVX_ERR_HIP, "hvx_mlp_create: %s", hipGetErrorString(e));
    }
    *out = M;
    return HVX_OK;
}

int hvx_mlp_destroy(hvx_mlp* M) {
    if (!M) return HVX_ERR_NULL;
    (void)hipDeviceSynchronize();
    for (void* p : M->batch_allocs) (void)hipFree(p);
    for (void* p : M->sep_allocs) (void)hipFree(p);
    for (void* p : M->allocs) (void)hipFree(p);
    if (M->enc) (void)hipFree(M->enc);
    if (M->encT) (void)hipFree(M->encT);
    if (M->cell_lo) (void)hipFree(M->cell_lo);
    delete M;
    return HVX_OK;
}

int hvx_mlp_get_params(hvx_mlp* M, float* host_params) {
    if (!M || !host_params) return HVX_ERR_NULL;
    const hipError_t e = hipMemcpy(host_params, M->P, hvx::kMlpParams * 4, hipMemcpyDeviceToHost);
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_get_params: %s", hipGetErrorString(e));
}

int hvx_mlp_set_params(hvx_mlp* M, const float* host_params) {
    if (!M || !host_params) return HVX_ERR_NULL;
    hipError_t e = hipMemcpy(M->P, host_params, hvx::kMlpParams * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        cast(M, nullptr);
        e = hipDeviceSynchronize();
    }
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_set_params: %s", hipGetErrorString(e));
}

int hvx_mlp_sample(hvx_mlp* M, const float* d_chain, uint32_t face, uint32_t mips, uint64_t seed, uint32_t n,
                   float* d_inputs, float* d_targets, void* stream) {
    if (!M || !d_chain || !d_inputs || !d_targets) return HVX_ERR_NULL;
    if (face == 0 || face > 16384 || mips == 0 || mips > hvx_mip_count(face) || n == 0)
        return mfail(M->ctx, HVX_ERR_INVALID_ARG, "hvx_mlp_sample: bad chain sizes or n");
    int st;
    if ((st = bind(M->ctx))) return st;
    hipLaunchKernelGGL(mlp_data_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                       reinterpret_cast<const float4*>(d_chain), face, mips, M->lod_max, seed, n,
                       reinterpret_cast<float4*>(d_inputs), reinterpret_cast<float4*>(d_targets));
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_sample: %s", hipGetErrorString(e));
}

int hvx_mlp_gradient(hvx_mlp* M, const float* d_inputs, const float* d_targets, uint32_t batch, float* d_grads,
                     float* d_loss, void* stream) {
    if (!M || !d_inputs || !d_targets || !d_grads) return HVX_ERR_NULL;
    if (batch == 0 || batch % 256 || batch > kMaxBatch)
        return mfail(M->ctx, HVX_ERR_INVALID_ARG, "batch must be a positive multiple of 256 (<= 2^20)");
    int st;
    if ((st = bind(M->ctx))) return st;
    hipError_t e = ensure_batch(M, batch);
    if (e != hipSuccess) return mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_gradient: %s", hipGetErrorString(e));
    const float4 *in = reinterpret_cast<const float4*>(d_inputs), *tg = reinterpret_cast<const float4*>(d_targets);
    if (M->ctx->mlp_separate) gradient_separate(M, in, Encoded{}, tg, batch, d_grads, d_loss, (hipStream_t)stream);
    else gradient_fused(M, in, nullptr, tg, batch, d_grads, nullptr, d_loss, (hipStream_t)stream);
    e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_gradient: %s", hipGetErrorString(e));
}

int hvx_mlp_train(hvx_mlp* M, const float* d_inputs, const float* d_targets, uint32_t n, uint32_t batch,
                  uint32_t steps, float lr, float* d_loss_curve, void* stream) {
    if (!M || !d_inputs || !d_targets) return HVX_ERR_NULL;
    if (batch == 0 || batch % 256 || batch > kMaxBatch || n < batch || !(lr > 0.0f))
        return mfail(M->ctx, HVX_ERR_INVALID_ARG, "hvx_mlp_train: batch a multiple of 256 <= n, lr > 0");
    int st;
    if ((st = bind(M->ctx))) return st;
    hipError_t e = ensure_batch(M, batch);
    if (e != hipSuccess) return mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_train: %s", hipGetErrorString(e));
    hipStream_t s = (hipStream_t)stream;
    const uint32_t per_epoch = n / batch;
    const float4* in = reinterpret_cast<const float4*>(d_inputs);
    const float4* tg = reinterpret_cast<const float4*>(d_targets);
    // Encode the call's samples once (256 B per sample, the separate launches'
    // transposed copy as much again) when they are revisited, instead of once
    // per step; without the memory, each step encodes its batch.
    const bool separate = M->ctx->mlp_separate != 0;
    const size_t npad = (size_t)per_epoch * batch;
    const bool revisit = steps > per_epoch;
    auto hold = [&](bf16*& p, size_t& cap) {
        if (cap >= npad) return true;
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
        if (hipMalloc(reinterpret_cast<void**>(&p), npad * kIn * sizeof(bf16)) == hipSuccess) {
            cap = npad;
            return true;
        }
        p = nullptr;
        (void)hipGetLastError();  // a failed allocation leaves the slower path, not an error
        return false;
    };
    const bool pre = revisit && hold(M->enc, M->enc_cap) && (!separate || hold(M->encT, M->encT_cap));
    if (pre) encode(in, (uint32_t)npad, (uint32_t)npad, M->lod_max, M->enc, separate ? M->encT : nullptr, s);
    if (!separate) M->transposes = false;
    for (uint32_t k = 0; k < steps; ++k) {
        const size_t off = (size_t)(k % per_epoch) * batch;
        float* loss = d_loss_curve ? d_loss_curve + k : nullptr;
        // cosine decay from lr to lr / 100 over the call
        const double ph = steps > 1 ? (double)k / (double)(steps - 1) : 0.0;
        const float lr_k = (float)(lr * (0.01 + 0.99 * 0.5 * (1.0 + std::cos(hvx::kMlpPi * ph))));
        ++M->steps_done;
        const float bc1 = (float)(1.0 - std::pow(0.9, (double)M->steps_done));
        const float bc2 = (float)(1.0 - std::pow(0.999, (double)M->steps_done));
        AdamArgs ad{M->P, M->m, M->v, lr_k, bc1, bc2, {M->W1, M->W2, M->W3, M->Ws, nullptr, nullptr}};
        if (separate) {
            ad.copies.W2T = M->W2T;
            ad.copies.W3T = M->W3T;
            const Encoded x = pre ? Encoded{M->enc + off * kIn, M->encT + off, (uint32_t)npad} : Encoded{};
            gradient_separate(M, in + off, x, tg + off, batch, M->G, loss, s);
            hipLaunchKernelGGL(adam_kernel, dim3((hvx::kMlpParams + 255) / 256), dim3(256), 0, s, ad, M->G,
                               (uint32_t)hvx::kMlpParams);
        } else {
            gradient_fused(M, in + off, pre ? M->enc + off * kIn : nullptr, tg + off, batch, nullptr, &ad, loss, s);
        }
    }
    e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_train: %s", hipGetErrorString(e));
}

// Workgroups of mlp_infer_kernel: each stages the weights (34 KB) once and
// loops over kInferStep samples, so a few per CU suffice.
static uint32_t infer_blocks(const hvx_mlp* M, uint32_t n) {
    const uint32_t cap = 4u * (uint32_t)std::max(M->ctx->num_cus, 1);
    return std::max(1u, std::min(cap, n / kInferStep + (n % kInferStep != 0)));
}

int hvx_mlp_eval(hvx_mlp* M, const float* d_inputs, uint32_t n, float* d_rgb, void* stream) {
    if (!M || !d_inputs || !d_rgb) return HVX_ERR_NULL;
    if (n == 0) return HVX_OK;
    int st;
    if ((st = bind(M->ctx))) return st;
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(infer_blocks(M, n)), dim3(256), 0, (hipStream_t)stream, hvx::mlp_view(M),
                       reinterpret_cast<const float4*>(d_inputs), n, d_rgb);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_eval: %s", hipGetErrorString(e));
}

int hvx_mlp_cell_errors(hvx_mlp* M, const float* d_chain, uint32_t face, uint32_t mips, uint32_t cell_face,
                        uint32_t lod_bins, float* d_err, void* stream) {
    if (!M || !d_chain || !d_err) return HVX_ERR_NULL;
    const uint32_t mask_face = cell_face;
    if (face == 0 || face > 16384 || mips == 0 || mips > hvx_mip_count(face) || mask_face == 0 || mask_face > 1024 ||
        lod_bins == 0 || lod_bins > 256)
        return mfail(M->ctx, HVX_ERR_INVALID_ARG, "hvx_mlp_cell_errors: sizes out of range");
    int st;
    if ((st = bind(M->ctx))) return st;
    const uint32_t cells = lod_bins * 6 * mask_face * mask_face;
    const size_t npts = (size_t)cells * kMaskPoints;
    if (npts > (1u << 28)) return mfail(M->ctx, HVX_ERR_INVALID_ARG, "hvx_mlp_cell_errors: too many cells");
    // set-up call: the point, prediction and raw-error buffers are allocated here
    float4* pts = nullptr;
    float* rgb = nullptr;
    float* raw = nullptr;
    hipError_t e;
    if ((e = hipMalloc(&pts, npts * sizeof(float4))) != hipSuccess ||
        (e = hipMalloc(&rgb, npts * 3 * sizeof(float))) != hipSuccess ||
        (e = hipMalloc(&raw, (size_t)cells * sizeof(float))) != hipSuccess) {
        if (pts) (void)hipFree(pts);
        if (rgb) (void)hipFree(rgb);
        return mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_cell_errors: %s", hipGetErrorString(e));
    }
    // the lower estimates travel with the network for hvx_cf_shade_learned
    if (M->lo_face * M->lo_face * 6 * M->lo_bins != cells || !M->cell_lo) {
        (void)hipDeviceSynchronize();  // a shading call may still read the old ones
        if (M->cell_lo) (void)hipFree(M->cell_lo);
        M->cell_lo = nullptr;
        M->lo_face = M->lo_bins = 0;
        if ((e = hipMalloc(&M->cell_lo, (size_t)cells * sizeof(float4))) != hipSuccess) {
            M->cell_lo = nullptr;
            (void)hipFree(pts);
            (void)hipFree(rgb);
            (void)hipFree(raw);
            return mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_cell_errors: %s", hipGetErrorString(e));
        }
    }
    M->lo_face = mask_face;
    M->lo_bins = lod_bins;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(mask_points_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, s, mask_face, lod_bins,
                       M->lod_max, pts);
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(infer_blocks(M, npts)), dim3(256), 0, s, hvx::mlp_view(M), pts,
                       (uint32_t)npts, rgb);
    hipLaunchKernelGGL(cell_error_kernel, dim3((cells + 255) / 256), dim3(256), 0, s, pts, rgb,
                       reinterpret_cast<const float4*>(d_chain), face, mips, cells, raw, M->cell_lo);
    hipLaunchKernelGGL(cell_margin_kernel, dim3((cells + 255) / 256), dim3(256), 0, s, raw, cells, d_err);
    e = hipStreamSynchronize(s);
    (void)hipFree(pts);
    (void)hipFree(rgb);
    (void)hipFree(raw);
    return e == hipSuccess ? HVX_OK : mfail(M->ctx, HVX_ERR_HIP, "hvx_mlp_cell_errors: %s", hipGetErrorString(e));
}

}  // extern "C"
