// contract.hip — the dense-contraction cube filter on FP16 MFMA
// (hvx_ibl_contract_* and hvx_ibl_filter_contract of include/hvx.h).
//
// The operator is defined in hvx_contract.h: per output mip a weight matrix
// W(o, k) of the canonical face, shared by all six faces. The geometry is
// also symmetric under the eight maps g of the square onto itself (u -> -u,
// v -> -v, u <-> v, acting on the output face's plane and, as rotations and
// reflections about its axis, on the whole sphere): W(g o, g k) = W(o, k). So
// a plan holds only the rows of one octant of the face (0 <= x <= y < So / 2)
// and a filter call multiplies each row into 6 faces x 8 maps x 3 channels:
//
//   C[rows, 144] = W[rows, K] * R[K, 144]    (FP16 MFMA, FP32 accumulate)
//
// where column (g, f, c) of R holds channel c of the input texel that output
// face f sees as g k: C's column (g, f, c) is the output at g o of face f. A
// row of weights (the matrices do not fit the caches) is thus read once for
// 48 output texels instead of 6; 144 columns are nine 16-wide MFMA column
// tiles without padding.
//
// K runs over units of eight texels along a row of the summed level (of the
// padded face plane for the near field). Rows are ordered along a Morton
// curve, so 128 consecutive ones (a block) lie close together on the face,
// and a block keeps only the units in which any of its rows has weight: half
// of the sphere lies behind a row, and a near window is a disk, not its
// bounding box.
//
// The weights are built on the GPU in FP64: the row normalisation sums are
// FP64 reductions, and each row is stored in FP16 scaled by a power of two
// that puts its largest weight just under 2^15. A filter call stages the
// input radiance as FP16 scaled per face by a power of two (largest value
// under 2^15).
//
// Measured (MI355X, whole calls, before: one row per output texel of the
// canonical face, 6 faces x 4 padded columns, windows as bounding boxes):
//   1024^2 -> 512^2 x 10, FP16           444 -> 128 us (weights 1606 -> 127 MB)
//   512^2 -> 256^2 x 9, split BF16       353 -> 100 us
//   24 probes 256^2 -> 128^2 x 8, FP16   855 -> 340 us
// The 128 us are 45 us of GEMM, 35 us of staging with the roughness-0 mip (100
// MB of level 0 read, 25 MB written), 23 us of the near rows' epilogue and 22 us
// of face maxima, plane maps and the other rows' epilogue.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "hvx_contract.h"
#include "hvx_device.h"
#include "hvx_internal.h"
#include "hvx_mfma.h"

namespace {

using hvx::ContractLevel;
using hvx::f32x4;
using hvx::f3;
using hvx::bf16x8;
using hvx::half8;
using hvx::normalize3;
using hvx::sample_cube;
using hvx::texel_dir;

enum Piece { PIECE_WHOLE = 0, PIECE_NEAR = 1, PIECE_FAR = 2 };

constexpr int kMaxJobs = 2 * hvx::kContractMaxMips;  // weight matrices (and staged inputs) of a plan
constexpr uint32_t kImages = 48;                     // output texels of a row: 8 maps x 6 faces
constexpr uint32_t kCols = 3 * kImages;              // columns of the contraction
constexpr uint32_t kBlockRows = 128;                 // rows that share a unit list
constexpr uint32_t kFaceMaxBlocks = 32;
constexpr uint32_t kMaxProbes = 4096;  // probes of one multi-probe call (grid dimension y)

// The probes of one filter call: input chains and output chains (one probe:
// the by-value pointers; several: device arrays of pointers), and where probe
// p's copy of the per-call scratch lives: a scratch pointer of the plan moves
// by delta + p * pstride bytes (0 and 0 for the plan's own scratch).
struct Probes {
    const float4* chain0;
    float4* out0;
    const float4* const* chains;
    float4* const* outs;
    uint64_t delta, pstride;
    uint32_t n;  // probes in the call
};
__device__ __forceinline__ const float4* probe_chain(const Probes& Q, uint32_t p) { return Q.chains ? Q.chains[p] : Q.chain0; }
__device__ __forceinline__ float4* probe_out(const Probes& Q, uint32_t p) { return Q.outs ? Q.outs[p] : Q.out0; }
template <class T> __device__ __forceinline__ T* scr(const Probes& Q, T* ptr, uint32_t p) {
    return reinterpret_cast<T*>(reinterpret_cast<uintptr_t>(ptr) + Q.delta + (uint64_t)p * Q.pstride);
}

// One weight matrix: the whole sum of a mip, or its near or far piece.
struct Job {
    int type, piece;
    double alpha2, t0, t1;
    uint32_t So;     // output face of the rows (far: the far grid's face)
    uint32_t Sf;     // near: the far map's face
    float4* map;     // far: the far map written; near: the far map added (scratch)
    float4* zmap;    // far: the far normaliser at the far grid, written at plan creation; near: read there
    size_t out_off;  // whole and near: the mip in the output chain, float4 units
};

// A row: canonical output texel (x, y) of its job's face, x <= y < So / 2.
struct Row {
    uint16_t x, y, job, block;
};

// A staged input: a level of the chain (pad 0: unit u holds texels 8u .. 8u+7
// of the 6 x S x S canonical level) or the face planes continued past the
// edges (pad 1: unit u holds texels 8 (u % Pw8) .. of row u / Pw8 of the
// Pw x Pw plane, Pw = S + 2B, whose texel (B, B) is the face's first).
struct Source {
    uint32_t pad, S, B, Pw8;
};

// 128 rows (fewer at a source's end) and the units they sum: nsteps K steps
// of four units, the weights as [step][row tile (nrt)][lane (64)][8], cut
// into K slices whose partial sums are added in slice order.
struct Block {
    uint32_t row0, nrows, nrt, nunits, nsteps;
    uint32_t unit0;  // first entry in the unit list (staged unit indices)
    uint32_t src, split, item0, nslices;
    uint64_t woff, w_lo;  // 16-byte units; w_lo: split BF16, from hi to lo
};

// K slice of a block: steps [s0, s0 + n); slot: its partial sums.
struct Item {
    uint32_t block, s0, n, slot;
};

// ---------------------------------------------------------- device helpers
// Map g of the square of n texels per edge onto itself: swap for g >= 4, then
// mirror x (bit 0) and y (bit 1).
__device__ __forceinline__ void image_of(uint32_t g, uint32_t n, uint32_t& x, uint32_t& y) {
    if (g & 4u) {
        const uint32_t t = x;
        x = y;
        y = t;
    }
    if (g & 1u) x = n - 1 - x;
    if (g & 2u) y = n - 1 - y;
}
// Whether map g writes its own image of row (x, y): a row on the diagonal
// (or on a 1 x 1 face) is its own mirror image and written once.
__device__ __forceinline__ bool image_written(uint32_t g, uint32_t n, uint32_t x, uint32_t y) {
    return n == 1 ? g == 0 : (g < 4 || x != y);
}

// Plane point (a, b) of face f at distance w from the centre (texel_dir's
// convention, as contract_face_point).
__host__ __device__ inline void face_ipoint(uint32_t f, int a, int b, int w, int p[3]) {
    switch (f) {
        case 0: p[0] = w; p[1] = -b; p[2] = -a; break;
        case 1: p[0] = -w; p[1] = -b; p[2] = a; break;
        case 2: p[0] = a; p[1] = w; p[2] = b; break;
        case 3: p[0] = a; p[1] = -w; p[2] = -b; break;
        case 4: p[0] = a; p[1] = -b; p[2] = w; break;
        default: p[0] = -a; p[1] = -b; p[2] = -w; break;
    }
}

// Texel (face, i, j) of a level of face s that output face f sees as g k, k the
// canonical input texel (x, y) of face t: exact integer arithmetic in doubled
// texel units (a texel centre of face t is the plane point (a, b), odd, at
// distance s; the canonical output face is (u, v, 1), so g acts on the first
// two components).
inline void dense_source(uint32_t f, uint32_t g, uint32_t t, int x, int y, int s, int out[3]) {
    int p[3], q[3];
    face_ipoint(t, 2 * x + 1 - s, 2 * y + 1 - s, s, p);
    if (g & 4u) std::swap(p[0], p[1]);
    if (g & 1u) p[0] = -p[0];
    if (g & 2u) p[1] = -p[1];
    face_ipoint(f, p[0], p[1], p[2], q);
    const int ax = std::abs(q[0]), ay = std::abs(q[1]), az = std::abs(q[2]);
    int nf, na, nb;
    if (ax >= ay && ax >= az) {
        nf = q[0] > 0 ? 0 : 1;
        na = q[0] > 0 ? -q[2] : q[2];
        nb = -q[1];
    } else if (ay >= az) {
        nf = q[1] > 0 ? 2 : 3;
        na = q[0];
        nb = q[1] > 0 ? q[2] : -q[2];
    } else {
        nf = q[2] > 0 ? 4 : 5;
        na = q[2] > 0 ? q[0] : -q[0];
        nb = -q[1];
    }
    out[0] = nf;
    out[1] = (na + s - 1) / 2;
    out[2] = (nb + s - 1) / 2;
}

// dense_source as data, entry [t][6 g + f]: the face (3 bits), then whether x
// and y swap (8), and then whether i (16) and j (32) run backwards.
std::vector<uint8_t> source_table() {
    std::vector<uint8_t> tab(6 * kImages);
    for (uint32_t t = 0; t < 6; ++t)
        for (uint32_t g = 0; g < 8; ++g)
            for (uint32_t f = 0; f < 6; ++f) {
                int o[3], a[3];
                dense_source(f, g, t, 0, 0, 2, o);
                dense_source(f, g, t, 1, 0, 2, a);
                tab[t * kImages + 6 * g + f] =
                    (uint8_t)(o[0] | (a[1] == o[1] ? 8 : 0) | (o[1] ? 16 : 0) | (o[2] ? 32 : 0));
            }
    return tab;
}

__device__ __forceinline__ void local_dir(double u, double v, double d[3]) {
    const double r = 1.0 / sqrt(1.0 + u * u + v * v);
    d[0] = u * r;
    d[1] = v * r;
    d[2] = r;
}

// Direction and solid angle of texel q of unit u of a source.
__device__ __forceinline__ void unit_texel(const Source& G, uint32_t unit, uint32_t q, double l[3], double* dw) {
    if (G.pad) {
        const uint32_t py = unit / G.Pw8, px = (unit - py * G.Pw8) * 8 + q;
        const double u = hvx::contract_coord((int)px - (int)G.B, G.S), v = hvx::contract_coord((int)py - (int)G.B, G.S);
        local_dir(u, v, l);
        *dw = hvx::contract_dw(u, v, G.S);
        return;
    }
    const uint32_t k = unit * 8 + q, S2 = G.S * G.S, t = k / S2, rem = k - t * S2, y = rem / G.S, x = rem - y * G.S;
    const double u = hvx::contract_coord((int)x, G.S), v = hvx::contract_coord((int)y, G.S);
    double p[3];
    hvx::contract_face_point((int)t, u, v, p);
    const double r = 1.0 / sqrt(1.0 + u * u + v * v);
    l[0] = p[0] * r;
    l[1] = p[1] * r;
    l[2] = p[2] * r;
    *dw = hvx::contract_dw(u, v, G.S);
}

__device__ __forceinline__ void row_dir(const Row& R, uint32_t So, double n[3]) {
    local_dir(hvx::contract_coord((int)R.x, So), hvx::contract_coord((int)R.y, So), n);
}

__device__ __forceinline__ double row_weight(const Job& J, const double n[3], const double l[3], double dw) {
    const double c = (n[0] * l[0] + n[1] * l[1]) + n[2] * l[2];
    double w = hvx::contract_weight(J.type, J.alpha2, c);
    if (w == 0.0) return 0.0;
    w *= dw;
    if (J.piece == PIECE_NEAR) w *= hvx::contract_phi(J.t0, J.t1, c);
    else if (J.piece == PIECE_FAR) w *= 1.0 - hvx::contract_phi(J.t0, J.t1, c);
    return w;
}

// Power-of-two exponent s with w_max * 2^s in (2^14, 2^15].
__host__ __device__ __forceinline__ int row_exponent(double wmax) {
    if (!(wmax > 0.0)) return 0;
    int e;
    (void)frexp(wmax, &e);  // wmax = m 2^e, m in [0.5, 1)
    return 15 - e;
}

// Deterministic block sum and max (256 threads) in double.
__device__ void block_sum_max(double s, double m, double* sh_s, double* sh_m, double* out_s, double* out_m) {
    const uint32_t t = threadIdx.x;
    sh_s[t] = s;
    sh_m[t] = m;
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
        if (t < h) {
            sh_s[t] = sh_s[t] + sh_s[t + h];
            sh_m[t] = sh_m[t] < sh_m[t + h] ? sh_m[t + h] : sh_m[t];
        }
        __syncthreads();
    }
    if (t == 0) {
        *out_s = sh_s[0];
        *out_m = sh_m[0];
    }
}

// ------------------------------------------------------------ plan: weights
// flags[b][u] = 1 when any row of block block0 + b may have weight in unit u:
// the texel lies in front of the row and, for the near piece, inside the
// window (each bound relaxed by more than the cosine's rounding).
__global__ __launch_bounds__(256) void unit_flag_kernel(Source G, const Job* __restrict__ jobs,
                                                        const Row* __restrict__ rows, const Block* __restrict__ blocks,
                                                        uint32_t block0, uint32_t raw, uint8_t* __restrict__ flags) {
    __shared__ double sd[kBlockRows][3], sc[kBlockRows];
    const Block B = blocks[block0 + blockIdx.y];
    for (uint32_t r = threadIdx.x; r < B.nrows; r += 256) {
        const Row R = rows[B.row0 + r];
        const Job& J = jobs[R.job];
        row_dir(R, J.So, sd[r]);
        sc[r] = (J.piece == PIECE_NEAR ? cos(J.t1) : 0.0) - 1e-9;
    }
    __syncthreads();
    const uint32_t u = blockIdx.x * 256 + threadIdx.x;
    if (u >= raw) return;
    bool any = false;
    for (uint32_t q = 0; q < 8 && !any; ++q) {
        double l[3], dw;
        unit_texel(G, u, q, l, &dw);
        for (uint32_t r = 0; r < B.nrows && !any; ++r)
            any = (sd[r][0] * l[0] + sd[r][1] * l[1]) + sd[r][2] * l[2] > sc[r];
    }
    flags[(size_t)blockIdx.y * raw + u] = any ? 1 : 0;
}

// Sum and largest weight of every row of a source (one workgroup per row).
// units: the source's staged units; ulist: the blocks' lists of them.
__global__ __launch_bounds__(256) void row_sum_kernel(Source G, const Job* __restrict__ jobs,
                                                      const Row* __restrict__ rows, const Block* __restrict__ blocks,
                                                      const uint32_t* __restrict__ ulist,
                                                      const uint32_t* __restrict__ units, uint32_t row0,
                                                      double* __restrict__ Z, double* __restrict__ wmax) {
    __shared__ double sh_s[256], sh_m[256];
    const uint32_t row = row0 + blockIdx.x;
    const Row R = rows[row];
    const Job J = jobs[R.job];
    const Block B = blocks[R.block];
    double n[3];
    row_dir(R, J.So, n);
    double s = 0.0, m = 0.0;
    for (uint32_t k = threadIdx.x; k < B.nunits * 8; k += 256) {
        double l[3], dw;
        unit_texel(G, units[ulist[B.unit0 + k / 8]], k & 7, l, &dw);
        const double w = row_weight(J, n, l, dw);
        s += w;
        m = m < w ? w : m;
    }
    block_sum_max(s, m, sh_s, sh_m, &Z[row], &wmax[row]);
}

// The MFMA A operands of a source's blocks (grid y: block; padding rows and
// units hold zeros). SPLIT: the scaled weight v as BF16 hi = bf16(v) and, at
// w_lo, lo = bf16(v - hi) (hi + lo carries ~16 significant bits).
template <bool SPLIT>
__global__ __launch_bounds__(256) void weight_fill_kernel(Source G, const Job* __restrict__ jobs,
                                                          const Row* __restrict__ rows,
                                                          const Block* __restrict__ blocks, uint32_t block0,
                                                          const uint32_t* __restrict__ ulist,
                                                          const uint32_t* __restrict__ units,
                                                          const double* __restrict__ wmax, half8* __restrict__ W) {
    const Block B = blocks[block0 + blockIdx.y];
    const uint32_t total = B.nsteps * B.nrt * 64;
    for (uint32_t id = blockIdx.x * 256 + threadIdx.x; id < total; id += gridDim.x * 256) {
        const uint32_t lane = id & 63, rt = (id >> 6) % B.nrt, step = (id >> 6) / B.nrt;
        const uint32_t r = rt * 16 + (lane & 15), u = step * 4 + (lane >> 4);
        double v[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (r < B.nrows && u < B.nunits) {
            const Row R = rows[B.row0 + r];
            const Job& J = jobs[R.job];
            double n[3];
            row_dir(R, J.So, n);
            const double sc = ldexp(1.0, row_exponent(wmax[B.row0 + r]));
            const uint32_t unit = units[ulist[B.unit0 + u]];
            for (uint32_t q = 0; q < 8; ++q) {
                double l[3], dw;
                unit_texel(G, unit, q, l, &dw);
                v[q] = row_weight(J, n, l, dw) * sc;
            }
        }
        if constexpr (SPLIT) {
            bf16x8 hi, lo;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                hi[q] = (__bf16)(float)v[q];
                lo[q] = (__bf16)(float)(v[q] - (double)(float)hi[q]);
            }
            reinterpret_cast<bf16x8*>(W)[B.woff + id] = hi;
            reinterpret_cast<bf16x8*>(W)[B.woff + id + B.w_lo] = lo;
        } else {
            half8 out;
#pragma unroll
            for (int q = 0; q < 8; ++q) out[q] = (_Float16)(float)v[q];
            W[B.woff + id] = out;
        }
    }
}

// Far rows: the normaliser at every image of the row (the same on all faces).
__global__ __launch_bounds__(256) void far_norm_kernel(const Job* __restrict__ jobs, const Row* __restrict__ rows,
                                                       uint32_t row0, uint32_t n, const double* __restrict__ Z) {
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= n * kImages) return;
    const uint32_t r = row0 + id / kImages, gf = id % kImages;
    const Row R = rows[r];
    const Job& J = jobs[R.job];
    if (J.piece != PIECE_FAR) return;
    uint32_t x = R.x, y = R.y;
    if (!image_written(gf / 6, J.So, x, y)) return;
    image_of(gf / 6, J.So, x, y);
    J.zmap[((gf % 6) * J.So + y) * J.So + x] = make_float4((float)Z[r], 0.0f, 0.0f, 0.0f);
}

// rowscale = 2^-s / Z (whole rows), 2^-s (far rows), 2^-s / (Z + far
// normaliser interpolated at the row's direction) (near rows, with the
// reciprocal of that sum in invZ).
__global__ __launch_bounds__(256) void row_scale_kernel(const Job* __restrict__ jobs, const Row* __restrict__ rows,
                                                        uint32_t n, const double* __restrict__ Z,
                                                        const double* __restrict__ wmax, float* __restrict__ rowscale,
                                                        float* __restrict__ invZ) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    const Row R = rows[r];
    const Job& J = jobs[R.job];
    double z = J.piece == PIECE_FAR ? 1.0 : Z[r];
    if (J.piece == PIECE_NEAR) {
        const f3 zf = sample_cube(J.zmap, (int)J.Sf, texel_dir(0, (int)R.x, (int)R.y, (int)J.So));
        z += (double)zf.x;
    }
    rowscale[r] = (float)(ldexp(1.0, -row_exponent(wmax[r])) / z);
    invZ[r] = (float)(1.0 / z);
}

// ------------------------------------------------------ per-call staging
// A filter call is at most six launches: face maxima, staging (with the
// roughness-0 mip), the maps of the staged planes, the GEMM over every weight
// matrix, the epilogue of the whole and far rows, that of the near rows.

// partial[f][b]: largest RGB magnitude of block b's share of face f
__global__ __launch_bounds__(256) void facemax_kernel(Probes Q, size_t level_off, uint32_t S, float* partial) {
    __shared__ float sh[256];
    const uint32_t f = blockIdx.y, S2 = S * S, pr = blockIdx.z;
    const float4* level = probe_chain(Q, pr) + level_off;
    partial = scr(Q, partial, pr);
    float m = 0.0f;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < S2; i += gridDim.x * 256) {
        const float4 v = level[(size_t)f * S2 + i];
        const float a = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fabsf(v.z));
        m = a > m ? a : m;  // NaN never replaces m
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[f * gridDim.x + blockIdx.x] = sh[0];
}

// Power-of-two exponent that brings m under 2^15 (0 for 0 and non-finite m).
__device__ __forceinline__ int scale_exponent(float m) {
    int e = 0;
    if (m > 0.0f && m <= 3.0e38f) {
        int ex;
        (void)frexpf(m, &ex);
        e = ex - 15;
    }
    return e;
}

// A workgroup's exponents from the face maxima (nb <= 32 partials a face):
// se[f] for the padded plane of face f (bounded by face f and its four
// neighbours), se[6] over all faces. Each staging workgroup forms them itself:
// a launch of their own costs more.
__device__ void block_exponents(const float* __restrict__ partial, uint32_t nb, int* se) {
    __shared__ float fm[6];
    const uint32_t t = threadIdx.x, f = t >> 5, b = t & 31;
    float m = f < 6 && b < nb ? partial[f * nb + b] : 0.0f;
    for (int d = 16; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    if (f < 6 && b == 0) fm[f] = m;
    __syncthreads();
    if (t < 7) {
        float v = 0.0f;
        for (uint32_t g = 0; g < 6; ++g)
            if (t == 6 || g != (t ^ 1u)) v = fmaxf(v, fm[g]);
        se[t] = scale_exponent(v);
    }
    __syncthreads();
}

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));

enum StageKind { STAGE_DENSE = 0, STAGE_PLANE = 1, STAGE_DELTA = 2 };
struct StageItem {
    int kind, split;
    uint32_t S, B, Pw;
    uint32_t n;              // units, plane texels or output texels (one face)
    uint32_t block_begin;    // first workgroup of the item
    size_t level_off;        // float4 offset of the level in the input chain (STAGE_DELTA: in the output chain)
    const uint32_t* list;    // dense: the staged units; planes: the texels needed (index in the Pw x Pw plane)
    half8* dst;              // dense: R[unit][144][8]
    uint64_t lo_off;         // split: offset of the lo parts (16-byte units; planes: in the texel's own record)
};
struct StageTable {
    StageItem it[kMaxJobs + 2];  // and the roughness-0 mip, and stage_rest's first
    uint32_t n, blocks;
    const uint32_t* map;  // source_table
};

// Writes the staged operand R[unit][col][8] of a few consecutive units (eight;
// four split-BF16): column 3 (6 g + f) + c, element q holds channel c of what
// face f sees as g (texel q of the unit). A wave takes one image (g, f) of all
// of the units' texels per pass (split: two), so that its loads cover a small
// patch of one face - consecutive units are stacked in y - and the values go
// through LDS to be stored unit by unit, each 2304 contiguous bytes. With a
// thread per (unit, image) instead, loading eight texels of its own, every
// load touched 64 cache lines: 24 probes 256^2 -> 128^2 x 8 took 220 us to
// stage and 80 us to map.
// fetch(unit, q, image): the texel; V::hi(c), V::lo(c) its staged channels.
constexpr uint32_t kColsPad = kCols + 1;  // LDS units: the eight rows of a pass fall into different banks
constexpr uint32_t kTileUnits = 8;
template <bool SPLIT>
constexpr uint32_t tile_units() { return SPLIT ? kTileUnits / 2 : kTileUnits; }
template <bool SPLIT, class V, class Fetch>
__device__ __forceinline__ void stage_tile(half8* sT, uint32_t u0, uint32_t nu, half8* __restrict__ R, uint64_t lo_off,
                                           Fetch fetch) {
    constexpr uint32_t UT = tile_units<SPLIT>(), kWide = 64 / (8 * UT), kPasses = kImages / (4 * kWide);
    const uint32_t t = threadIdx.x, lane = t & 63, q = lane & 7, u = (lane >> 3) % UT, sub = lane / (8 * UT);
    const uint32_t m = min(UT, nu - u0);
    const uint32_t image0 = (t >> 6) * kPasses * kWide + sub;
    V v[kPasses];
#pragma unroll
    for (uint32_t k = 0; k < kPasses; ++k) v[k] = fetch(min(u, m - 1), q, image0 + k * kWide);
#pragma unroll
    for (uint32_t k = 0; k < kPasses; ++k) {
        const size_t e = (u * kColsPad + 3 * (image0 + k * kWide)) * 8 + q;
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            if constexpr (SPLIT) {
                reinterpret_cast<__bf16*>(sT)[e + 8 * c] = v[k].hi(c);
                reinterpret_cast<__bf16*>(sT + UT * kColsPad)[e + 8 * c] = v[k].lo(c);
            } else {
                reinterpret_cast<_Float16*>(sT)[e + 8 * c] = v[k].hi(c);
            }
        }
    }
    __syncthreads();
    for (uint32_t e = t; e < m * kCols; e += 256) {
        const uint32_t at = e / kCols * kColsPad + e % kCols;
        R[(size_t)u0 * kCols + e] = sT[at];
        if constexpr (SPLIT) R[lo_off + (size_t)u0 * kCols + e] = sT[UT * kColsPad + at];
    }
}

// Texel of a level, scaled, as the staged formats.
template <bool SPLIT>
struct LevelTexel {
    float4 t;
    float s;
    __device__ float at(uint32_t c) const { return (c == 0 ? t.x : c == 1 ? t.y : t.z) * s; }
    __device__ auto hi(uint32_t c) const {
        if constexpr (SPLIT) return (__bf16)at(c);
        else return (_Float16)at(c);
    }
    __device__ __bf16 lo(uint32_t c) const { return (__bf16)(at(c) - (float)(__bf16)at(c)); }
};
// Texel of a staged plane.
template <bool SPLIT>
struct PlaneTexel {
    std::conditional_t<SPLIT, bf16x8, half4v> t;
    __device__ auto hi(uint32_t c) const { return t[c]; }
    __device__ __bf16 lo(uint32_t c) const { return (__bf16)t[4 + c]; }
};

// A level's units: face f sees canonical texel (x, y) of face t as g k where
// source_table says.
template <bool SPLIT>
__device__ __forceinline__ void stage_dense(const float4* __restrict__ level, const StageItem& I, float s,
                                            half8* __restrict__ R, uint32_t blk, half8* sT, const uint8_t* sMap) {
    constexpr uint32_t UT = tile_units<SPLIT>();
    const uint32_t u0 = blk * UT, m = min(UT, I.n - u0), lane = threadIdx.x & 63, S = I.S;
    const uint32_t k = I.list[u0 + min((lane >> 3) % UT, m - 1)] * 8 + (lane & 7);
    const uint32_t S2 = S * S, t = k / S2, rem = k - t * S2, y = rem / S, x = rem - y * S;
    stage_tile<SPLIT, LevelTexel<SPLIT>>(sT, u0, I.n, R, I.lo_off, [&](uint32_t, uint32_t, uint32_t image) {
        const uint32_t b = sMap[t * kImages + image];
        uint32_t i = b & 8u ? y : x, j = b & 8u ? x : y;
        i = b & 16u ? S - 1 - i : i;
        j = b & 32u ? S - 1 - j : j;
        return LevelTexel<SPLIT>{level[((b & 7u) * S + j) * S + i], s};
    });
}

// T[f][py][px]: the scaled texel of face f's plane continued past its edges:
// inside the face the texel itself, outside the bilinear seamless sample of
// the level at the plane point's direction; four FP16 values (RGB, 0), or
// four BF16 hi then four lo. One thread per needed (texel, face).
template <bool SPLIT>
__device__ __forceinline__ void stage_plane(const float4* __restrict__ level, const StageItem& I, const int* se,
                                            half8* __restrict__ dst, uint32_t id) {
    const uint32_t f = id / I.n, p = I.list[id - f * I.n], py = p / I.Pw, px = p - py * I.Pw;
    const int x = (int)px - (int)I.B, y = (int)py - (int)I.B;
    f3 t;
    if (x >= 0 && y >= 0 && x < (int)I.S && y < (int)I.S) {
        const float4 v = level[((size_t)f * I.S + y) * I.S + x];
        t = f3{v.x, v.y, v.z};
    } else {
        // plane points in doubled texel units: exact in FP32, and the sample
        // needs no unit direction
        int q[3];
        face_ipoint(f, 2 * x + 1 - (int)I.S, 2 * y + 1 - (int)I.S, (int)I.S, q);
        const f3 d = {(float)q[0], (float)q[1], (float)q[2]};
        // taps first, so that their loads run together also at the face edges
        const hvx::CubeTaps c = hvx::cube_taps((int)I.S, d);
        const float4 w[4] = {level[c.idx[0]], level[c.idx[1]], level[c.idx[2]], level[c.idx[3]]};
        t = hvx::cube_combine(level, (int)I.S, d, c, w);
    }
    const float s = ldexpf(1.0f, -se[f]), v[3] = {t.x * s, t.y * s, t.z * s};
    const size_t at = (size_t)f * I.Pw * I.Pw + p;
    if constexpr (SPLIT) {
        bf16x8 h;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            h[c] = (__bf16)v[c];
            h[4 + c] = (__bf16)(v[c] - (float)h[c]);
        }
        h[3] = h[7] = (__bf16)0.0f;
        reinterpret_cast<bf16x8*>(dst)[at] = h;
    } else {
        reinterpret_cast<half4v*>(dst)[at] = half4v{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)0.0f};
    }
}

// sc[f] = 2^e_f of face f's plane, sc[6] = 2^e of the whole levels: what the
// epilogues multiply by. delta0 (nullable): the chain the roughness-0 mip
// samples instead of the probe's.
__global__ __launch_bounds__(256) void stage_kernel(Probes Q, StageTable T, const float* partial, uint32_t nb,
                                                    float* sc, const float4* delta0, uint32_t S0) {
    __shared__ half8 sT[kTileUnits * kColsPad];
    __shared__ uint32_t sMap[6 * kImages / 4];
    const uint32_t pr = blockIdx.y, blk = blockIdx.x;
    uint32_t j = 0;
    while (j + 1 < T.n && blk >= T.it[j + 1].block_begin) ++j;  // uniform over the workgroup
    const StageItem& I = T.it[j];
    const uint32_t id = (blk - I.block_begin) * 256 + threadIdx.x;
    if (I.kind == STAGE_DELTA) {
        // roughness 0: the bilinear seamless sample of level 0 at the texel direction
        const uint32_t So = I.S, So2 = So * So;
        if (id >= 6 * So2) return;
        const uint32_t f = id / So2, o = id - f * So2, Y = o / So, X = o - Y * So;
        const f3 c = sample_cube(delta0 ? delta0 : probe_chain(Q, pr), (int)S0, texel_dir((int)f, (int)X, (int)Y, (int)So));
        probe_out(Q, pr)[I.level_off + id] = make_float4(c.x, c.y, c.z, 1.0f);
        return;
    }
    __shared__ int se[7];
    if (threadIdx.x < 6 * kImages / 4) sMap[threadIdx.x] = T.map[threadIdx.x];
    block_exponents(scr(Q, partial, pr), nb, se);
    if (blk == 0 && threadIdx.x < 7) scr(Q, sc, pr)[threadIdx.x] = ldexpf(1.0f, se[threadIdx.x]);
    const float4* level = probe_chain(Q, pr) + I.level_off;
    half8* dst = scr(Q, I.dst, pr);
    if (I.kind == STAGE_DENSE) {
        const float s = ldexpf(1.0f, -se[6]);
        const uint8_t* map = reinterpret_cast<const uint8_t*>(sMap);
        if (I.split) stage_dense<true>(level, I, s, dst, blk - I.block_begin, sT, map);
        else stage_dense<false>(level, I, s, dst, blk - I.block_begin, sT, map);
    } else {
        if (id >= I.n * 6) return;
        if (I.split) stage_plane<true>(level, I, se, dst, id);
        else stage_plane<false>(level, I, se, dst, id);
    }
}

struct MapItem {
    uint32_t Pw, n, block_begin;
    const uint32_t* list;  // the staged units
    const half8* T;        // stage_plane's texels
    half8* dst;            // R[unit][144][8]
    uint64_t lo_off;       // 0: FP16
};
struct MapTable {
    MapItem it[kMaxJobs];
    uint32_t n, blocks;
};

// The staged operand of the padded planes: texel (px, py) of the plane maps to
// g (px, py) of face f's plane.
template <bool SPLIT>
__device__ __forceinline__ void map_plane(const MapItem& I, const half8* T, half8* R, uint32_t blk, half8* sT) {
    constexpr uint32_t UT = tile_units<SPLIT>();
    using V = PlaneTexel<SPLIT>;
    const V* P = reinterpret_cast<const V*>(T);
    const uint32_t u0 = blk * UT, m = min(UT, I.n - u0), lane = threadIdx.x & 63, Pw = I.Pw;
    const uint32_t unit = I.list[u0 + min((lane >> 3) % UT, m - 1)], py = unit / (Pw / 8);
    const uint32_t px = (unit - py * (Pw / 8)) * 8 + (lane & 7);
    stage_tile<SPLIT, V>(sT, u0, I.n, R, I.lo_off, [&](uint32_t, uint32_t, uint32_t image) {
        const uint32_t g = image / 6, f = image - 6 * g;
        uint32_t x = px, y = py;
        image_of(g, Pw, x, y);
        return P[(f * Pw + y) * Pw + x];
    });
}

__global__ __launch_bounds__(256) void plane_map_kernel(Probes Q, MapTable M) {
    __shared__ half8 sT[kTileUnits * kColsPad];
    const uint32_t pr = blockIdx.y;
    uint32_t j = 0;
    while (j + 1 < M.n && blockIdx.x >= M.it[j + 1].block_begin) ++j;  // uniform over the workgroup
    const MapItem& I = M.it[j];
    const half8* T = scr(Q, I.T, pr);
    half8* R = scr(Q, I.dst, pr);
    if (I.lo_off) map_plane<true>(I, T, R, blockIdx.x - I.block_begin, sT);
    else map_plane<false>(I, T, R, blockIdx.x - I.block_begin, sT);
}

// ------------------------------------------------------------- MFMA GEMM
struct GemmArgs {
    const half8* W;
    const Block* blocks;
    const Item* items;
    const uint32_t* ulist;
    float* part;  // [slot][kBlockRows][kCols]
    uint32_t nitems;
    const half8* R[kMaxJobs];
    uint64_t r_lo[kMaxJobs];
    // gemm_direct: ulist as the levels count their units, stage_kernel's
    // scales, source_table, the levels
    const uint32_t* raw_ulist;
    const float* sc;
    const uint32_t* map;
    uint64_t level_off[kMaxJobs];
    uint32_t log2_S[kMaxJobs];
};
static_assert(sizeof(StageTable) < 4000 && sizeof(MapTable) < 4000 && sizeof(GemmArgs) < 4000,
              "launch tables must fit the kernel argument space");

constexpr uint32_t kGroup = 4;        // K steps staged per barrier (half as many split-BF16 ones)
constexpr uint32_t kDGroup = 2;       // K steps per barrier in gemm_direct: there 4 hold up short slices
constexpr uint32_t kMinSlice = 8;     // K steps of an item, at least
constexpr uint32_t kGoodSlice = 32;   // and at least in plans that fill the chip
constexpr uint32_t kMaxSlice = 64;    // K steps of an item, at most
constexpr uint32_t kXcds = 8;
constexpr uint32_t kNt = kCols / 16;  // MFMA column tiles

// Bound by what reaches the CUs: at 512^2 x 10 127 MB of weights and 125 MB of
// staged units (each read by the blocks whose windows hold it) in 45 us, 190 MB
// of it past the L2, while its MFMAs (36 GFLOP with the padding of rows) need 14
// us and its LDS reads 7 us.
// One workgroup per (item, probe): four waves of two 16-row tiles each over
// the item's K steps, all 144 columns, so a wave's 18 accumulators reuse each
// weight fragment nine times and each B fragment twice. The B operand of a
// step (four units of 144 half8, contiguous) is shared by the waves and
// staged in LDS, kGroup steps per barrier, double buffered, a group ahead;
// weights go straight to registers, a group ahead.
template <bool SPLIT>
__device__ __forceinline__ void gemm_item(const GemmArgs& A, const Block& B, const Item& I, const half8* Rp,
                                          half8 (*sB)[kGroup * 4 * kCols], const uint32_t* sU, f32x4 (&acc)[2][kNt]) {
    constexpr uint32_t G = SPLIT ? kGroup / 2 : kGroup;  // steps per group
    constexpr uint32_t kStepB = 4 * kCols * (SPLIT ? 2 : 1);
    constexpr uint32_t kPer = G * kStepB / 256;
    constexpr int kWs = SPLIT ? 4 : 2;
    static_assert(G * kStepB % 256 == 0, "whole passes of the workgroup");
    using GH = const __attribute__((address_space(1))) half8*;
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6, i = lane & 15, g = lane >> 4;
    const uint32_t nrt = B.nrt, rt0 = 2 * wave, n = I.n;
    const bool live = rt0 < nrt, has1 = rt0 + 1 < nrt;  // uniform per wave
    const GH w0 = (GH)(A.W + B.woff + ((size_t)I.s0 * nrt + (live ? rt0 : 0)) * 64 + lane);
    const GH w1 = has1 ? w0 + 64 : w0;
    const size_t wstep = (size_t)nrt * 64, w_lo = B.w_lo, r_lo = A.r_lo[B.src];
    const GH R = (GH)Rp;
    // steps past the slice's last repeat it (loaded, not used)
    auto w_load = [&](uint32_t s, half8 (&x)[G][kWs]) {
#pragma unroll
        for (uint32_t k = 0; k < G; ++k) {
            const size_t o = (size_t)(s + k < n ? s + k : n - 1) * wstep;
            x[k][0] = w0[o];
            x[k][1] = w1[o];
            if constexpr (SPLIT) {
                x[k][2] = w0[o + w_lo];
                x[k][3] = w1[o + w_lo];
            }
        }
    };
    // sU holds the slice's units, padded to whole groups
    auto b_load = [&](uint32_t s, half8 (&v)[kPer]) {
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            const uint32_t e = t + 256u * k, st = e / kStepB, r = e % kStepB, lo = r / (4 * kCols), rr = r % (4 * kCols);
            v[k] = R[(size_t)sU[(s + st) * 4 + rr / kCols] * kCols + rr % kCols + (lo ? r_lo : 0)];
        }
    };
    auto b_store = [&](uint32_t buf, const half8 (&v)[kPer]) {
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) sB[buf][t + 256u * k] = v[k];
    };
    half8 nb[kPer], xw[G][kWs], xn[G][kWs];
    b_load(0, nb);
    w_load(0, xw);
    b_store(0, nb);
    __syncthreads();
    const uint32_t groups = (n + G - 1) / G;
    for (uint32_t gi = 0; gi < groups; ++gi) {
        const uint32_t s = gi * G, sn = gi + 1 < groups ? s + G : s;
        w_load(sn, xn);
        b_load(sn, nb);
        __asm__ volatile("" ::: "memory");
        const half8* sb = sB[gi & 1];
#pragma unroll
        for (uint32_t k = 0; k < G; ++k) {
            if (live && s + k < n) {
#pragma unroll
                for (uint32_t nt = 0; nt < kNt; ++nt) {
                    const half8* bk = sb + k * kStepB + g * kCols + nt * 16 + i;
                    if constexpr (SPLIT) {
                        const bf16x8 b = __builtin_bit_cast(bf16x8, bk[0]), c = __builtin_bit_cast(bf16x8, bk[4 * kCols]);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const bf16x8 x = __builtin_bit_cast(bf16x8, xw[k][h]);
                            const bf16x8 y = __builtin_bit_cast(bf16x8, xw[k][2 + h]);
                            // hi*hi + hi*lo + lo*hi (lo*lo is below the FP32 accumulation's resolution)
                            acc[h][nt] = hvx::mfma16x16x32(x, b, acc[h][nt]);
                            acc[h][nt] = hvx::mfma16x16x32(x, c, acc[h][nt]);
                            acc[h][nt] = hvx::mfma16x16x32(y, b, acc[h][nt]);
                        }
                    } else {
                        const half8 b = bk[0];
                        acc[0][nt] = hvx::mfma16x16x32(xw[k][0], b, acc[0][nt]);
                        acc[1][nt] = hvx::mfma16x16x32(xw[k][1], b, acc[1][nt]);
                    }
                }
            }
        }
        b_store((gi & 1) ^ 1, nb);  // its readers passed the previous barrier
#pragma unroll
        for (uint32_t k = 0; k < G; ++k)
#pragma unroll
            for (int u = 0; u < kWs; ++u) xw[k][u] = xn[k][u];
        __syncthreads();
    }
}

// The same products (and sums, to the bit) with the B operand staged from the
// level by the workgroup that multiplies it, for levels that one block of rows
// sums: their staged units would be written to memory (2,304 bytes each) to be
// read once. With many probes of small outputs that was most of the call:
// 1,024 probes 32^2 -> 16^2 x 5 take 423 us so, 825 staged. A wave loads one image
// of eight units' texels at a time, as stage_tile does (a thread per (unit, image)
// instead, loads of 64 lines each: 591). Two K steps per barrier: four hold up the
// short slices of small outputs (1,024 probes 16^2 -> 8^2 x 4 128 us against 117;
// 256 probes 64^2 -> 32^2 x 6, whose slices are long, 587 against 647). level: the
// probe's; sU: the slice's units as the level counts them; sc: 1 / the levels' scale.
__device__ __forceinline__ void gemm_direct(const GemmArgs& A, const Block& B, const Item& I,
                                            const float4* __restrict__ level, uint32_t ls, float sc,
                                            half8 (*sB)[kDGroup * 4 * kColsPad], const uint32_t* sU,
                                            const uint32_t* sMap, f32x4 (&acc)[2][kNt]) {
    constexpr uint32_t kWaveImages = kImages / 4;
    static_assert(kDGroup % 2 == 0 && kWaveImages % 4 == 0, "whole eights of units, whole words of the map");
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6, i = lane & 15, g = lane >> 4;
    const uint32_t nrt = B.nrt, rt0 = 2 * wave, n = I.n, S = 1u << ls;
    const bool live = rt0 < nrt, has1 = rt0 + 1 < nrt;  // uniform per wave
    const half8* w0 = A.W + B.woff + ((size_t)I.s0 * nrt + (live ? rt0 : 0)) * 64 + lane;
    const half8* w1 = has1 ? w0 + 64 : w0;
    const size_t wstep = (size_t)nrt * 64;
    auto stage = [&](uint32_t s, uint32_t buf) {
#pragma unroll
        for (uint32_t h = 0; h < kDGroup / 2; ++h) {
            const uint32_t u = 8 * h + lane / 8, k8 = sU[s * 4 + u] * 8 + lane % 8;
            const uint32_t x = k8 & (S - 1), y = k8 >> ls & (S - 1), f = k8 >> (2 * ls);
            uint32_t m[kWaveImages / 4];
            float4 v[kWaveImages];
#pragma unroll
            for (uint32_t k = 0; k < kWaveImages / 4; ++k) m[k] = sMap[(f * kImages + wave * kWaveImages) / 4 + k];
#pragma unroll
            for (uint32_t k = 0; k < kWaveImages; ++k) {
                const uint32_t b = m[k / 4] >> (8 * (k % 4));
                uint32_t a = b & 8u ? y : x, c = b & 8u ? x : y;
                a = b & 16u ? S - 1 - a : a;
                c = b & 32u ? S - 1 - c : c;
                v[k] = level[((b & 7u) * S + c) * S + a];
            }
#pragma unroll
            for (uint32_t k = 0; k < kWaveImages; ++k) {
                const LevelTexel<false> T{v[k], sc};
                _Float16* o = reinterpret_cast<_Float16*>(&sB[buf][u * kColsPad + 3 * (wave * kWaveImages + k)]) + lane % 8;
                o[0] = T.hi(0);
                o[8] = T.hi(1);
                o[16] = T.hi(2);
            }
        }
    };
    stage(0, 0);
    __syncthreads();
    const uint32_t groups = (n + kDGroup - 1) / kDGroup;
    for (uint32_t gi = 0; gi < groups; ++gi) {
        const uint32_t s = gi * kDGroup;
        half8 x[kDGroup][2];
#pragma unroll
        for (uint32_t k = 0; k < kDGroup; ++k) {
            const size_t o = (size_t)(s + k < n ? s + k : n - 1) * wstep;
            x[k][0] = w0[o];
            x[k][1] = w1[o];
        }
        if (gi + 1 < groups) stage(s + kDGroup, (gi & 1) ^ 1);  // its readers passed the previous barrier
        const half8* sb = sB[gi & 1];
#pragma unroll
        for (uint32_t k = 0; k < kDGroup; ++k)
            if (live && s + k < n) {
#pragma unroll
                for (uint32_t nt = 0; nt < kNt; ++nt) {
                    const half8 b = sb[(k * 4 + g) * kColsPad + nt * 16 + i];
                    acc[0][nt] = hvx::mfma16x16x32(x[k][0], b, acc[0][nt]);
                    acc[1][nt] = hvx::mfma16x16x32(x[k][1], b, acc[1][nt]);
                }
            }
        __syncthreads();
    }
}

template <bool DIRECT>
__global__ __launch_bounds__(256, 2) void contract_gemm_kernel(Probes Q, GemmArgs A) {
    __shared__ half8 sB[2][DIRECT ? kDGroup * 4 * kColsPad : kGroup * 4 * kCols];
    __shared__ uint32_t sU[(kMaxSlice + kGroup) * 4], sMap[DIRECT ? 6 * kImages / 4 : 1];
    // hardware workgroup b runs on XCD b % 8: each XCD takes one run of the
    // items, whose neighbours share staged units, and of an item's probes,
    // which share its weights
    const uint32_t run = (A.nitems * Q.n + kXcds - 1) / kXcds;
    const uint32_t id = blockIdx.x % kXcds * run + blockIdx.x / kXcds;
    if (id >= A.nitems * Q.n) return;  // uniform; padding of the last run
    const uint32_t item = id / Q.n, pr = id - item * Q.n, t = threadIdx.x;
    const Item I = A.items[item];
    const Block B = A.blocks[I.block];
    const uint32_t left = B.nunits - I.s0 * 4;  // units from the slice's first on (its last step may be short of four)
    const uint32_t* ulist = DIRECT ? A.raw_ulist : A.ulist;
    for (uint32_t k = t; k < (kMaxSlice + kGroup) * 4; k += 256)
        sU[k] = ulist[B.unit0 + I.s0 * 4 + min(k, min(I.n * 4, left) - 1)];
    if (DIRECT && t < 6 * kImages / 4) sMap[t] = A.map[t];
    __syncthreads();
    f32x4 acc[2][kNt];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (uint32_t nt = 0; nt < kNt; ++nt) acc[h][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (DIRECT) {
        gemm_direct(A, B, I, probe_chain(Q, pr) + A.level_off[B.src], A.log2_S[B.src], 1.0f / scr(Q, A.sc, pr)[6], sB,
                    sU, sMap, acc);
    } else {
        const half8* R = scr(Q, A.R[B.src], pr);
        if (B.split) gemm_item<true>(A, B, I, R, sB, sU, acc);
        else gemm_item<false>(A, B, I, R, sB, sU, acc);
    }
    const uint32_t lane = t & 63, i = lane & 15, g = lane >> 4, rt0 = 2 * (t >> 6);
    float* p = scr(Q, A.part, pr) + (size_t)I.slot * kBlockRows * kCols;
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
        if (rt0 + h >= B.nrt) break;
#pragma unroll
        for (uint32_t nt = 0; nt < kNt; ++nt)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                p[((rt0 + h) * 16 + 4 * g + r) * kCols + nt * 16 + i] = acc[h][nt][r];
    }
}

// The far map (face Sf) at the centre of output texel (x, y) of face f: the
// texel's plane coordinates are exact in FP32 (sizes are powers of two), so
// inside the face the four taps need no direction.
__device__ __forceinline__ f3 far_sample(const float4* __restrict__ map, uint32_t Sf, uint32_t f, uint32_t x,
                                         uint32_t y, uint32_t So) {
    const float r = (float)Sf / (float)So;
    const float u = ((float)x + 0.5f) * r - 0.5f, v = ((float)y + 0.5f) * r - 0.5f;
    const float fu = floorf(u), fv = floorf(v), a = u - fu, b = v - fv;
    const int i = (int)fu, j = (int)fv;
    if (i < 0 || j < 0 || i + 1 >= (int)Sf || j + 1 >= (int)Sf)
        return sample_cube(map, (int)Sf, texel_dir((int)f, (int)x, (int)y, (int)So));
    const float4* p = map + ((size_t)f * Sf + j) * Sf + i;
    const float4 q00 = p[0], q10 = p[1], q01 = p[Sf], q11 = p[Sf + 1];
    const float w00 = (1.0f - a) * (1.0f - b), w10 = a * (1.0f - b), w01 = (1.0f - a) * b, w11 = a * b;
    return {((w00 * q00.x + w10 * q10.x) + w01 * q01.x) + w11 * q11.x,
            ((w00 * q00.y + w10 * q10.y) + w01 * q01.y) + w11 * q11.y,
            ((w00 * q00.z + w10 * q10.z) + w01 * q01.z) + w11 * q11.z};
}

// Output texel (g o, f) of each row from the slices' sums, in slice order. NEAR
// false: whole rows into the chain, far rows into their map (not normalised);
// true: near rows plus the far field interpolated at the texel, over Z.
template <bool NEAR>
__global__ __launch_bounds__(256) void epilogue_kernel(Probes Q, const Job* __restrict__ jobs,
                                                       const Row* __restrict__ rows, const Block* __restrict__ blocks,
                                                       const float* part, const float* __restrict__ rowscale,
                                                       const float* __restrict__ invZ, const float* sc, uint32_t row0,
                                                       uint32_t n) {
    const uint32_t id = blockIdx.x * 256 + threadIdx.x, pr = blockIdx.y;
    if (id >= n * kImages) return;
    const uint32_t r = row0 + id / kImages, gf = id % kImages, g = gf / 6, f = gf - 6 * g;
    const Row R = rows[r];
    const Job& J = jobs[R.job];
    uint32_t x = R.x, y = R.y;
    if (!image_written(g, J.So, x, y)) return;
    image_of(g, J.So, x, y);
    const Block& B = blocks[R.block];
    const uint32_t ns = B.nslices;
    const float* p = scr(Q, part, pr) + ((size_t)B.item0 * kBlockRows + (r - B.row0)) * kCols + 3 * gf;
    float v[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (uint32_t s = 0; s < ns; ++s, p += kBlockRows * kCols) {
        v[0] += p[0];
        v[1] += p[1];
        v[2] += p[2];
    }
    const size_t o = ((size_t)f * J.So + y) * J.So + x;
    const float* q = scr(Q, sc, pr);
    if constexpr (NEAR) {
        const float k = rowscale[r], sf = q[f], z = invZ[r];
        const f3 F = far_sample(scr(Q, J.map, pr), J.Sf, f, x, y, J.So);
        probe_out(Q, pr)[J.out_off + o] =
            make_float4(v[0] * k * sf + F.x * z, v[1] * k * sf + F.y * z, v[2] * k * sf + F.z * z, 1.0f);
    } else {
        const float k = rowscale[r] * q[6];
        const bool far = J.piece == PIECE_FAR;
        float4* out = far ? scr(Q, J.map, pr) : probe_out(Q, pr) + J.out_off;
        out[o] = make_float4(v[0] * k, v[1] * k, v[2] * k, far ? 0.0f : 1.0f);
    }
}

// --------------------------------------------------- bright-texel split
// (hvx_contract.h): threshold from a histogram of the largest channel's float
// pattern, clamped level 0, the hot texels in texel order, and their exact
// level-0 sum added to every non-delta output texel.
struct HotArgs {
    const float4* level0;  // the caller's level 0
    float4* clamped;       // level 0 of the clamped chain
    uint32_t S, K;
    uint32_t* hist;        // kHotBins counts, zero between calls
    uint32_t* cnt;         // [0] hot texels found, [1] hot texels listed, [2] blocks
    float* T;
    uint32_t* idx;         // kHotMax texel indices; after the sort, the member range of each block
    float4* list;          // per listed texel: (direction, 0), (solid angle * excess, 0)
    float4* groups;        // per 4x4 block: (mean direction, radius), (summed excess, member range)
};

__device__ __forceinline__ float hot_largest(float4 t) { return fmaxf(fmaxf(t.x, t.y), t.z); }

__global__ __launch_bounds__(256) void hot_hist_kernel(HotArgs H) {
    __shared__ uint32_t sh[hvx::kHotBins];
    for (uint32_t b = threadIdx.x; b < hvx::kHotBins; b += 256) sh[b] = 0u;
    __syncthreads();
    const size_t n = 6ull * H.S * H.S, stride = (size_t)gridDim.x * 256;
    const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x;
    // four texels in flight per thread; the bins are then counted one by one
    for (size_t i = i0; i < n; i += 4 * stride) {
        float m4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t k = i + q * stride;
            m4[q] = k < n ? hot_largest(H.level0[k]) : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float m = m4[q];
            const uint32_t bin = m > 0.0f ? hvx::contract_hot_bin(__float_as_uint(m)) : 0xffffffffu;
            // neighbouring texels mostly share a bin: one LDS atomic per wave then
            const uint32_t b0 = __builtin_amdgcn_readfirstlane(bin);
            if (__all(bin == b0)) {
                const unsigned long long act = __ballot(1);
                if (b0 != 0xffffffffu && (threadIdx.x & 63) == (uint32_t)__ffsll(act) - 1)
                    atomicAdd(&sh[b0], (uint32_t)__popcll(act));
            } else if (bin != 0xffffffffu) {
                atomicAdd(&sh[bin], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < hvx::kHotBins; b += 256)
        if (sh[b]) atomicAdd(&H.hist[b], sh[b]);
}

// One workgroup of 1024: c(b) = texels in bins >= b (a scan over the bins
// from the top, two per thread), T from the number of bins with c(b) > K;
// clears the histogram and the counters for the next call.
__global__ __launch_bounds__(1024) void hot_select_kernel(HotArgs H) {
    __shared__ uint32_t s_wave[16];
    const uint32_t t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const uint32_t b_hi = hvx::kHotBins - 1 - 2 * t, b_lo = b_hi - 1;  // thread t: bins 2047-2t, 2046-2t
    const uint32_t h_hi = H.hist[b_hi], h_lo = H.hist[b_lo];
    H.hist[b_hi] = 0u;
    H.hist[b_lo] = 0u;
    uint32_t inc = h_hi + h_lo;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(inc, d, 64);
        if ((int)lane >= d) inc += u;
    }
    if (lane == 63) s_wave[wv] = inc;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wv; ++w) before += s_wave[w];
    const uint32_t c_lo = before + inc, c_hi = c_lo - h_lo;  // c(b_lo), c(b_hi)
    const int over = __syncthreads_count(c_hi > H.K) + __syncthreads_count(c_lo > H.K);
    if (t == 0) {
        H.T[0] = __uint_as_float(hvx::contract_hot_threshold_bits((uint32_t)over));
        H.cnt[0] = 0u;
        H.cnt[1] = 0u;
        H.cnt[2] = 0u;
    }
}

__global__ __launch_bounds__(256) void hot_compact_kernel(HotArgs H) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= 6ull * H.S * H.S) return;
    const float T = H.T[0];
    float4 v = H.level0[i];
    const float m = hot_largest(v);
    if (m > 0.0f && m >= T) {
        const uint32_t k = atomicAdd(&H.cnt[0], 1u);
        if (k < H.K) H.idx[k] = (uint32_t)i;
        v.x = v.x > T ? T : v.x;
        v.y = v.y > T ? T : v.y;
        v.z = v.z > T ? T : v.z;
    }
    H.clamped[i] = v;
}

// One workgroup of 1024: sorts the found texels by (face, 4x4 block, texel
// in block) so that the sum order is fixed and each 4x4 block's texels are
// contiguous, then writes each texel's direction and solid angle times
// excess (FP64 geometry, as the oracle's level-0 sum) and the member range
// of every block.
__device__ __forceinline__ uint32_t hot_key(uint32_t i, uint32_t S) {
    const uint32_t S2 = S * S, g = i / S2, r = i - g * S2, y = r / S, x = r - y * S, Q = S >> 2;
    return (((g * Q + (y >> 2)) * Q + (x >> 2)) << 4) | ((y & 3u) << 2) | (x & 3u);
}
__device__ __forceinline__ uint32_t hot_index(uint32_t key, uint32_t S) {
    const uint32_t Q = S >> 2, blk = key >> 4, bx = blk % Q, by = (blk / Q) % Q, g = blk / (Q * Q);
    const uint32_t y = (by << 2) | ((key >> 2) & 3u), x = (bx << 2) | (key & 3u);
    return (g * S + y) * S + x;
}

__global__ __launch_bounds__(1024) void hot_list_kernel(HotArgs H) {
    __shared__ uint32_t s[hvx::kHotMax];
    __shared__ uint32_t s_wave[16];
    const uint32_t n = min(H.cnt[0], H.K), t = threadIdx.x, lane = t & 63, wv = t >> 6;
    for (uint32_t j = t; j < hvx::kHotMax; j += 1024) s[j] = j < n ? hot_key(H.idx[j], H.S) : 0xffffffffu;  // S >= 4
    __syncthreads();
    for (uint32_t size = 2; size <= hvx::kHotMax; size <<= 1)
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t j = t; j < hvx::kHotMax / 2; j += 1024) {
                const uint32_t lo = 2 * j - (j & (stride - 1)), hi = lo + stride;
                const bool up = (lo & size) == 0;
                const uint32_t a = s[lo], b = s[hi];
                if ((a > b) == up) {
                    s[lo] = b;
                    s[hi] = a;
                }
            }
            __syncthreads();
        }
    const float T = H.T[0];
    const uint32_t S2 = H.S * H.S;
    for (uint32_t k = t; k < n; k += 1024) {
        const uint32_t i = hot_index(s[k], H.S), g = i / S2, r = i - g * S2, y = r / H.S, x = r - y * H.S;
        const double u = hvx::contract_coord((int)x, H.S), v = hvx::contract_coord((int)y, H.S);
        double p[3];
        hvx::contract_face_point((int)g, u, v, p);
        const double rl = 1.0 / sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]), dw = hvx::contract_dw(u, v, H.S);
        const float4 c = H.level0[i];
        const float ex = c.x > T ? c.x - T : 0.0f, ey = c.y > T ? c.y - T : 0.0f, ez = c.z > T ? c.z - T : 0.0f;
        H.list[2 * k] = make_float4((float)(p[0] * rl), (float)(p[1] * rl), (float)(p[2] * rl), 0.0f);
        H.list[2 * k + 1] = make_float4((float)(dw * ex), (float)(dw * ey), (float)(dw * ez), 0.0f);
    }
    // block starts: thread t owns entries 4t .. 4t+3; exclusive scan of the counts
    uint32_t starts = 0;
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t k = 4 * t + q;
        starts += (k < n && (k == 0 || (s[k] >> 4) != (s[k - 1] >> 4))) ? 1u : 0u;
    }
    uint32_t inc = starts;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(inc, d, 64);
        if ((int)lane >= d) inc += u;
    }
    if (lane == 63) s_wave[wv] = inc;
    __syncthreads();
    uint32_t gi = inc - starts;
    for (uint32_t w = 0; w < wv; ++w) gi += s_wave[w];
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t k = 4 * t + q;
        if (!(k < n && (k == 0 || (s[k] >> 4) != (s[k - 1] >> 4)))) continue;
        uint32_t e = k + 1;
        while (e < n && (s[e] >> 4) == (s[k] >> 4)) ++e;
        H.idx[gi++] = k | ((e - k) << 16);  // the found indices are consumed: idx now holds block ranges
    }
    if (t == 1023) {
        H.cnt[1] = n;
        H.cnt[2] = gi;
    }
}

// One thread per block of hot texels: excess-weighted mean direction, the
// angular radius of the members around it, the summed excess.
__global__ __launch_bounds__(256) void hot_group_kernel(HotArgs H) {
    const uint32_t gi = blockIdx.x * 256 + threadIdx.x;
    if (gi >= H.cnt[2]) return;
    const uint32_t pk = H.idx[gi], k = pk & 0xffffu, e = k + (pk >> 16);
    double E[3] = {0.0, 0.0, 0.0}, m[3] = {0.0, 0.0, 0.0};
    for (uint32_t j = k; j < e; ++j) {
        const float4 L = H.list[2 * j], X = H.list[2 * j + 1];
        const double wgt = (double)X.x + (double)X.y + (double)X.z;
        E[0] += X.x;
        E[1] += X.y;
        E[2] += X.z;
        m[0] += wgt * L.x;
        m[1] += wgt * L.y;
        m[2] += wgt * L.z;
    }
    double ml = sqrt(m[0] * m[0] + m[1] * m[1] + m[2] * m[2]);
    if (!(ml > 0.0)) {  // no excess in the block: any member direction
        const float4 L = H.list[2 * k];
        m[0] = L.x;
        m[1] = L.y;
        m[2] = L.z;
        ml = 1.0;
    }
    double rad = 0.0;
    for (uint32_t j = k; j < e; ++j) {
        const float4 L = H.list[2 * j];
        const double c = (m[0] * L.x + m[1] * L.y + m[2] * L.z) / ml;
        rad = fmax(rad, acos(fmin(1.0, fmax(-1.0, c))));
    }
    H.groups[2 * gi] = make_float4((float)(m[0] / ml), (float)(m[1] / ml), (float)(m[2] / ml),
                                   (float)(rad * (1.0 + 1e-6) + 1e-7));
    H.groups[2 * gi + 1] = make_float4((float)E[0], (float)E[1], (float)E[2], __uint_as_float(pk));
}

struct HotMip {
    uint32_t So, first;  // output face; first output of the mip in the launch (a multiple of 64: one mip per workgroup)
    float alpha2, h1;    // GGX a^2 and (1 - a^2) / 2
    float scale;         // a^2 / pi / (weight integral); diffuse: 1 / pi
    uint32_t _pad;
    size_t out_off;      // the mip in the output chain, float4 units
};
struct HotAdd {
    HotMip m[hvx::kContractMaxMips];
    uint32_t nm, blocks;
    const float4* list;
    const float4* groups;
    const uint32_t* cnt;
    float4* out;
    float theta_near;  // blocks farther than this (radians) from every output direction may enter as one entry
};

// w'(n . l) E: w' = c / d^2 (GGX, d = a^2 + (1 - c)(1 - a^2)/2 = N.H^2 (a^2 - 1)
// + 1) or c (cosine), 0 for c <= 0; 1 - c is formed as |n - l|^2 / 2, which
// keeps its relative accuracy for nearby directions.
template <bool DIFFUSE>
__device__ __forceinline__ void hot_term(const f3& n, const float4 L, const float4 E, float a2, float h1, float& ax,
                                         float& ay, float& az) {
    const float dx = n.x - L.x, dy = n.y - L.y, dz = n.z - L.z;
    const float q = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));  // 2 (1 - c)
    const float c = __builtin_fmaf(q, -0.5f, 1.0f);
    float w;
    if constexpr (DIFFUSE) {
        w = fmaxf(c, 0.0f);
    } else {
        const float d = __builtin_fmaf(q, h1, a2);  // h1 holds (1 - a^2) / 4 here
        w = fmaxf(c, 0.0f) * __builtin_amdgcn_rcpf(d * d);
    }
    ax = __builtin_fmaf(w, E.x, ax);
    ay = __builtin_fmaf(w, E.y, ay);
    az = __builtin_fmaf(w, E.z, az);
}

// out(o) += scale * sum over the hot texels of w'(n_o . l_k) E_k. A workgroup
// holds 64 output texels of one mip. A 4x4 block of hot texels whose cone
// lies more than theta_near outside the workgroup's cone of output
// directions, and wholly in front of every one of them (c > 0: clear of the
// kink of w at c = 0), enters as one entry at its excess-weighted mean
// direction (the terms linear in the offsets cancel; the rest is of relative
// order 10 (block extent / distance)^2); a block wholly behind every output
// direction adds exactly 0 and is skipped; every other block is summed texel
// by texel.
template <bool DIFFUSE>
__global__ __launch_bounds__(256) void hot_add_kernel(HotAdd A) {
    constexpr uint32_t kG = 32, kE = kG * 16;  // blocks per round; entries they can expand to
    __shared__ float4 se[2 * kE];
    __shared__ uint32_t s_ne;
    __shared__ float s_acc[3][3][64];
    // 64 output texels per workgroup (an 8 x 8 tile of one face when the face
    // has at least 8 texels), one per lane; the four waves split the entries
    const uint32_t b0 = blockIdx.x * 64, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    uint32_t mi = 0;
    while (mi + 1 < A.nm && b0 >= A.m[mi + 1].first) ++mi;  // uniform over the workgroup
    const HotMip M = A.m[mi];
    const uint32_t So2 = M.So * M.So, loc0 = b0 + lane - M.first;
    const bool live = loc0 < 6 * So2;
    uint32_t f, X, Y;
    {
        const uint32_t l = live ? loc0 : 0u;
        f = l / So2;
        const uint32_t w = l - f * So2;
        if (M.So >= 8) {  // So^2 is a multiple of 64
            const uint32_t te = M.So >> 3, tile = w >> 6, e = w & 63u;
            X = (tile % te) * 8 + (e & 7u);
            Y = (tile / te) * 8 + (e >> 3);
        } else {
            Y = w / M.So;
            X = w - Y * M.So;
        }
    }
    const uint32_t loc = (f * M.So + Y) * M.So + X;
    const f3 n = texel_dir((int)f, (int)X, (int)Y, (int)M.So);
    // the workgroup's cone (every wave holds the same 64 directions): mean
    // direction of the live texels, smallest cosine to it
    float cx = live ? n.x : 0.0f, cy = live ? n.y : 0.0f, cz = live ? n.z : 0.0f;
    for (int d = 32; d > 0; d >>= 1) {
        cx += __shfl_xor(cx, d, 64);
        cy += __shfl_xor(cy, d, 64);
        cz += __shfl_xor(cz, d, 64);
    }
    const float cl = sqrtf(cx * cx + cy * cy + cz * cz);
    const bool cone = cl > 1e-3f;  // else: directions all round the sphere, no cone
    if (cone) {
        cx /= cl;
        cy /= cl;
        cz /= cl;
    }
    float cmin = live ? n.x * cx + n.y * cy + n.z * cz : 1.0f;
    for (int d = 32; d > 0; d >>= 1) cmin = fminf(cmin, __shfl_xor(cmin, d, 64));
    // radius of the output cone, rounded up (a few 1e-6 rad)
    const float rad_o = acosf(fmaxf(-1.0f, fminf(1.0f, cmin))) * 1.0001f + 1e-5f;
    const float kHalfPi = 1.57079633f;
    const float h1 = DIFFUSE ? 0.0f : 0.5f * M.h1;
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    const uint32_t ng = A.cnt[2];
    for (uint32_t base = 0; base < ng; base += kG) {
        const uint32_t cg = min(kG, ng - base);
        __syncthreads();  // the previous round's entries are consumed
        if (wv == 0) {
            // the first wave sorts this round's blocks into skipped (0 entries),
            // aggregated (1) and summed texel by texel (its members), and
            // expands them into the entry list at their prefix offsets
            uint32_t mode = 2u, cnt = 0u, pk = 0u;
            float4 G0 = make_float4(0.f, 0.f, 0.f, 0.f), G1 = G0;
            if (lane < cg) {
                G0 = A.groups[2 * (base + lane)];
                G1 = A.groups[2 * (base + lane) + 1];
                pk = __float_as_uint(G1.w);
                const float ang = acosf(fmaxf(-1.0f, fminf(1.0f, G0.x * cx + G0.y * cy + G0.z * cz)));
                const float lo = ang * 0.9999f - 1e-5f - rad_o - G0.w, hi = ang * 1.0001f + 1e-5f + rad_o + G0.w;
                mode = !cone ? 0u : lo > kHalfPi + 1e-4f ? 2u : (lo > A.theta_near && hi < kHalfPi - 1e-4f) ? 1u : 0u;
                cnt = mode == 2u ? 0u : mode == 1u ? 1u : (pk >> 16);
            }
            uint32_t inc = cnt;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t u = __shfl_up(inc, d, 64);
                if ((int)lane >= d) inc += u;
            }
            const uint32_t off = inc - cnt;
            if (lane == 63) s_ne = inc;
            if (mode == 1u) {
                se[2 * off] = G0;
                se[2 * off + 1] = G1;
            } else if (mode == 0u) {
                const uint32_t k0 = pk & 0xffffu;
                for (uint32_t j = 0; j < cnt; ++j) {
                    se[2 * (off + j)] = A.list[2 * (k0 + j)];
                    se[2 * (off + j) + 1] = A.list[2 * (k0 + j) + 1];
                }
            }
        }
        __syncthreads();
        const uint32_t ne = s_ne;
        for (uint32_t j = wv; j < ne; j += 4) hot_term<DIFFUSE>(n, se[2 * j], se[2 * j + 1], M.alpha2, h1, ax, ay, az);
    }
    // the waves' partial sums, added in wave order
    if (wv > 0) {
        s_acc[0][wv - 1][lane] = ax;
        s_acc[1][wv - 1][lane] = ay;
        s_acc[2][wv - 1][lane] = az;
    }
    __syncthreads();
    if (wv != 0 || !live) return;
    ax = ((ax + s_acc[0][0][lane]) + s_acc[0][1][lane]) + s_acc[0][2][lane];
    ay = ((ay + s_acc[1][0][lane]) + s_acc[1][1][lane]) + s_acc[1][2][lane];
    az = ((az + s_acc[2][0][lane]) + s_acc[2][1][lane]) + s_acc[2][2][lane];
    float4& r = A.out[M.out_off + loc];
    r.x = __builtin_fmaf(ax, M.scale, r.x);
    r.y = __builtin_fmaf(ay, M.scale, r.y);
    r.z = __builtin_fmaf(az, M.scale, r.z);
}


// -------------------------------------------------------------- host side
uint32_t ilog2(uint32_t v) {
    uint32_t l = 0;
    while ((1u << (l + 1)) <= v) ++l;
    return l;
}

// Rows of an So x So face: the octant 0 <= x <= y < So / 2 (the one texel of a
// 1 x 1 face) along a Morton curve, so that runs of rows are compact patches.
std::vector<Row> octant_rows(uint32_t So, uint16_t job) {
    const uint32_t h = std::max(So / 2, 1u);
    std::vector<Row> rows;
    rows.reserve((size_t)h * (h + 1) / 2);
    for (uint64_t m = 0; m < (uint64_t)h * h; ++m) {  // h is a power of two
        uint32_t x = 0, y = 0;
        for (uint32_t b = 0; (1u << b) < h; ++b) {
            x |= (uint32_t)((m >> (2 * b)) & 1) << b;
            y |= (uint32_t)((m >> (2 * b + 1)) & 1) << b;
        }
        if (x <= y) rows.push_back(Row{(uint16_t)x, (uint16_t)y, job, 0});
    }
    return rows;
}

// Texels by which the angular caps of radius t1 around the output texels of a
// face reach past the near level's face on its plane, and four more, rounded
// up to whole units. By symmetry the octant's rows reach the furthest, and of
// those the ones along the face's edge (y = 0).
uint32_t plane_border(uint32_t So, uint32_t Si, double t1) {
    const double ct = std::cos(t1), st = std::sin(t1);
    double reach = 1.0;
    for (uint32_t x = 0; x < std::max(So / 2, 1u); ++x) {
        const double u = hvx::contract_coord((int)x, So), v = hvx::contract_coord(0, So);
        const double r = 1.0 / std::sqrt(1.0 + u * u + v * v), n[3] = {u * r, v * r, r};
        // e1, e2: any two directions orthogonal to n and to each other
        const double a[3] = {std::fabs(n[0]) < 0.9 ? 1.0 : 0.0, std::fabs(n[0]) < 0.9 ? 0.0 : 1.0, 0.0};
        double e1[3] = {a[1] * n[2] - a[2] * n[1], a[2] * n[0] - a[0] * n[2], a[0] * n[1] - a[1] * n[0]};
        const double l = std::sqrt(e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2]);
        for (double& e : e1) e /= l;
        const double e2[3] = {n[1] * e1[2] - n[2] * e1[1], n[2] * e1[0] - n[0] * e1[2], n[0] * e1[1] - n[1] * e1[0]};
        for (int j = 0; j < 256; ++j) {
            const double w = 2.0 * hvx::kContractPi * j / 256.0, ca = std::cos(w), sa = std::sin(w);
            double p[3];
            for (int q = 0; q < 3; ++q) p[q] = ct * n[q] + st * (ca * e1[q] + sa * e2[q]);
            reach = std::max({reach, std::fabs(p[0] / p[2]), std::fabs(p[1] / p[2])});
        }
    }
    const uint32_t B = (uint32_t)std::ceil((reach - 1.0) * 0.5 * Si) + 4;
    return (B + 7) / 8 * 8;
}

// Reserves `bytes` (256-byte aligned) at the end of a scratch layout.
size_t scratch_take(size_t* total, size_t bytes) {
    const size_t at = (*total + 255) & ~(size_t)255;
    *total = at + bytes;
    return at;
}

// A source while the plan is built: its geometry, the jobs that sum it, and
// the staged units (those any row has weight in).
struct SourcePlan {
    Source G{};
    uint32_t level = 0;  // of the input chain
    bool split = false;
    uint32_t raw = 0;    // units of the whole level or plane
    uint32_t row0 = 0, rows = 0, block0 = 0, nblocks = 0;
    std::vector<uint32_t> units, need;  // need (planes): the texels the staged units' images read
    size_t units_off = 0, need_off = 0;  // in the plan's tables
    size_t r_off = 0, t_off = 0;  // staged operand in the per-call scratch, plane texels in its last part
};

struct MipPlan {
    ContractLevel L{};
    uint64_t weight_bytes = 0;
};

}  // namespace

struct hvx_contract_plan {
    hvx_ctx* ctx = nullptr;
    int type = 0, precision = 0;
    uint32_t S = 0, So = 0, mips = 0;
    std::vector<MipPlan> mp;
    // Per-call scratch, carved from one block of scratch_bytes: far maps,
    // staged levels and planes, face maxima, scales, K-slice partial sums.
    // Multi-probe calls of up to mcap probes use mcopies further copies of the
    // block (mscratch), that many probes at a time.
    char* scratch = nullptr;
    size_t scratch_bytes = 0;
    char* mscratch = nullptr;
    uint32_t mcap = 0, mcopies = 0;
    float* fmax = nullptr;  // per-face partial maxima [6][kFaceMaxBlocks]
    float* sc = nullptr;
    uint32_t min_level = 0;  // deepest input chain level read
    uint32_t scale_level = ~0u;  // finest staged level: its maxima bound every staged value
    StageTable stage{}, stage_rest{};  // stage_rest: for gemm_direct
    MapTable maps{};
    GemmArgs gemm{};
    uint32_t items = 0, direct_units = 0;  // direct_units: of the levels, if gemm_direct can take them
    uint32_t dense_rows = 0, near_rows = 0;  // rows [0, dense_rows) whole and far, then the near ones
    const Job* d_jobs = nullptr;
    const Row* d_rows = nullptr;
    const float *rowscale = nullptr, *invZ = nullptr;
    // bright-texel split (hvx_ibl_contract_plan_set_hot): off while hot_k == 0
    uint32_t hot_k = 0;
    float* hot_chain = nullptr;  // the clamped chain, min_level + 1 levels
    uint32_t* hot_hist = nullptr;
    uint32_t* hot_cnt = nullptr;
    float* hot_T = nullptr;
    uint32_t* hot_idx = nullptr;
    float4* hot_list = nullptr;
    float4* hot_groups = nullptr;
    std::vector<void*> allocs;

    template <class T> hipError_t alloc(T** p, size_t count) {
        void* q = nullptr;
        const hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
        if (e == hipSuccess) allocs.push_back(q);
        *p = static_cast<T*>(q);
        return e;
    }
};

namespace {

int pfail(hvx_ctx* ctx, int st, const char* fmt, ...) __attribute__((format(printf, 3, 4)));
int pfail(hvx_ctx* ctx, int st, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (ctx) ctx->last_error = buf;
    return st;
}

// Memory used while a plan is built, released with it.
struct Scratch {
    void* p = nullptr;
    ~Scratch() {
        if (p) (void)hipFree(p);
    }
    template <class T> hipError_t get(T** q, size_t n) {
        const hipError_t e = hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T));
        *q = static_cast<T*>(p);
        return e;
    }
};

// A plan's tables, put together on the host and uploaded as one allocation:
// a call on a new plan then misses in few pages.
struct Tables {
    std::vector<char> bytes;
    template <class T> size_t add(const T* v, size_t n) {
        const size_t at = (bytes.size() + 255) / 256 * 256;
        bytes.resize(at + n * sizeof(T));
        if (v && n) std::memcpy(bytes.data() + at, v, n * sizeof(T));
        return at;
    }
    template <class T> size_t add(const std::vector<T>& v) { return add(v.data(), v.size()); }
};

// Index of the source (added if new) for a level of face S.
uint32_t source_index(std::vector<SourcePlan>& src, uint32_t face, uint32_t S, bool split) {
    for (size_t i = 0; i < src.size(); ++i)
        if (!src[i].G.pad && src[i].G.S == S && src[i].split == split) return (uint32_t)i;
    SourcePlan s;
    s.G.S = S;
    s.split = split;
    s.level = ilog2(face / S);
    s.raw = 6 * S * S / 8;
    src.push_back(s);
    return (uint32_t)src.size() - 1;
}

// Rows, blocks, unit lists, weights, slices and launch tables of a plan whose
// levels are chosen. Sources are ordered levels first, planes after, so that
// the far normalisers exist when the near rows need them.
hipError_t build_plan(hvx_contract_plan* P, int ctype, bool split) {
    hipError_t e;
    std::vector<Job> jobs;
    std::vector<uint32_t> job_src, job_mip;
    std::vector<SourcePlan> src;
    size_t sbytes = 0, tbytes = 0;  // the scratch and, in it, the planes' texels
    std::vector<std::pair<uint32_t, size_t>> map_at;  // (far job, offset of its map in the scratch)
    uint32_t delta_mip = ~0u;
    size_t ztotal = 0;  // far normaliser maps, needed only here
    for (uint32_t m = 0; m < P->mips; ++m) {
        const ContractLevel& L = P->mp[m].L;
        if (L.kind == hvx::CONTRACT_DELTA) {
            delta_mip = m;
            continue;
        }
        Job J{};
        J.type = ctype;
        J.alpha2 = L.alpha2;
        J.t0 = L.t0;
        J.t1 = L.t1;
        J.out_off = hvx::cube_level_offset_floats(P->So, m) / 4;
        if (L.kind == hvx::CONTRACT_FULL) {
            J.piece = PIECE_WHOLE;
            J.So = L.So;
            job_src.push_back(source_index(src, P->S, L.Si, false));
        } else {
            J.piece = PIECE_FAR;
            J.So = L.Sf;
            job_src.push_back(source_index(src, P->S, L.Sf, split));  // low-roughness mips: near and far
            map_at.emplace_back((uint32_t)jobs.size(), scratch_take(&sbytes, 6 * (size_t)L.Sf * L.Sf * sizeof(float4)));
            J.zmap = (float4*)(ztotal * sizeof(float4));  // offset, until the maps are allocated
            ztotal += 6 * (size_t)L.Sf * L.Sf;
        }
        jobs.push_back(J);
        job_mip.push_back(m);
    }
    const uint32_t far_jobs = (uint32_t)map_at.size();
    for (uint32_t k = 0; k < far_jobs; ++k) {  // the near job of each far job, with a plane of its own
        const uint32_t m = job_mip[map_at[k].first];
        const ContractLevel& L = P->mp[m].L;
        Job J = jobs[map_at[k].first];
        J.piece = PIECE_NEAR;
        J.So = L.So;
        J.Sf = L.Sf;
        SourcePlan s;
        s.G.pad = 1;
        s.G.S = L.Si;
        s.G.B = plane_border(L.So, L.Si, L.t1);
        s.G.Pw8 = (L.Si + 2 * s.G.B) / 8;
        s.split = split;
        s.level = ilog2(P->S / L.Si);
        s.raw = (L.Si + 2 * s.G.B) * s.G.Pw8;
        job_src.push_back((uint32_t)src.size());
        src.push_back(s);
        map_at.emplace_back((uint32_t)jobs.size(), map_at[k].second);
        jobs.push_back(J);
        job_mip.push_back(m);
    }
    // rows and blocks by source
    std::vector<Row> rows;
    std::vector<Block> blocks;
    for (uint32_t s = 0; s < src.size(); ++s) {
        SourcePlan& S = src[s];
        S.row0 = (uint32_t)rows.size();
        S.block0 = (uint32_t)blocks.size();
        for (uint32_t j = 0; j < jobs.size(); ++j)
            if (job_src[j] == s) {
                const std::vector<Row> r = octant_rows(jobs[j].So, (uint16_t)j);
                rows.insert(rows.end(), r.begin(), r.end());
            }
        S.rows = (uint32_t)rows.size() - S.row0;
        for (uint32_t r = 0; r < S.rows; r += kBlockRows) {
            Block B{};
            B.row0 = S.row0 + r;
            B.nrows = std::min(kBlockRows, S.rows - r);
            B.nrt = (B.nrows + 15) / 16;
            B.src = s;
            B.split = S.split;
            for (uint32_t k = 0; k < B.nrows; ++k) rows[B.row0 + k].block = (uint16_t)blocks.size();
            blocks.push_back(B);
        }
        S.nblocks = (uint32_t)blocks.size() - S.block0;
        (S.G.pad ? P->near_rows : P->dense_rows) += S.rows;
        P->min_level = std::max(P->min_level, S.level);
        P->scale_level = std::min(P->scale_level, S.level);
    }
    Scratch zmaps;
    float4* d_zmaps = nullptr;
    if ((e = zmaps.get(&d_zmaps, ztotal)) != hipSuccess) return e;
    for (Job& J : jobs)
        if (J.piece != PIECE_WHOLE) J.zmap = d_zmaps + (size_t)J.zmap / sizeof(float4);
    // unit lists: the blocks' units with weight, as indices into the source's staged units
    std::vector<uint32_t> ulist, raw_ulist;  // raw: as the level or plane counts them
    Tables first;
    const size_t fj = first.add(jobs), fr = first.add(rows), fb = first.add(blocks);
    Scratch first_mem;
    char* d_first = nullptr;
    if ((e = first_mem.get(&d_first, first.bytes.size())) != hipSuccess ||
        (!first.bytes.empty() &&
         (e = hipMemcpy(d_first, first.bytes.data(), first.bytes.size(), hipMemcpyHostToDevice)) != hipSuccess))
        return e;
    for (SourcePlan& S : src) {
        Scratch mem;
        uint8_t* d_flags = nullptr;
        const size_t nf = (size_t)S.nblocks * S.raw;
        std::vector<uint8_t> flags(nf);
        if ((e = mem.get(&d_flags, nf)) != hipSuccess) return e;
        hipLaunchKernelGGL(unit_flag_kernel, dim3((S.raw + 255) / 256, S.nblocks), dim3(256), 0, nullptr, S.G,
                           (const Job*)(d_first + fj), (const Row*)(d_first + fr), (const Block*)(d_first + fb),
                           S.block0, S.raw, d_flags);
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = hipMemcpy(flags.data(), d_flags, nf, hipMemcpyDeviceToHost)) != hipSuccess)
            return e;
        std::vector<uint8_t> any(S.raw, 0);
        std::vector<uint32_t> index(S.raw, ~0u);
        for (uint32_t b = 0; b < S.nblocks; ++b)
            for (uint32_t u = 0; u < S.raw; ++u) any[u] |= flags[(size_t)b * S.raw + u];
        for (uint32_t u = 0; u < S.raw; ++u)
            if (any[u]) S.units.push_back(u);
        // stacked in y, eight rows at a time, so that staging works on square patches
        const uint32_t w = S.G.pad ? S.G.Pw8 : std::max(S.G.S / 8, 1u);
        auto key = [&](uint32_t u) { return ((uint64_t)(u / w / 8) * w + u % w) * 8 + u / w % 8; };
        std::sort(S.units.begin(), S.units.end(), [&](uint32_t a, uint32_t b) { return key(a) < key(b); });
        for (uint32_t k = 0; k < S.units.size(); ++k) index[S.units[k]] = k;
        for (uint32_t b = 0; b < S.nblocks; ++b) {
            Block& B = blocks[S.block0 + b];
            B.unit0 = (uint32_t)ulist.size();
            for (uint32_t u : S.units)
                if (flags[(size_t)b * S.raw + u]) ulist.push_back(index[u]), raw_ulist.push_back(u);
            B.nunits = (uint32_t)ulist.size() - B.unit0;
            B.nsteps = (B.nunits + 3) / 4;
        }
        if (S.G.pad) {  // the texels that the staged units' eight images read
            const uint32_t Pw = 8 * S.G.Pw8;
            std::vector<uint8_t> seen((size_t)Pw * Pw, 0);
            for (uint32_t u : S.units)
                for (uint32_t q = 0; q < 8; ++q) {
                    const uint32_t x = (u % S.G.Pw8) * 8 + q, y = u / S.G.Pw8, xr = Pw - 1 - x, yr = Pw - 1 - y;
                    for (const auto& p : {std::pair{x, y}, {xr, y}, {x, yr}, {xr, yr}}) {
                        seen[(size_t)p.second * Pw + p.first] = 1;
                        seen[(size_t)p.first * Pw + p.second] = 1;
                    }
                }
            // texels of the face itself, then those sampled inside another
            // face, then those whose taps meet an edge: the last kind takes
            // several times the instructions and would hold up most waves
            // (a row of the plane crosses two edges)
            auto kind = [&](uint32_t p) {
                const int s1 = (int)S.G.S, a = std::abs(2 * ((int)(p % Pw) - (int)S.G.B) + 1 - s1),
                          b = std::abs(2 * ((int)(p / Pw) - (int)S.G.B) + 1 - s1), m = std::max(a, b);
                if (m < s1) return 0;
                // the sample's coordinates off the other face's centre: S and min(a, b), over m
                const double hi = 0.5 * s1 * (1.0 + (double)std::max(s1, std::min(a, b)) / m) - 0.5;
                return hi + 1.0 < s1 - 1e-3 ? 1 : 2;
            };
            for (int k = 0; k < 3; ++k)
                for (uint32_t p = 0; p < Pw * Pw; ++p)
                    if (seen[p] && kind(p) == k) S.need.push_back(p);
            S.t_off = scratch_take(&tbytes, 6 * (size_t)Pw * Pw * (S.split ? 16 : 8));
        }
        S.r_off = scratch_take(&sbytes, S.units.size() * kCols * sizeof(half8) * (S.split ? 2 : 1));
    }
    // K slices: at most two workgroups per CU (what fits: one round, without a
    // tail) of kGoodSlice to kMaxSlice steps, a split step counting as two;
    // plans too small to fill the chip that way have shorter ones, for the
    // latency of a single probe (irradiance 32^2: 19.6 us against 25.4 with slices of 32). A
    // slice costs its 74 KB of partial sums, written and read once: 24 probes
    // 256^2 -> 128^2 x 8 took 384 us with slices of at least 16 steps, 361 us
    // with 24, 349 us with 32, 347 us with 40 (one probe 512^2 -> 256^2 x 9 in
    // split BF16 100 us up to 32, 103 us with 40; each timed before the kernels
    // around the GEMM had their present form); the 512^2 x 10 chain 10 us more
    // with 541 slices, in two rounds, than with 440 in one.
    uint64_t wunits = 0;
    const uint32_t slots = 2u * (uint32_t)std::max(P->ctx->num_cus, 1);
    auto slices = [&](const Block& B, uint32_t len) {
        const uint32_t groups = (B.nsteps + kGroup - 1) / kGroup, per = (B.split ? len / 2 : len) / kGroup;
        return (groups + per - 1) / per;
    };
    uint32_t len = kMinSlice;
    for (; len < kMaxSlice; len += 2 * kGroup) {
        uint32_t n = 0;
        for (const Block& B : blocks) n += slices(B, len);
        if (n <= (len < kGoodSlice ? slots / 8 : slots)) break;
    }
    std::vector<Item> items;
    for (uint32_t b = 0; b < blocks.size(); ++b) {
        Block& B = blocks[b];
        const uint64_t n = (uint64_t)B.nsteps * B.nrt * 64;
        B.woff = wunits;
        B.w_lo = B.split ? n : 0;
        wunits += B.split ? 2 * n : n;
        const uint32_t groups = (B.nsteps + kGroup - 1) / kGroup;
        B.nslices = slices(B, len);
        B.item0 = (uint32_t)items.size();
        for (uint32_t s = 0; s < B.nslices; ++s) {
            const uint32_t s0 = s * groups / B.nslices * kGroup, s1 = std::min((s + 1) * groups / B.nslices * kGroup, B.nsteps);
            items.push_back(Item{b, s0, s1 - s0, (uint32_t)items.size()});
        }
        for (uint32_t r = 0; r < B.nrows; ++r)
            P->mp[job_mip[rows[B.row0 + r].job]].weight_bytes += (uint64_t)B.nsteps * 32 * 2 * (B.split ? 2 : 1);
    }
    P->items = (uint32_t)items.size();
    // a level's blocks sum much the same units: slices at the same place of
    // their lists run side by side. Planes stay block by block: neighbouring
    // blocks have neighbouring windows.
    std::stable_sort(items.begin(), items.end(), [&](const Item& a, const Item& b) {
        const Block &A = blocks[a.block], &B = blocks[b.block];
        if (A.src != B.src) return A.src < B.src;
        return !src[A.src].G.pad && a.s0 < b.s0;
    });
    // per-call scratch
    const size_t fmax_off = scratch_take(&sbytes, 6 * kFaceMaxBlocks * sizeof(float));
    const size_t sc_off = scratch_take(&sbytes, 8 * sizeof(float));
    // the planes' texels are read for the last time before the first partial sum is written
    const size_t part_off = scratch_take(&sbytes, std::max((size_t)P->items * kBlockRows * kCols * sizeof(float), tbytes));
    P->scratch_bytes = (sbytes + 255) & ~(size_t)255;
    if ((e = P->alloc(&P->scratch, P->scratch_bytes)) != hipSuccess) return e;
    P->fmax = reinterpret_cast<float*>(P->scratch + fmax_off);
    P->sc = reinterpret_cast<float*>(P->scratch + sc_off);
    for (const auto& [j, off] : map_at) jobs[j].map = reinterpret_cast<float4*>(P->scratch + off);
    // pages touched here are not first touched by a call
    if ((e = hipMemset(P->scratch, 0, P->scratch_bytes)) != hipSuccess) return e;
    Tables tab;
    const size_t tj = tab.add(jobs), tr = tab.add(rows), tb = tab.add(blocks), ti = tab.add(items), tu = tab.add(ulist), traw = tab.add(raw_ulist);
    for (SourcePlan& S : src) {
        S.units_off = tab.add(S.units);
        S.need_off = tab.add(S.need);
    }
    const size_t tm = tab.add(source_table()), ts = tab.add<float>(nullptr, rows.size()),
                 tz = tab.add<float>(nullptr, rows.size());
    char* d_tab = nullptr;
    half8* W = nullptr;
    if ((e = P->alloc(&d_tab, tab.bytes.size())) != hipSuccess || (e = P->alloc(&W, wunits)) != hipSuccess ||
        (e = hipMemcpy(d_tab, tab.bytes.data(), tab.bytes.size(), hipMemcpyHostToDevice)) != hipSuccess)
        return e;
    const Job* d_jobs = reinterpret_cast<const Job*>(d_tab + tj);
    const Row* d_rows = reinterpret_cast<const Row*>(d_tab + tr);
    const Block* d_blocks = reinterpret_cast<const Block*>(d_tab + tb);
    const uint32_t* d_ulist = reinterpret_cast<const uint32_t*>(d_tab + tu);
    float *rowscale = reinterpret_cast<float*>(d_tab + ts), *invZ = reinterpret_cast<float*>(d_tab + tz);
    auto d_units = [&](const SourcePlan& S) { return reinterpret_cast<const uint32_t*>(d_tab + S.units_off); };
    // weights
    if (!rows.empty()) {
        Scratch zmem, wmem;
        double *Z = nullptr, *wm = nullptr;
        if ((e = zmem.get(&Z, rows.size())) != hipSuccess || (e = wmem.get(&wm, rows.size())) != hipSuccess) return e;
        for (const SourcePlan& S : src) {
            hipLaunchKernelGGL(row_sum_kernel, dim3(S.rows), dim3(256), 0, nullptr, S.G, d_jobs, d_rows, d_blocks,
                               d_ulist, d_units(S), S.row0, Z, wm);
            uint32_t most = 0;
            for (uint32_t b = 0; b < S.nblocks; ++b) {
                const Block& B = blocks[S.block0 + b];
                most = std::max(most, (B.nsteps * B.nrt * 64 + 255) / 256);
            }
            const dim3 grid(std::min(most, 4096u), S.nblocks);
            if (S.split)
                hipLaunchKernelGGL(weight_fill_kernel<true>, grid, dim3(256), 0, nullptr, S.G, d_jobs, d_rows,
                                   d_blocks, S.block0, d_ulist, d_units(S), wm, W);
            else
                hipLaunchKernelGGL(weight_fill_kernel<false>, grid, dim3(256), 0, nullptr, S.G, d_jobs, d_rows,
                                   d_blocks, S.block0, d_ulist, d_units(S), wm, W);
            hipLaunchKernelGGL(far_norm_kernel, dim3((S.rows * kImages + 255) / 256), dim3(256), 0, nullptr, d_jobs,
                               d_rows, S.row0, S.rows, Z);
        }
        hipLaunchKernelGGL(row_scale_kernel, dim3((uint32_t)(rows.size() + 255) / 256), dim3(256), 0, nullptr, d_jobs,
                           d_rows, (uint32_t)rows.size(), Z, wm, rowscale, invZ);
        if ((e = hipGetLastError()) != hipSuccess || (e = hipDeviceSynchronize()) != hipSuccess) return e;
    }
    P->d_jobs = d_jobs;
    P->d_rows = d_rows;
    P->rowscale = rowscale;
    P->invZ = invZ;
    // launch tables
    GemmArgs& A = P->gemm;
    A.W = W;
    A.blocks = d_blocks;
    A.items = reinterpret_cast<const Item*>(d_tab + ti);
    A.ulist = d_ulist;
    A.nitems = P->items;
    A.part = reinterpret_cast<float*>(P->scratch + part_off);
    StageTable& ST = P->stage;
    MapTable& MT = P->maps;
    auto stage_item = [&](StageItem I, uint32_t workgroups) {
        I.block_begin = ST.blocks;
        ST.blocks += workgroups;
        ST.it[ST.n++] = I;
    };
    ST.map = reinterpret_cast<const uint32_t*>(d_tab + tm);
    for (uint32_t s = 0; s < src.size(); ++s) {
        const SourcePlan& S = src[s];
        const uint32_t nu = (uint32_t)S.units.size();
        const uint64_t lo = S.split ? (uint64_t)nu * kCols : 0;
        const uint32_t ut = S.split ? tile_units<true>() : tile_units<false>(), tiles = (nu + ut - 1) / ut;
        half8* R = reinterpret_cast<half8*>(P->scratch + S.r_off);
        A.R[s] = R;
        A.r_lo[s] = lo;
        StageItem I{};
        I.split = S.split;
        I.S = S.G.S;
        I.level_off = hvx::cube_level_offset_floats(P->S, S.level) / 4;
        if (S.G.pad) {
            I.kind = STAGE_PLANE;
            I.B = S.G.B;
            I.Pw = 8 * S.G.Pw8;
            I.n = (uint32_t)S.need.size();
            I.list = reinterpret_cast<const uint32_t*>(d_tab + S.need_off);
            I.dst = reinterpret_cast<half8*>(P->scratch + part_off + S.t_off);
            stage_item(I, (6 * I.n + 255) / 256);
            MT.it[MT.n++] = MapItem{I.Pw, nu, MT.blocks, d_units(S), I.dst, R, lo};
            MT.blocks += tiles;
        } else {
            I.kind = STAGE_DENSE;
            I.n = nu;
            I.list = d_units(S);
            I.dst = R;
            I.lo_off = lo;
            stage_item(I, tiles);
            A.level_off[s] = I.level_off;
            A.log2_S[s] = ilog2(I.S);
            P->direct_units += nu;
        }
    }
    A.map = ST.map;
    A.sc = P->sc;
    A.raw_ulist = reinterpret_cast<const uint32_t*>(d_tab + traw);
    if (delta_mip != ~0u) {
        StageItem I{};
        I.kind = STAGE_DELTA;
        I.S = P->mp[delta_mip].L.So;
        I.level_off = hvx::cube_level_offset_floats(P->So, delta_mip) / 4;
        stage_item(I, (6 * I.S * I.S + 255) / 256);
    }
    // gemm_direct takes plans of levels that one block of rows sums each (mixed
    // with others, its slower slices left some XCDs waiting). What is left to
    // stage: an item of no texels, whose workgroup writes the scales, and the
    // roughness-0 mip
    for (const SourcePlan& S : src)
        if (S.nblocks != 1 || S.split || S.G.pad) P->direct_units = 0;
    StageTable& SR = P->stage_rest;
    SR.it[SR.n++] = StageItem{.kind = STAGE_PLANE};
    SR.blocks = 1;
    SR.map = ST.map;
    if (delta_mip != ~0u) {
        SR.it[SR.n] = ST.it[ST.n - 1];
        SR.it[SR.n++].block_begin = SR.blocks;
        SR.blocks += ST.blocks - ST.it[ST.n - 1].block_begin;
    }
    return hipSuccess;
}

// From this many units over all probes on, plans that it can take go through
// gemm_direct; below, the latency of its staging counts. us staged / direct: 64
// probes 16^2 -> 16^2 x 5 31.1 / 26.3, 1,024 242 / 145; 64 probes 8^2 -> 8^2 x 4
// (3,072 units) 25.7 / 28.0, 256 37.1 / 28.5; 24 probes 32^2 -> 16^2 x 5 31.9 / 24;
// 8 probes 64^2 -> 32^2 x 6 42 / 37, 24 78 / 69, 256 876 / 647.
constexpr uint64_t kDirectUnits = 8192;

// The launches of a filter call over n probes (grid dimension y, z for the
// face maxima, interleaved for the GEMM: probe). delta_chain (single probe,
// nullable): the chain the delta mip samples instead of the probe's chain.
int launch_call(hvx_contract_plan* P, const Probes& Q, uint32_t n, uint32_t chain_levels, hipStream_t s,
                const char* what, const float4* delta_chain = nullptr) {
    hvx_ctx* ctx = P->ctx;
    if (chain_levels <= P->min_level)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "the input chain needs %u levels (has %u); build it with "
                     "hvx_ibl_cube_mips", P->min_level + 1, chain_levels);
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || (cur != ctx->device && hipSetDevice(ctx->device) != hipSuccess))
        return pfail(ctx, HVX_ERR_HIP, "cannot bind device %d", ctx->device);
    // exponent scales from the finest staged level: coarser levels are its box
    // means and padded texels its bilinear samples, so its maxima bound them
    uint32_t nb = 0;
    if (P->items) {
        const uint32_t Sl = std::max(P->S >> P->scale_level, 1u), S2 = Sl * Sl;
        nb = std::min(kFaceMaxBlocks, (S2 + 255) / 256);
        hipLaunchKernelGGL(facemax_kernel, dim3(nb, 6, n), dim3(256), 0, s, Q,
                           hvx::cube_level_offset_floats(P->S, P->scale_level) / 4, Sl, P->fmax);
    }
    const bool direct = n * (uint64_t)P->direct_units >= kDirectUnits;
    const StageTable& stage = direct ? P->stage_rest : P->stage;
    if (stage.blocks)
        hipLaunchKernelGGL(stage_kernel, dim3(stage.blocks, n), dim3(256), 0, s, Q, stage, P->fmax, nb, P->sc,
                           delta_chain, P->S);
    if (P->maps.blocks)
        hipLaunchKernelGGL(plane_map_kernel, dim3(P->maps.blocks, n), dim3(256), 0, s, Q, P->maps);
    if (P->items) {
        hipLaunchKernelGGL(direct ? contract_gemm_kernel<true> : contract_gemm_kernel<false>,
                           dim3((P->items * n + kXcds - 1) / kXcds * kXcds), dim3(256), 0, s, Q, P->gemm);
        hipLaunchKernelGGL(epilogue_kernel<false>, dim3((P->dense_rows * kImages + 255) / 256, n), dim3(256), 0, s, Q,
                           P->d_jobs, P->d_rows, P->gemm.blocks, P->gemm.part, P->rowscale, P->invZ, P->sc, 0u,
                           P->dense_rows);
    }
    if (P->near_rows)
        hipLaunchKernelGGL(epilogue_kernel<true>, dim3((P->near_rows * kImages + 255) / 256, n), dim3(256), 0, s, Q,
                           P->d_jobs, P->d_rows, P->gemm.blocks, P->gemm.part, P->rowscale, P->invZ, P->sc,
                           P->dense_rows, P->near_rows);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : pfail(ctx, HVX_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

// Copies of the per-call scratch that a multi-probe call over n probes runs
// in: all of them up to 16 GiB, then the call is cut. Cutting it further, so
// that what one launch stages stays in the caches for the next, mostly does not
// pay: 24 probes 256^2 -> 128^2 x 8 take 341 us at once, 374 cut at 192 MiB, 425
// at 96 MiB; 256 probes 64^2 -> 64^2 x 7 1,316 us, 1,170 cut at 256 MiB, 1,644 at 64.
constexpr size_t kMultiBytes = 16ull << 30;
uint32_t multi_copies(size_t scratch_bytes, uint32_t n) {
    const size_t fit = kMultiBytes / std::max<size_t>(scratch_bytes, 1);
    return (uint32_t)std::min<size_t>(n, std::max<size_t>(fit, 4));
}

// Hot-texel blocks at least max(0.5, 300 level-0 texel widths) radians
// outside a workgroup's cone of output directions enter its sum as one
// entry: the relative error of that entry is about 10 (block extent /
// distance)^2, under 2e-4 for 4x4 level-0 blocks (rms extent about 1.3
// texel widths); faces below 1024 therefore aggregate little or nothing.
float hot_near(uint32_t S) { return std::max(0.5f, 300.0f * 1.5707963f / (float)S); }

// A single-probe call with the bright-texel split: threshold, clamped level 0
// and its box levels, the hot list, the contraction of the clamped chain (the
// delta mip samples the caller's chain), then the hot texels' exact sum.
int launch_hot_call(hvx_contract_plan* P, const float* d_chain, uint32_t chain_levels, float* d_out, hipStream_t s) {
    hvx_ctx* ctx = P->ctx;
    if (chain_levels <= P->min_level)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "the input chain needs %u levels (has %u); build it with "
                     "hvx_ibl_cube_mips", P->min_level + 1, chain_levels);
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || (cur != ctx->device && hipSetDevice(ctx->device) != hipSuccess))
        return pfail(ctx, HVX_ERR_HIP, "cannot bind device %d", ctx->device);
    const HotArgs H{reinterpret_cast<const float4*>(d_chain), reinterpret_cast<float4*>(P->hot_chain), P->S,
                    P->hot_k, P->hot_hist, P->hot_cnt, P->hot_T, P->hot_idx, P->hot_list, P->hot_groups};
    const size_t texels = 6ull * P->S * P->S;
    hipLaunchKernelGGL(hot_hist_kernel, dim3((uint32_t)std::min<size_t>(1024, (texels + 1023) / 1024)), dim3(256), 0,
                       s, H);
    hipLaunchKernelGGL(hot_select_kernel, dim3(1), dim3(1024), 0, s, H);
    hipLaunchKernelGGL(hot_compact_kernel, dim3((uint32_t)((texels + 255) / 256)), dim3(256), 0, s, H);
    hipLaunchKernelGGL(hot_list_kernel, dim3(1), dim3(1024), 0, s, H);
    hipLaunchKernelGGL(hot_group_kernel, dim3((hvx::kHotMax + 255) / 256), dim3(256), 0, s, H);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pfail(ctx, HVX_ERR_HIP, "bright-texel split: %s", hipGetErrorString(e));
    if (P->min_level > 0 && (e = hvx::launch_cube_mips(P->hot_chain, P->S, P->min_level + 1, s)) != hipSuccess)
        return pfail(ctx, HVX_ERR_HIP, "clamped chain levels: %s", hipGetErrorString(e));
    const Probes Q{reinterpret_cast<const float4*>(P->hot_chain), reinterpret_cast<float4*>(d_out), nullptr, nullptr,
                   0, 0, 1};
    int st = launch_call(P, Q, 1, chain_levels, s, "hvx_ibl_filter_contract", reinterpret_cast<const float4*>(d_chain));
    if (st) return st;
    HotAdd A{};
    uint32_t first = 0;
    const int ctype = P->type == HVX_FILTER_DIFFUSE ? hvx::CONTRACT_DIFFUSE : hvx::CONTRACT_SPECULAR;
    for (uint32_t m = 0; m < P->mips; ++m) {
        const ContractLevel& L = P->mp[m].L;
        if (L.kind == hvx::CONTRACT_DELTA) continue;
        HotMip& M = A.m[A.nm++];
        M.So = L.So;
        M.first = first;
        M.alpha2 = (float)L.alpha2;
        M.h1 = (float)(0.5 * (1.0 - L.alpha2));
        const double z = hvx::contract_weight_integral(ctype, L.alpha2);
        M.scale = (float)((ctype == hvx::CONTRACT_DIFFUSE ? 1.0 : L.alpha2 / hvx::kContractPi) / z);
        M.out_off = hvx::cube_level_offset_floats(P->So, m) / 4;
        first += (6 * L.So * L.So + 63) / 64 * 64;
    }
    if (A.nm == 0) return HVX_OK;
    A.blocks = first / 64;
    A.list = P->hot_list;
    A.groups = P->hot_groups;
    A.cnt = P->hot_cnt;
    A.theta_near = hot_near(P->S);
    A.out = reinterpret_cast<float4*>(d_out);
    if (ctype == hvx::CONTRACT_DIFFUSE)
        hipLaunchKernelGGL(hot_add_kernel<true>, dim3(A.blocks), dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL(hot_add_kernel<false>, dim3(A.blocks), dim3(256), 0, s, A);
    e = hipGetLastError();
    return e == hipSuccess ? HVX_OK : pfail(ctx, HVX_ERR_HIP, "bright-texel sum: %s", hipGetErrorString(e));
}

}  // namespace

extern "C" {

int hvx_ibl_contract_plan_create(hvx_ctx* ctx, int type, uint32_t face, uint32_t out_face, uint32_t out_mips,
                                 int precision, hvx_contract_plan** out) {
    if (!ctx || !out) return HVX_ERR_NULL;
    *out = nullptr;
    if (type != HVX_FILTER_DIFFUSE && type != HVX_FILTER_SPECULAR)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "unknown filter type %d", type);
    if (precision != HVX_PRECISION_FP16_SCALED && precision != HVX_PRECISION_BF16_SPLIT)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "unknown precision %d", precision);
    const bool split = precision == HVX_PRECISION_BF16_SPLIT;
    if (type == HVX_FILTER_DIFFUSE && out_mips != 1)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "the diffuse filter writes one mip");
    if (face < 4 || face > 8192 || (face & (face - 1)) || out_face < 1 || out_face > 4096 ||
        (out_face & (out_face - 1)) || out_mips < 1 || out_mips > hvx_mip_count(out_face) ||
        out_mips > hvx::kContractMaxMips)
        return pfail(ctx, HVX_ERR_INVALID_ARG, "sizes: face %u and out_face %u must be powers of two (face >= 4), "
                     "out_mips in [1, mips(out_face)]", face, out_face);
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || (cur != ctx->device && hipSetDevice(ctx->device) != hipSuccess))
        return pfail(ctx, HVX_ERR_HIP, "cannot bind device %d", ctx->device);
    hvx_contract_plan* P = new (std::nothrow) hvx_contract_plan();
    if (!P) return HVX_ERR_HIP;
    P->ctx = ctx;
    P->type = type;
    P->precision = precision;
    P->S = face;
    P->So = out_face;
    P->mips = out_mips;
    ContractLevel lv[hvx::kContractMaxMips];
    const int ctype = type == HVX_FILTER_DIFFUSE ? hvx::CONTRACT_DIFFUSE : hvx::CONTRACT_SPECULAR;
    hvx::contract_levels(ctype, face, out_face, out_mips, lv);
    P->mp.resize(out_mips);
    for (uint32_t m = 0; m < out_mips; ++m) P->mp[m].L = lv[m];
    hipError_t e;
    try {
        e = build_plan(P, ctype, split);
    } catch (const std::bad_alloc&) {
        e = hipErrorOutOfMemory;
    }
    if (e != hipSuccess) {
        hvx_ibl_contract_plan_destroy(P);
        return pfail(ctx, HVX_ERR_HIP, "contraction plan: %s", hipGetErrorString(e));
    }
    *out = P;
    return HVX_OK;
}

int hvx_ibl_contract_plan_destroy(hvx_contract_plan* P) {
    if (!P) return HVX_ERR_NULL;
    (void)hipDeviceSynchronize();
    for (void* p : P->allocs) (void)hipFree(p);
    if (P->mscratch) (void)hipFree(P->mscratch);
    delete P;
    return HVX_OK;
}

int hvx_ibl_contract_plan_query(const hvx_contract_plan* P, uint32_t mip, hvx_contract_mip_info* info) {
    if (!P || !info) return HVX_ERR_NULL;
    if (mip >= P->mips) return HVX_ERR_INVALID_ARG;
    const MipPlan& M = P->mp[mip];
    info->kind = M.L.kind;
    info->out_face = M.L.So;
    info->in_face = M.L.Si;
    info->far_face = M.L.Sf;
    info->window_t0 = (float)M.L.t0;
    info->window_t1 = (float)M.L.t1;
    info->weight_bytes = M.weight_bytes;
    info->min_input_level = P->min_level;
    return HVX_OK;
}

int hvx_ibl_filter_contract(hvx_contract_plan* P, const float* d_chain, uint32_t chain_levels, float* d_out,
                            void* stream) {
    if (!P) return HVX_ERR_NULL;
    hvx_ctx* ctx = P->ctx;
    if (!d_chain || !d_out) return pfail(ctx, HVX_ERR_NULL, "NULL chain or output");
    if (((uintptr_t)d_chain | (uintptr_t)d_out) % 16) return pfail(ctx, HVX_ERR_ALIGN, "chains need 16-byte alignment");
    if (P->hot_k) return launch_hot_call(P, d_chain, chain_levels, d_out, (hipStream_t)stream);
    const Probes Q{reinterpret_cast<const float4*>(d_chain), reinterpret_cast<float4*>(d_out), nullptr, nullptr, 0, 0, 1};
    return launch_call(P, Q, 1, chain_levels, (hipStream_t)stream, "hvx_ibl_filter_contract");
}

int hvx_ibl_contract_plan_set_hot(hvx_contract_plan* P, uint32_t max_hot) {
    if (!P) return HVX_ERR_NULL;
    if (max_hot > hvx::kHotMax)
        return pfail(P->ctx, HVX_ERR_INVALID_ARG, "max_hot must be in [0, %u]", hvx::kHotMax);
    if (max_hot && !P->hot_chain) {
        hipError_t e;
        if ((e = P->alloc(&P->hot_chain, hvx::cube_level_offset_floats(P->S, P->min_level + 1))) != hipSuccess ||
            (e = P->alloc(&P->hot_hist, hvx::kHotBins)) != hipSuccess ||
            (e = P->alloc(&P->hot_cnt, 3)) != hipSuccess || (e = P->alloc(&P->hot_T, 1)) != hipSuccess ||
            (e = P->alloc(&P->hot_idx, hvx::kHotMax)) != hipSuccess ||
            (e = P->alloc(&P->hot_list, 2 * hvx::kHotMax)) != hipSuccess ||
            (e = P->alloc(&P->hot_groups, 2 * hvx::kHotMax)) != hipSuccess ||
            (e = hipMemset(P->hot_hist, 0, hvx::kHotBins * sizeof(uint32_t))) != hipSuccess ||
            (e = hipMemset(P->hot_cnt, 0, 3 * sizeof(uint32_t))) != hipSuccess ||
            (e = hipDeviceSynchronize()) != hipSuccess) {
            P->hot_chain = nullptr;  // the partial allocations are released with the plan
            return pfail(P->ctx, HVX_ERR_HIP, "bright-texel split buffers: %s", hipGetErrorString(e));
        }
    }
    P->hot_k = max_hot;
    return HVX_OK;
}

int hvx_ibl_contract_hot_info(hvx_contract_plan* P, float* threshold, uint32_t* n_hot) {
    if (!P || !threshold || !n_hot) return HVX_ERR_NULL;
    if (!P->hot_chain) return pfail(P->ctx, HVX_ERR_INVALID_ARG, "the bright-texel split was never enabled");
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(threshold, P->hot_T, sizeof(float), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(n_hot, P->hot_cnt + 1, sizeof(uint32_t), hipMemcpyDeviceToHost);
    return e == hipSuccess ? HVX_OK : pfail(P->ctx, HVX_ERR_HIP, "hvx_ibl_contract_hot_info: %s", hipGetErrorString(e));
}

int hvx_ibl_contract_plan_reserve(hvx_contract_plan* P, uint32_t max_probes) {
    if (!P) return HVX_ERR_NULL;
    if (max_probes == 0 || max_probes > kMaxProbes)
        return pfail(P->ctx, HVX_ERR_INVALID_ARG, "max_probes must be in [1, %u]", kMaxProbes);
    if (max_probes <= P->mcap) return HVX_OK;
    uint32_t copies = multi_copies(P->scratch_bytes, max_probes);
    if (copies <= P->mcopies) {
        P->mcap = max_probes;
        return HVX_OK;
    }
    (void)hipDeviceSynchronize();  // the old copies may be in use
    if (P->mscratch) (void)hipFree(P->mscratch);
    P->mscratch = nullptr;
    P->mcap = P->mcopies = 0;
    // where the memory is short, fewer copies and more passes
    hipError_t e;
    while ((e = hipMalloc(reinterpret_cast<void**>(&P->mscratch), P->scratch_bytes * copies)) != hipSuccess && copies > 1) {
        (void)hipGetLastError();
        copies = (copies + 1) / 2;
    }
    if (e != hipSuccess || (e = hipMemset(P->mscratch, 0, P->scratch_bytes * copies)) != hipSuccess) {
        if (P->mscratch) (void)hipFree(P->mscratch);
        P->mscratch = nullptr;
        return pfail(P->ctx, HVX_ERR_HIP, "multi-probe scratch (%zu bytes): %s", P->scratch_bytes * copies,
                     hipGetErrorString(e));
    }
    P->mcap = max_probes;
    P->mcopies = copies;
    return HVX_OK;
}

int hvx_ibl_filter_contract_multi(hvx_contract_plan* P, uint32_t n, const float* const* d_chains,
                                  uint32_t chain_levels, float* const* d_outs, void* stream) {
    if (!P) return HVX_ERR_NULL;
    if (!d_chains || !d_outs) return pfail(P->ctx, HVX_ERR_NULL, "NULL pointer arrays");
    if (n == 0) return HVX_OK;
    if (n > P->mcap)
        return pfail(P->ctx, HVX_ERR_CAPACITY, "%u probes but scratch reserved for %u (hvx_ibl_contract_plan_reserve)",
                     n, P->mcap);
    if (P->hot_k)
        return pfail(P->ctx, HVX_ERR_UNSUPPORTED, "the bright-texel split serves single-probe calls only");
    for (uint32_t p = 0; p < n; p += P->mcopies) {
        const uint32_t m = std::min(n - p, P->mcopies);
        const Probes Q{nullptr, nullptr, reinterpret_cast<const float4* const*>(d_chains) + p,
                       reinterpret_cast<float4* const*>(d_outs) + p,
                       (uint64_t)(reinterpret_cast<uintptr_t>(P->mscratch) - reinterpret_cast<uintptr_t>(P->scratch)),
                       (uint64_t)P->scratch_bytes, m};
        const int st = launch_call(P, Q, m, chain_levels, (hipStream_t)stream, "hvx_ibl_filter_contract_multi");
        if (st) return st;
    }
    return HVX_OK;
}

}  // extern "C"
