// ibl_kernels.hip — image-based-lighting precompute on gfx950.
//
// Reference shaders (HelloVulkan/Shaders/IBL) and their kernels here:
//   BRDFLUT.comp:26-71             -> brdf_lut_kernel (workgroup per LUT row;
//                                     the row's GGX half-vectors staged in LDS)
//   Equirect2Cube.frag:87-107      -> equirect_kernel (lane per cube texel)
//   VulkanImage::GenerateMipmap    -> mip_kernel (2x2 boxes, five levels a launch)
//   CubeFilterDiffuse.frag:35-136  -> diffuse_stage_kernel (four bilinear
//                                     footprints to a 128-byte line) and
//                                     diffuse_kernel (64 to 256 lanes per
//                                     output texel evaluate samples, loads one
//                                     round ahead; one lane per texel and
//                                     channel sums them in order; the
//                                     phi/theta sin/cos grid in LDS)
//   CubeFilterSpecular.frag:34-146 -> ggx_table_kernel (tangent-space GGX
//                                     samples per mip, computed once),
//                                     specular_delta_kernel (mip 0, roughness
//                                     0: the n identical samples evaluated
//                                     once, lane per texel) and
//                                     specular_split_kernel (mips >= 1: each
//                                     texel's samples spread over 16 lanes, the
//                                     terms summed in sample order through
//                                     LDS; tap loads one round ahead)
// The per-sample sequence and every summation order are the reference's, so
// outputs reproduce the FP32 oracle to the bit; the precomputed tables hold
// exactly the values the per-sample code would compute (same functions, same
// inputs), they are only hoisted out of the per-texel loops.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "hvx_device.h"
#include "hvx_internal.h"
#include "spec_tiles.h"

namespace hvx {
namespace {

// ImportanceSampleGGX (IBL/Header.glsl:14-28): tangent-space half vector of
// Hammersley sample i of n at roughness `rough`.
__device__ __forceinline__ float4 ggx_tangent_sample(uint32_t i, uint32_t n, float rough) {
    const float xix = (float)i / (float)n;
    const float xiy = radical_inverse_vdc(i);
    const float a = rough * rough;
    const float phi = (2.0f * kPiF) * xix;
    const float cosTheta = sqrtf_((1.0f - xiy) / (1.0f + (a * a - 1.0f) * xiy));
    const float sinTheta = sqrtf_(1.0f - cosTheta * cosTheta);
    return make_float4(cosf_(phi) * sinTheta, sinf_(phi) * sinTheta, cosTheta, 0.0f);
}

// tangent frame of IBL/Header.glsl:31-35
struct Frame {
    f3 t, b;
};
__device__ __forceinline__ Frame ggx_frame(f3 N) {
    const f3 up = absf(N.z) < 0.999f ? make3(0.0f, 0.0f, 1.0f) : make3(1.0f, 0.0f, 0.0f);
    const f3 t = normalize3(cross3(up, N));
    return {t, cross3(N, t)};
}

__device__ __forceinline__ f3 ggx_world(const Frame& fr, f3 N, float4 h) {
    const f3 sv = add3(add3(mul3(fr.t, h.x), mul3(fr.b, h.y)), mul3(N, h.z));
    return normalize3(sv);
}

// ---------------------------------------------------------------- BRDF LUT
constexpr int kLutChunk = 1024;

// A workgroup per row (its roughness' half vectors staged in LDS), PER texels
// per lane. Bound by VALU issue. The shader's N is (0, 0, 1) and V = (x, 0, z):
// the products with their zeros only ever add a zero, and of the light vector
// only its length and z count, so they are left out (signs of zero cannot
// reach the sums: every factor they meet is a positive sum or a product with
// N.L > 0); G's V half is the texel's, N.H the sample's. FAST (sample counts
// up to 2^20, where no half vector is horizontal): the exact divisions without
// scaling and the exact normalisation from the length's bit pattern (|L| = 1
// up to rounding). 512^2 x 1024: 428 us (1,186 us with four texels per lane, half of them
// past the row's end, and the general operations).
template <int PER, bool FAST>
__global__ __launch_bounds__(512) void brdf_lut_kernel(uint32_t W, uint32_t H, uint32_t n, float2* __restrict__ lut) {
    __shared__ float4 s_h[kLutChunk];
    const uint32_t y = blockIdx.x;
    const float rough = 1.0f - ((float)y + 0.5f) / (float)H;
    const f3 N = make3(0.0f, 0.0f, 1.0f);
    const Frame fr = ggx_frame(N);
    const float alpha = (rough * rough) / 2.0f;  // AlphaIBL
    const float oma = 1.0f - alpha;
    float lx[PER], ly[PER], nov[PER], vx[PER], GV[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const uint32_t x = threadIdx.x + q * blockDim.x;
        nov[q] = ((float)min(x, W - 1) + 0.5f) / (float)W;
        vx[q] = sqrtf_(1.0f - nov[q] * nov[q]);
        GV[q] = nov[q] / (nov[q] * oma + alpha);
        lx[q] = 0.0f;
        ly[q] = 0.0f;
    }
    for (uint32_t c0 = 0; c0 < n; c0 += kLutChunk) {
        const uint32_t cn = min((uint32_t)kLutChunk, n - c0);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < cn; i += blockDim.x) {
            const float4 h = ggx_tangent_sample(c0 + i, n, rough);
            const f3 w = ggx_world(fr, N, h);
            s_h[i] = make_float4(w.x, w.y, w.z, gmax(w.z, 0.0f));
        }
        __syncthreads();
        for (uint32_t i = 0; i < cn; ++i) {
            const float4 h = s_h[i];
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const float vh = vx[q] * h.x + nov[q] * h.z, k = 2.0f * vh;
                const float Lx = h.x * k - vx[q], Ly = h.y * k, Lz = h.z * k - nov[q];
                const float len2 = (Lx * Lx + Ly * Ly) + Lz * Lz;
                const float dotNL = Lz * (FAST ? inv_unit_length(len2) : 1.0f / sqrtf_(len2));
                if (dotNL > 0.0f) {
                    const float dotVH = gmax(vh, 0.0f);
                    const float gl = dotNL * oma + alpha, d = h.w * nov[q];
                    const float GL = FAST ? div_rn_normal(dotNL, gl) : dotNL / gl;
                    const float g = (GL * GV[q]) * dotVH;
                    const float G_Vis = FAST ? div_rn_normal(g, d) : g / d;
                    const float Fc = pow5f(1.0f - dotVH);
                    lx[q] = lx[q] + (1.0f - Fc) * G_Vis;
                    ly[q] = ly[q] + Fc * G_Vis;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const uint32_t x = threadIdx.x + q * blockDim.x;
        if (x < W) lut[(size_t)y * W + x] = make_float2(lx[q] / (float)n, ly[q] / (float)n);
    }
}

// ------------------------------------------------------------ equirect->cube
// A workgroup takes 64 x 4 texels of a face. What bounds it: at 1024^2 from
// 2048 x 1024 the 33 MB read and 100 MB written are 27 us; it took 86 us with the
// double-precision functions and wrapped indices as they are written (six
// divisions and four remainders a texel), 47 with their short forms.
__global__ __launch_bounds__(256) void equirect_kernel(const float4* __restrict__ eq, uint32_t w, uint32_t h,
                                                       float4* __restrict__ cube, uint32_t S) {
    const uint32_t x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + threadIdx.x / 64, face = blockIdx.z;
    if (x >= S || y >= S) return;
    const f3 d = texel_dir((int)face, (int)x, (int)y, (int)S);
    const float rpi = rcp_rn_normal(kPiF);
    const float s = 0.5f + div_by_normal(0.5f * atan2f_rn(d.z, d.x), kPiF, rpi);
    const float t = 1.0f - div_by_normal(acosf_rn(d.y), kPiF, rpi);
    const f3 c = sample_2d_rgba_repeat(eq, (int)w, (int)h, s, t);
    cube[((size_t)face * S + y) * S + x] = make_float4(c.x, c.y, c.z, 1.0f);
}

// ---------------------------------------------------------------- mip chain
// Up to five levels per launch: a workgroup takes a 32 x 32 tile of a face of
// level `sp` (the whole face if it is smaller) down to one texel, each level
// from the one before in LDS, so the chain of a 1024^2 cube is two launches
// (52 us one level each, 26 so). Grid dimension y: chains `pstride` float4s apart.
constexpr uint32_t kMipLevels = 5;
struct MipArgs {
    const float4* src;
    float4* dst[kMipLevels];
    uint32_t sp, levels;
    size_t pstride;
};
__device__ __forceinline__ float4 mip_mean(float4 a, float4 b, float4 c, float4 d) {
    return make_float4(((a.x + b.x) + (c.x + d.x)) * 0.25f, ((a.y + b.y) + (c.y + d.y)) * 0.25f,
                       ((a.z + b.z) + (c.z + d.z)) * 0.25f, ((a.w + b.w) + (c.w + d.w)) * 0.25f);
}
__global__ __launch_bounds__(256) void mip_kernel(MipArgs a) {
    __shared__ float4 sh[2][16][16];
    const uint32_t T = min(a.sp, 32u), per = a.sp / T;  // tiles per row of a face
    const uint32_t tx = blockIdx.x % per, ty = blockIdx.x / per % per, f = blockIdx.x / (per * per);
    const size_t chain = blockIdx.y * a.pstride;
    uint32_t n = T / 2, x = threadIdx.x % 16, y = threadIdx.x / 16;
    if (x < n && y < n) {
        const float4* p = a.src + chain + ((size_t)f * a.sp + ty * T + 2 * y) * a.sp + tx * T + 2 * x;
        const float4 m = mip_mean(p[0], p[1], p[a.sp], p[a.sp + 1]);
        const uint32_t sn = a.sp / 2;
        a.dst[0][chain + ((size_t)f * sn + ty * n + y) * sn + tx * n + x] = m;
        sh[0][y][x] = m;
    }
#pragma unroll 1
    for (uint32_t l = 1; l < a.levels; ++l) {
        __syncthreads();
        n /= 2;
        if (threadIdx.x < n * n) {
            x = threadIdx.x % n;
            y = threadIdx.x / n;
            const float4(*s)[16] = sh[(l - 1) & 1];
            const float4 m = mip_mean(s[2 * y][2 * x], s[2 * y][2 * x + 1], s[2 * y + 1][2 * x], s[2 * y + 1][2 * x + 1]);
            const uint32_t sn = a.sp >> (l + 1);
            a.dst[l][chain + ((size_t)f * sn + ty * n + y) * sn + tx * n + x] = m;
            sh[l & 1][y][x] = m;
        }
    }
}

// Orders a wave's LDS stores before its later LDS loads of what other lanes
// of the same wave stored (no workgroup barrier needed).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------- diffuse
// The reference sums 252 x 63 = 15,876 samples per output texel in one
// sequential loop (phi outer, theta inner). A lane per texel leaves the GPU
// idle (6,144 texels at 32^2), so here a workgroup owns TEX texels and its
// THREADS lanes evaluate THREADS / TEX consecutive samples of each texel per
// round; the weighted values go to LDS and one "summer" lane per texel and
// channel adds them in the reference's order. Results are bit-identical to
// the sequential loop. The kernel waits on gathers (at 1024^2 every sample
// reads about two fresh 128-byte lines; a few percent of its time issues
// arithmetic), so samples read their footprint from a staged copy
// (diffuse_stage_kernel, one line per sample), a lane's loads are issued
// one round ahead of their use, and the LDS rounds are double-buffered: the
// gathers of round r+1 are in flight while round r is weighted, stored and
// summed. 32^2 from 1024^2 (staging included): 3.54 ms with 16 texels and no
// loads ahead; gathered from the cube (the path for stream capture before the
// context holds a staging buffer) 2.66 ms with 4 texels per 256-lane workgroup
// (3.11 / 3.31 / 2.77 ms with 8 / 16 / 2); 1.77 ms with a staged 64-byte entry
// per footprint and 8 texels; 1.64 with four footprints to a line; 1.58 with 4
// texels. Small maps wait for their rounds, so they take fewer texels and more
// samples a round (us with 1 / 2 / 4 texels per workgroup): 4^2 from 32^2 159 /
// 196 / 221, 16^2 from 128^2 183 / 207 / 240 and 18^2 198 / 214 / 243, but 20^2 (2,400
// workgroups of one texel do not fit the card at once) 327 / 228 / 256; from larger
// faces the fabric sets in earlier: 12^2 from 256^2 177 / 209 / 232 and from 512^2
// 292 / 228 / 240, 16^2 from 1024^2 535 / 502 / 477; 10^2 from 512^2 184 / 216 / 239
// and from 1024^2 289 / 276 / 299; 24^2 from 64^2 363 / 249 / 270, from 512^2 802 /
// 790 / 826 (18^2: 506 / 489 / 439), 32^2 from 64^2 589 / 426 / 348.
constexpr int kMaxPhi = 512, kMaxTheta = 128;
#ifndef HVX_DIFFUSE_TEX
#define HVX_DIFFUSE_TEX 4
#endif
constexpr int kDTex = HVX_DIFFUSE_TEX;  // texels per workgroup
static_assert(kDTex == 1 || kDTex == 2 || kDTex == 4 || kDTex == 8 || kDTex == 16, "texels per workgroup: 1, 2, 4, 8 or 16");
#ifndef HVX_DIFFUSE_THREADS
#define HVX_DIFFUSE_THREADS 256
#endif
constexpr int kDThreads = HVX_DIFFUSE_THREADS;  // lanes per workgroup
static_assert(kDThreads == 128 || kDThreads == 256, "lanes per workgroup: 128 or 256");
#ifndef HVX_DIFFUSE_WAVES_PER_EU
#define HVX_DIFFUSE_WAVES_PER_EU 4
#endif

// Staged footprints: a bilinear footprint of level 0 with first texel (i0, j0),
// -1 <= i0, j0 <= S - 1, on face f is two columns of two texels, and four
// neighbouring footprints of a row are five columns: one 128-byte line at
// (f (S+1) + j0 + 1) stage_lines(S) + (i0 + 1) / 4 holds columns 4 k - 1 .. 4 k + 3
// as (texel j0, texel j0 + 1) RGB RGB, 24 bytes each, exactly as sample_cube
// reads the taps (texels across an edge folded onto the neighbouring face, a
// tap off both edges the mean of three texels). A sample reads the 48 bytes from
// column (i0 + 1) % 4 on: one line instead of two rows of texels (2.3 lines on
// average), and the bilinear sums are unchanged to the bit. Twice the cube (202
// MB at 1024^2), so it stays in the 256 MB of last-level cache: with an entry of
// 64 bytes for every footprint (403 MB) 32^2 from 1024^2 took 1.77 ms, so 1.64 (with
// 4 texels to a workgroup 11 GB of lines at 7.2 TB/s).
__host__ __device__ inline uint32_t stage_lines(uint32_t S) { return (S + 4) / 4; }
__global__ __launch_bounds__(256) void diffuse_stage_kernel(const float4* __restrict__ cube, uint32_t S,
                                                           float2* __restrict__ lines) {
    // eight lanes per line: five write a column, the sixth the 8 bytes left over
    const uint32_t L = stage_lines(S), rows = 6u * (S + 1);
    const uint32_t l = blockIdx.x * 32u + threadIdx.x / 8u, k = threadIdx.x % 8u, r = blockIdx.y + gridDim.y * blockIdx.z;
    if (l >= L || r >= rows || k > 5u) return;
    float2* out = lines + ((size_t)r * L + l) * 16 + 3 * k;
    if (k == 5u) {
        *out = make_float2(0.0f, 0.0f);
        return;
    }
    const uint32_t f = r / (S + 1);
    const int Si = (int)S, i = (int)(4u * l + k) - 1, j = (int)(r - f * (S + 1)) - 1;
    f3 a, b;
    if (i > Si) {  // past the last footprint's second column: never read
        a = b = make3(0.0f, 0.0f, 0.0f);
    } else if (i >= 0 && i < Si && j >= 0 && j + 1 < Si) {
        const float4 p = cube[((size_t)f * S + j) * S + i], q = cube[((size_t)f * S + j + 1) * S + i];
        a = {p.x, p.y, p.z};
        b = {q.x, q.y, q.z};
    } else {
        a = cube_texel_seamless(cube, Si, (int)f, i, j);
        b = cube_texel_seamless(cube, Si, (int)f, i, j + 1);
    }
    out[0] = make_float2(a.x, a.y);
    out[1] = make_float2(a.z, b.x);
    out[2] = make_float2(b.y, b.z);
}

// One lane's sample of one round: direction, theta terms, taps and loads
// (gathered: q[k] = tap k's texel; staged: q[0..2] = the footprint's entry).
struct DiffSample {
    f3 L;
    float ct, st;
    CubeTaps taps;
    float4 q[4];
};

// STAGED: the samples read staged footprints (48 bytes of one line, aligned to
// 8); otherwise their four taps from the cube. Four lanes loading one footprint
// together (16 lines per load instruction instead of 64, the parts passed on
// through LDS) measured slower while each had an entry of 64 bytes: 2.36 ms
// against 1.82.
template <int TEX, int THREADS, bool STAGED>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(HVX_DIFFUSE_WAVES_PER_EU, 8))) void
diffuse_kernel(const float4* __restrict__ cube, uint32_t S, const float* __restrict__ stage, float4* __restrict__ out,
               uint32_t Sd) {
    constexpr uint32_t SLOT = THREADS / TEX;  // samples per texel per round
    __shared__ float s_phi[kMaxPhi], s_theta[kMaxTheta];
    __shared__ float s_sp[kMaxPhi], s_cp[kMaxPhi], s_st[kMaxTheta], s_ct[kMaxTheta];
    __shared__ float s_buf[2][SLOT][TEX][3];
    __shared__ uint32_t s_np, s_nt;
    const float TWO_PI = kPiF * 2.0f, HALF_PI = kPiF * 0.5f;
    const float delta = 0.025f;
    const uint32_t l = threadIdx.x;
    if (l == 0) {
        uint32_t np = 0;
        for (float phi = 0.0f; phi < TWO_PI && np < (uint32_t)kMaxPhi; phi = phi + delta) s_phi[np++] = phi;
        uint32_t nt = 0;
        for (float th = 0.0f; th < HALF_PI && nt < (uint32_t)kMaxTheta; th = th + delta) s_theta[nt++] = th;
        s_np = np;
        s_nt = nt;
    }
    __syncthreads();
    const uint32_t np = s_np, nt = s_nt, total = np * nt;
    for (uint32_t i = l; i < np; i += blockDim.x) {
        s_sp[i] = sinf_(s_phi[i]);
        s_cp[i] = cosf_(s_phi[i]);
    }
    for (uint32_t i = l; i < nt; i += blockDim.x) {
        s_st[i] = sinf_(s_theta[i]);
        s_ct[i] = cosf_(s_theta[i]);
    }
    __syncthreads();
    const uint32_t ntex = 6u * Sd * Sd;
    // sample lane: texel l % TEX, slot l / TEX
    const uint32_t ti = l % TEX, slot = l / TEX;
    const uint32_t texel = min(blockIdx.x * TEX + ti, ntex - 1);
    const uint32_t x = texel % Sd, y = (texel / Sd) % Sd, face = texel / (Sd * Sd);
    const f3 N = texel_dir((int)face, (int)x, (int)y, (int)Sd);
    f3 up = make3(0.0f, 1.0f, 0.0f);
    const f3 right = normalize3(cross3(up, N));
    up = normalize3(cross3(N, right));
    // summer lane: l < 3 * TEX -> texel l / 3, channel l % 3
    const bool summer = l < 3u * TEX;
    const uint32_t st_i = l / 3, st_c = l % 3;
    float acc = 0.0f;
    const uint32_t rounds = (total + SLOT - 1) / SLOT;
    // sample r * SLOT + slot; slots past the last sample evaluate the last
    // one again (in range, never summed), so the loads stay unconditional
    auto begin = [&](DiffSample& p, uint32_t r) {
        const uint32_t sidx = min(r * SLOT + slot, total - 1);
        const uint32_t ip = sidx / nt, it = sidx % nt;
        const float sp = s_sp[ip], cp = s_cp[ip];
        p.st = s_st[it];
        p.ct = s_ct[it];
        const float tx = p.st * cp, ty = p.st * sp, tz = p.ct;
        p.L = add3(add3(mul3(right, tx), mul3(up, ty)), mul3(N, tz));
        p.taps = cube_taps<true>((int)S, p.L);
        if constexpr (STAGED) {
            // i0, j0 lie in [-1, S - 1] (the face coordinates are in [0, 1]);
            // the clamp only keeps the index inside the table
            const int i0 = min(max(p.taps.i0, -1), (int)S - 1), j0 = min(max(p.taps.j0, -1), (int)S - 1);
            const uint32_t r = (uint32_t)p.taps.face * (S + 1) + (uint32_t)(j0 + 1), e = (uint32_t)(i0 + 1);
            // 24-byte steps: loads aligned to 8
            const float* q = stage + ((size_t)r * stage_lines(S) + e / 4u) * 32 + 6u * (e % 4u);
            __builtin_memcpy(p.q, q, 48);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) p.q[k] = cube[p.taps.idx[k]];
        }
    };
    // weight round r's sample, store it, and (summers) add the round's terms
    // in sample order; every lane of the workgroup calls it for every r
    auto sum_round = [&](uint32_t r, const DiffSample& p) {
        float (*buf)[TEX][3] = s_buf[r & 1];
        f3 c;
        if constexpr (STAGED) {
            // sample_cube's bilinear sum of the entry's taps
            const float4 q0 = p.q[0], q1 = p.q[1], q2 = p.q[2];
            const CubeTaps& t = p.taps;
            c = {((t.w00 * q0.x + t.w10 * q1.z) + t.w01 * q0.w) + t.w11 * q2.y,
                 ((t.w00 * q0.y + t.w10 * q1.w) + t.w01 * q1.x) + t.w11 * q2.z,
                 ((t.w00 * q0.z + t.w10 * q2.x) + t.w01 * q1.y) + t.w11 * q2.w};
        } else {
            c = cube_combine(cube, (int)S, p.L, p.taps, p.q);
        }
        buf[slot][ti][0] = (c.x * p.ct) * p.st;
        buf[slot][ti][1] = (c.y * p.ct) * p.st;
        buf[slot][ti][2] = (c.z * p.ct) * p.st;
        __syncthreads();
        if (summer && r < rounds) {
            const uint32_t kmax = min(SLOT, total - r * SLOT);
            for (uint32_t k = 0; k < kmax; ++k) acc = acc + buf[k][st_i][st_c];
        }
    };
    DiffSample A, B;
    begin(A, 0);
    for (uint32_t r = 0; r < rounds; r += 2) {
        begin(B, r + 1);
        sum_round(r, A);
        begin(A, r + 2);
        sum_round(r + 1, B);
    }
    if (summer) {
        const uint32_t t = blockIdx.x * TEX + st_i;
        if (t < ntex) {
            const float inv = 1.0f / (float)total;
            reinterpret_cast<float*>(out + t)[st_c] = (kPiF * acc) * inv;
            if (st_c == 0) reinterpret_cast<float*>(out + t)[3] = 1.0f;
        }
    }
}

// ---------------------------------------------------------------- specular
__global__ __launch_bounds__(256) void ggx_table_kernel(uint32_t mips, uint32_t n, float4* __restrict__ table) {
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= mips * n) return;
    const uint32_t m = id / n, i = id % n;
    // PipelineCubeFilter.cpp:305-311: roughness = float(i) / float(mips - 1)
    const float rough = mips <= 1 ? 0.0f : (float)m / (float)(mips - 1);
    table[id] = ggx_tangent_sample(i, n, rough);
}

constexpr int kMaxMips = 16;
constexpr uint32_t kRepeatSamples = 430;  // samples up to which their equal terms are added one by one

// One output texel of the GGX prefilter (CubeFilterSpecular.frag:34-75) at
// direction-grid position (face, x, y) of a D x D viewport; `tab` holds the
// mip's n tangent-space samples; rough0 marks the roughness-0 mip.
__device__ __forceinline__ float4 specular_texel_value(const float4* __restrict__ cube, uint32_t S,
                                                       const float4* __restrict__ tab, uint32_t n, bool rough0,
                                                       int face, int x, int y, int D) {
    const f3 N = texel_dir(face, x, y, D);
    const f3 V = N;
    const Frame fr = ggx_frame(N);
    float acc0 = 0.0f, acc1 = 0.0f, acc2 = 0.0f, wsum = 0.0f;
    if (rough0) {
        // roughness 0 (PipelineCubeFilter.cpp:305-311 gives mip 0 roughness 0):
        // cos(theta) = sqrt((1-y)/(1-y)) = 1 and sin(theta) = 0 for every
        // Hammersley sample, so each sample's half vector is normalize(N + (+-0))
        // and all n samples produce the same L, NoL and texel value. Evaluate it
        // once and form the reference's sequential sums of the n identical terms,
        // one addition after the other, or past kRepeatSamples of them a binade
        // at a time (6 x 512^2 texels: 25 / 41 us with 64 samples, 44 / 57 with 256,
        // 60 / 63 with 400, 71 / 64 with 512, 126 / 71 with 1,024; 6 x 16^2: 7.6 / 9.8,
        // 10.4 / 12.3, 13.3 / 13.4, 15.6 / 13.3, 25.9 / 14.6).
        const f3 Hh = ggx_world(fr, N, tab[0]);
        const f3 L = normalize3(sub3(mul3(Hh, 2.0f * dot3(V, Hh)), V));
        const float NoL = gmax(dot3(N, L), 0.0f);
        if (NoL > 0.0f) {
            const f3 c = sample_cube(cube, (int)S, L);
            const float t0 = c.x * NoL, t1 = c.y * NoL, t2 = c.z * NoL;
            if (n <= kRepeatSamples) {
                for (uint32_t i = 0; i < n; ++i) {
                    acc0 = acc0 + t0;
                    acc1 = acc1 + t1;
                    acc2 = acc2 + t2;
                    wsum = wsum + NoL;
                }
            } else {
                acc0 = repeat_sum(t0, n);
                acc1 = repeat_sum(t1, n);
                acc2 = repeat_sum(t2, n);
                wsum = repeat_sum(NoL, n);
            }
        }
    } else {
        for (uint32_t i = 0; i < n; ++i) {
            const f3 Hh = ggx_world(fr, N, tab[i]);
            const f3 L = normalize3(sub3(mul3(Hh, 2.0f * dot3(V, Hh)), V));
            const float NoL = gmax(dot3(N, L), 0.0f);
            if (NoL > 0.0f) {
                const f3 c = sample_cube(cube, (int)S, L);
                acc0 = acc0 + c.x * NoL;
                acc1 = acc1 + c.y * NoL;
                acc2 = acc2 + c.z * NoL;
                wsum = wsum + NoL;
            }
        }
    }
    return make_float4(acc0 / wsum, acc1 / wsum, acc2 / wsum, 1.0f);
}

// Mip 0 has roughness 0 (PipelineCubeFilter.cpp:305-311): one lane per texel.
__global__ __launch_bounds__(256) void specular_delta_kernel(const float4* __restrict__ cube, uint32_t S,
                                                             float4* __restrict__ out, uint32_t So,
                                                             const float4* __restrict__ table, uint32_t n) {
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= 6u * So * So) return;
    const uint32_t x = id % So, y = (id / So) % So, face = id / (So * So);
    out[id] = specular_texel_value(cube, S, table, n, true, (int)face, (int)x, (int)y, (int)So);
}

// Mips of roughness > 0, samples spread over lanes. A wave owns kSpecTPW
// texels of a tile and evaluates kSpecSPR = 64 / kSpecTPW consecutive
// samples of each per round; every lane writes its sample's four terms
// (c * NoL, NoL; -0 for a rejected sample, the exact identity of x + y) to
// LDS, and one "summer" lane per texel and term adds that round's terms in
// sample order, so every sum is the reference's sequential sum (bit-exact).
// Few texels per wave keep the texels in flight per XCD few, so the GGX lobes
// being read at any time share the XCD's L2: tiles are taken in 16x16-tile
// supertiles, and XCD x (workgroups b with b % 8 = x) gets run x of every
// mip's tiles.
// What bounds it (512^2 x 10 from 1024^2, 1024 samples): the texture
// addresser, at about a lane per cycle for gathers of lanes in different lines,
// then VALU issue (236 instructions per 64 samples). So the two lanes of a pair
// load the two texels of a footprint row together, one sample of the pair per
// load (pair_exchange): lanes side by side in one line are one access.
//   one run of all mips' tiles per XCD                   7.43 ms
//   (two XCDs held the tiles of mip 2, which cost about
//   twice those of mip 1; six waited for them)
//   a run of every mip per XCD                           4.33 ms
//   lengths from bit patterns, faces by selects          4.33 ms (still the addresser)
//   footprint rows loaded by lane pairs                  3.78 ms (addresser 88 -> 70 % busy)
//   no length checks, 32-bit offsets                     3.71 ms (VALU 81 % busy)
//   roughness 0 summed by binades                        3.60 ms
//   pairs exchanged by selects that read across lanes    3.53 ms
struct SpecSplitArgs {
    const float4* cube;
    uint32_t S;
    float4* out;
    uint32_t So, mips, n, emulate;
    uint32_t run_begin[kMaxMips + 1];  // first workgroup of mip m (mips 1..) in an XCD's sequence, run_begin[1] = 0
    const float4* table;
};

// One GGX sample of the specular loop, split so its texel loads overlap other
// work: spec_begin forms L and NoL and issues the four tap loads of the pair's
// samples (always, so the loads are not under a branch; a rejected sample's
// taps are valid texels whose values are not used), spec_term forms the
// sample's terms.
struct SpecSample {
    f3 L;
    float nol;
    CubeTaps taps;
    f3 q[4];  // [2 r + s]: row r, column (lane & 1) of the footprint of the pair's sample s
};

// Exchanges between the lanes of a pair (2k, 2k + 1): a = (even lane: its x,
// odd lane: the even lane's y), b = (even lane: the odd lane's x, odd lane: its
// y), three values at a time. Each is one select that reads one operand through
// the lane crossing; the compiler writes the crossing and the select as two
// instructions each (it forms the crossing select only for a condition that is
// already in vcc). The leading no-op is the two wait states between a vector
// write of an operand and its reading across lanes.
__device__ __forceinline__ void pair_exchange(const float (&x)[3], const float (&y)[3], float (&a)[3], float (&b)[3]) {
    __asm__ volatile("s_nop 1\n\t"
            "s_mov_b32 vcc_lo, 0x55555555\n\t"
            "s_mov_b32 vcc_hi, 0x55555555\n\t"
            "v_cndmask_b32_dpp %0, %9, %6, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %1, %10, %7, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %2, %11, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_not_b64 vcc, vcc\n\t"
            "v_cndmask_b32_dpp %3, %6, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %4, %7, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %5, %8, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
            : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2])
            : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(y[0]), "v"(y[1]), "v"(y[2])
            : "vcc", "scc");
}
// The same for two pairs of texel indices.
__device__ __forceinline__ void pair_exchange(const int (&x)[2], const int (&y)[2], int (&a)[2], int (&b)[2]) {
    __asm__ volatile("s_nop 1\n\t"
            "s_mov_b32 vcc_lo, 0x55555555\n\t"
            "s_mov_b32 vcc_hi, 0x55555555\n\t"
            "v_cndmask_b32_dpp %0, %6, %4, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %1, %7, %5, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_not_b64 vcc, vcc\n\t"
            "v_cndmask_b32_dpp %2, %4, %6, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %3, %5, %7, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
            : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0]), "=&v"(b[1])
            : "v"(x[0]), "v"(x[1]), "v"(y[0]), "v"(y[1])
            : "vcc", "scc");
}

// Texel i of a cube level. WIDE false: the level is smaller than 4 GiB (faces up
// to kNarrowFace), so a 32-bit byte offset from the uniform base will do.
template <bool WIDE>
__device__ __forceinline__ float4 cube_at(const float4* __restrict__ cube, int i) {
    if constexpr (WIDE) return cube[i];
    else return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(cube) + ((uint32_t)i << 4));
}

template <bool WIDE>
__device__ __forceinline__ void spec_begin(SpecSample& p, const float4* __restrict__ cube, int S, const Frame& fr,
                                           f3 N, float4 h) {
    // both vectors are unit length up to rounding
    const f3 Hh = normalize3_unit(add3(add3(mul3(fr.t, h.x), mul3(fr.b, h.y)), mul3(N, h.z)));  // ggx_world
    p.L = normalize3_unit(sub3(mul3(Hh, 2.0f * dot3(N, Hh)), N));                              // V = N
    p.nol = gmax(dot3(N, p.L), 0.0f);
    p.taps = cube_taps<true>(S, p.L);
    // the first load takes the even lane's sample (even lane texel 0, odd lane
    // texel 1 of the row), the second the odd lane's
    const int (&id)[4] = p.taps.idx;
    const int t0[2] = {id[0], id[2]}, t1[2] = {id[1], id[3]};
    int first[2], second[2];
    pair_exchange(t0, t1, first, second);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float4 v0 = cube_at<WIDE>(cube, first[r]), v1 = cube_at<WIDE>(cube, second[r]);
        p.q[2 * r] = {v0.x, v0.y, v0.z};
        p.q[2 * r + 1] = {v1.x, v1.y, v1.z};
    }
}

// (c * NoL, NoL) of a sample that counts (NoL > 0); -0 in every term of one
// that does not (a rejected or padding sample): x + (-0) == x for every x.
__device__ __forceinline__ float4 spec_term(const SpecSample& p, bool live, const float4* __restrict__ cube, int S) {
    float4 q[4];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const f3 &u = p.q[2 * r], &v = p.q[2 * r + 1];
        const float x[3] = {u.x, u.y, u.z}, y[3] = {v.x, v.y, v.z};
        float t0[3], t1[3];
        pair_exchange(x, y, t0, t1);
        q[2 * r] = make_float4(t0[0], t0[1], t0[2], 0.0f);
        q[2 * r + 1] = make_float4(t1[0], t1[1], t1[2], 0.0f);
    }
    if (!(live && p.nol > 0.0f)) return make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
    const f3 c = cube_combine(cube, S, p.L, p.taps, q);
    return make_float4(c.x * p.nol, c.y * p.nol, c.z * p.nol, p.nol);
}

// One tile of the sample-split specular loop (four waves, each independent):
// texels of face `face` of a mip of size Sm whose directions lie on a D x D
// grid, out_level that mip's texels, tab its n tangent-space samples, s_buf
// the workgroup's [4][2][TPW][kRow] summation buffer.
template <bool WIDE, int TPW>
__device__ __forceinline__ void specular_split_tile(const float4* __restrict__ cube, int S,
                                                    float4* __restrict__ out_level, uint32_t Sm, uint32_t D,
                                                    const float4* __restrict__ tab, uint32_t n, uint32_t face,
                                                    uint32_t tx, uint32_t ty, float* s_buf) {
    using Sh = SpecShape<TPW>;
    constexpr int kSPR = Sh::kSPR, kTW = Sh::kTW, kRPW = Sh::kRPW, kTH = Sh::kTH, kRow = Sh::kRow;
    const uint32_t wave = threadIdx.x / 64u, lane = threadIdx.x % 64u;
    // evaluating lane: texel t of the wave, sample slot s
    const uint32_t t = lane / kSPR, s = lane % kSPR;
    const uint32_t x = min(tx * kTW + t % kTW, Sm - 1),
                   y = min(ty * kTH + wave * kRPW + t / kTW, Sm - 1);
    const f3 N = texel_dir((int)face, (int)x, (int)y, (int)D);
    const Frame fr = ggx_frame(N);
    // summing lane: texel st of the wave, term sc (R, G, B, NoL)
    const bool summer = lane < 4u * TPW;
    const uint32_t st = lane / 4u, sc = lane % 4u;
    float acc = 0.0f;
    constexpr uint32_t kHalf = (uint32_t)TPW * kRow;  // floats between the two buffers
    float* const wbuf = s_buf + wave * 2u * kHalf + t * kRow + 4u * s;
    const float* const rbuf = s_buf + wave * 2u * kHalf + st * kRow + sc;
    // rounds in pairs (A: even, B: odd); sample i of round r is r * SPR + s,
    // table entries are fetched two rounds ahead and tap loads one round
    // ahead of their use
    const uint32_t rounds = (n + kSPR - 1) / kSPR;
    auto tab_at = [&](uint32_t r) { return tab[min(r * kSPR + s, n - 1)]; };
    auto sum_round = [&](uint32_t parity, float4 term) {
        *reinterpret_cast<float4*>(wbuf + parity * kHalf) = term;
        wave_lds_sync();
        if (summer) {
#pragma unroll
            for (int q = 0; q < kSPR; ++q) acc = acc + rbuf[parity * kHalf + 4 * q];
        }
    };
    SpecSample A, B;
    float4 hA = tab_at(0), hB = tab_at(1);
    spec_begin<WIDE>(A, cube, S, fr, N, hA);
    hA = tab_at(2);
    for (uint32_t r = 0; r < rounds; r += 2) {
        spec_begin<WIDE>(B, cube, S, fr, N, hB);
        hB = tab_at(r + 3);
        sum_round(0, spec_term(A, r * kSPR + s < n, cube, S));
        spec_begin<WIDE>(A, cube, S, fr, N, hA);
        hA = tab_at(r + 4);
        sum_round(1, spec_term(B, (r + 1) * kSPR + s < n, cube, S));
    }
    const float wsum = __shfl(acc, (int)((lane & ~3u) | 3u));
    const uint32_t xs = tx * kTW + st % kTW, ys = ty * kTH + wave * kRPW + st / kTW;
    if (summer && xs < Sm && ys < Sm) {
        float* o = reinterpret_cast<float*>(out_level + (face * Sm + ys) * Sm + xs);
        o[sc] = sc == 3u ? 1.0f : acc / wsum;
    }
    // the next tile of this workgroup reuses the buffers: keep its first
    // writes after these reads
    wave_lds_sync();
}

#ifndef HVX_SPEC_WAVES_PER_EU
#define HVX_SPEC_WAVES_PER_EU 4
#endif
template <bool WIDE, int TPW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HVX_SPEC_WAVES_PER_EU, 8))) void
specular_split_kernel(SpecSplitArgs a) {
    __shared__ __align__(16) float s_buf[4][2][TPW][SpecShape<TPW>::kRow];
    // XCD x (workgroups b with b % 8 = x) works through run x of every mip's
    // tiles in turn: a mip's tiles cost about the same, but those of different
    // mips up to several times each other (wider lobes miss the L2 more)
    const uint32_t x = blockIdx.x % 8u, k = blockIdx.x / 8u;
    uint32_t m = 1;
    while (k >= a.run_begin[m + 1]) ++m;
    const uint32_t Sm = max(a.So >> m, 1u);
    const SpecTileGeom g = spec_tile_geom<TPW>(Sm);
    const uint32_t tile = x * (a.run_begin[m + 1] - a.run_begin[m]) + k - a.run_begin[m];
    if (tile >= 6u * g.per_face) return;  // the last run may be short
    uint32_t face, tx, ty;
    spec_tile_at(g, tile, face, tx, ty);
    specular_split_tile<WIDE, TPW>(a.cube, (int)a.S, a.out + cube_level_offset_floats(a.So, m) / 4, Sm, a.emulate ? a.So : Sm,
                        a.table + (size_t)m * a.n, a.n, face, tx, ty, &s_buf[0][0][0][0]);
}

// ------------------------------------------------- batched probe prefilter
// Persistent: the workgroups on XCD x (workgroup b runs on XCD b % 8) pull
// items from queue x, which serves the run [xcd_begin[x], xcd_begin[x+1]) of
// the item list (make_probe_items: XCD x's share of every mip of every probe).
// Items of mip 0 are texel ranges (lane per texel, as specular_delta_kernel);
// other items are runs of tiles (specular_split_tile).
template <bool WIDE, int TPW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HVX_SPEC_WAVES_PER_EU, 8))) void
probe_batch_kernel(const ProbeJob* __restrict__ jobs, const ProbeItem* __restrict__ items,
                   const uint32_t* __restrict__ xcd_begin, const float4* __restrict__ tables,
                   uint32_t* __restrict__ queues) {
    __shared__ __align__(16) float s_buf[4][2][TPW][SpecShape<TPW>::kRow];
    __shared__ uint32_t s_item;
    const uint32_t x = blockIdx.x % 8u;
    const uint32_t begin = xcd_begin[x], end = xcd_begin[x + 1];
    for (;;) {
        if (threadIdx.x == 0) s_item = begin + atomicAdd(queues + x, 1u);
        __syncthreads();
        const uint32_t item = s_item;
        __syncthreads();
        if (item >= end) break;
        const ProbeItem it = items[item];
        const ProbeJob& j = jobs[it.probe];
        const uint32_t m = it.mip;
        const uint32_t Sm = max(j.So >> m, 1u);
        const float4* tab = tables + j.table + (size_t)m * j.n;
        float4* out = j.out + cube_level_offset_floats(j.So, m) / 4;
        if (m == 0) {
            for (uint32_t t = threadIdx.x; t < it.count; t += blockDim.x) {
                const uint32_t local = it.first + t;
                const uint32_t tx = local % Sm, ty = (local / Sm) % Sm, face = local / (Sm * Sm);
                out[local] = specular_texel_value(j.cube, j.S, tab, j.n, true, (int)face, (int)tx, (int)ty, (int)Sm);
            }
        } else {
            const SpecTileGeom g = spec_tile_geom<TPW>(Sm);
            for (uint32_t k = it.first; k < it.first + it.count; ++k) {
                uint32_t face, tx, ty;
                spec_tile_at(g, k, face, tx, ty);
                specular_split_tile<WIDE, TPW>(j.cube, (int)j.S, out, Sm, Sm, tab, j.n, face, tx, ty, &s_buf[0][0][0][0]);
            }
        }
    }
}

}  // namespace

// ================================================================ launchers
hipError_t launch_brdf_lut(uint32_t w, uint32_t h, uint32_t n, float* d_lut, hipStream_t s) {
    // one texel per lane up to 256 lanes (rounded to whole waves), then two:
    // 512^2 takes the same time either way (429 and 430 us)
    const bool one = w <= 256, fast = n <= (1u << 20);
    const uint32_t lanes = (one ? w : (w + 1) / 2), threads = (lanes + 63) / 64 * 64;  // w <= 1024
    float2* lut = reinterpret_cast<float2*>(d_lut);
    const auto kernel = fast ? (one ? brdf_lut_kernel<1, true> : brdf_lut_kernel<2, true>)
                             : (one ? brdf_lut_kernel<1, false> : brdf_lut_kernel<2, false>);
    hipLaunchKernelGGL(kernel, dim3(h), dim3(threads), 0, s, w, h, n, lut);
    return hipGetLastError();
}

hipError_t launch_equirect_to_cube(const float* d_eq, uint32_t w, uint32_t h, float* d_cube, uint32_t S,
                                   hipStream_t s) {
    hipLaunchKernelGGL(equirect_kernel, dim3((S + 63) / 64, (S + 3) / 4, 6), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(d_eq), w, h, reinterpret_cast<float4*>(d_cube), S);
    return hipGetLastError();
}

hipError_t launch_cube_mips(float* d_chain, uint32_t S, uint32_t levels, hipStream_t s, uint32_t n,
                            size_t chain_stride_floats) {
    for (uint32_t m = 0; m + 1 < levels;) {  // levels m + 1 .. m + a.levels from level m
        MipArgs a{};
        a.sp = S >> m;
        a.pstride = chain_stride_floats / 4;
        a.src = reinterpret_cast<const float4*>(d_chain + cube_level_offset_floats(S, m));
        while (a.levels < kMipLevels && m + a.levels + 1 < levels) {
            a.dst[a.levels] = reinterpret_cast<float4*>(d_chain + cube_level_offset_floats(S, m + a.levels + 1));
            ++a.levels;
        }
        const uint32_t per = a.sp / std::min(a.sp, 32u);
        hipLaunchKernelGGL(mip_kernel, dim3(6 * per * per, n), dim3(256), 0, s, a);
        m += a.levels;
    }
    return hipGetLastError();
}

// dst + p * dst_stride <- src[p], `count` float4s, for p < n (grid dimension y)
__global__ __launch_bounds__(256) void gather_copy_kernel(const float4* const* __restrict__ src, size_t count,
                                                          float4* __restrict__ dst, size_t dst_stride) {
    const float4* from = src[blockIdx.y];
    float4* to = dst + blockIdx.y * dst_stride;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256) to[i] = from[i];
}

hipError_t launch_gather_copy(const float* const* d_src, size_t floats, float* d_dst, size_t dst_stride_floats,
                              uint32_t n, hipStream_t s) {
    const size_t count = floats / 4;
    const uint32_t blocks = (uint32_t)std::min<size_t>((count + 255) / 256, 1024);
    hipLaunchKernelGGL(gather_copy_kernel, dim3(std::max(blocks, 1u), n), dim3(256), 0, s,
                       reinterpret_cast<const float4* const*>(d_src), count, reinterpret_cast<float4*>(d_dst),
                       dst_stride_floats / 4);
    return hipGetLastError();
}

size_t diffuse_stage_size(uint32_t S) {
    const size_t b = (size_t)6 * (S + 1) * stage_lines(S) * 128;
    return b <= kDiffuseStageMaxBytes ? b : 0;
}

hipError_t launch_diffuse(const float* d_cube, uint32_t S, float* d_out, uint32_t Sd, float* d_stage, hipStream_t s) {
    const float4* cube = reinterpret_cast<const float4*>(d_cube);
    float* stage = diffuse_stage_size(S) ? d_stage : nullptr;
    const uint32_t T = 6u * Sd * Sd;
    float4* out = reinterpret_cast<float4*>(d_out);
    if (stage) {
        const uint32_t rows = 6u * (S + 1), gy = std::min(rows, 32768u);
        hipLaunchKernelGGL(diffuse_stage_kernel, dim3((stage_lines(S) + 31) / 32, gy, (rows + gy - 1) / gy), dim3(256), 0,
                           s, cube, S, reinterpret_cast<float2*>(stage));
        // few texels: fewer to a workgroup, for more workgroups and fewer
        // rounds, as long as they are all in flight (eight per CU) and, past
        // 640, the face is small for the texels; large faces of medium maps
        // stay with the fabric's best
        auto run = [&](auto tex) {
            constexpr int kTex = decltype(tex)::value;
            hipLaunchKernelGGL((diffuse_kernel<kTex, kDThreads, true>), dim3((T + kTex - 1) / kTex), dim3(kDThreads), 0,
                               s, cube, S, stage, out, Sd);
        };
        if (T <= 640 || (T <= 2048 && T * S <= (1u << 18))) run(std::integral_constant<int, 1>());
        else if (T <= 4096 && S <= 512) run(std::integral_constant<int, 2>());
        else run(std::integral_constant<int, kDTex>());
    } else {
        hipLaunchKernelGGL((diffuse_kernel<kDTex, kDThreads, false>), dim3((T + kDTex - 1) / kDTex), dim3(kDThreads),
                           0, s, cube, S, nullptr, out, Sd);
    }
    return hipGetLastError();
}

hipError_t launch_specular(const float* d_cube, uint32_t S, float* d_out, uint32_t So, uint32_t mips, uint32_t n,
                           bool emulate_static_viewport, float4* ggx_table, hipStream_t s) {
    if (mips > (uint32_t)kMaxMips) return hipErrorInvalidValue;
    hipLaunchKernelGGL(ggx_table_kernel, dim3((mips * n + 255) / 256), dim3(256), 0, s, mips, n, ggx_table);
    const float4* cube = reinterpret_cast<const float4*>(d_cube);
    float4* out = reinterpret_cast<float4*>(d_out);
    // mip 0 (roughness 0) covers its whole face whether or not the viewport
    // is emulated: its size is the base size
    hipLaunchKernelGGL(specular_delta_kernel, dim3((6u * So * So + 255) / 256), dim3(256), 0, s, cube, S, out, So,
                       ggx_table, n);
    if (mips > 1) {
        SpecSplitArgs a{};
        a.cube = cube;
        a.S = S;
        a.out = out;
        a.So = So;
        a.mips = mips;
        a.n = n;
        a.emulate = emulate_static_viewport ? 1u : 0u;
        a.table = ggx_table;
        auto run = [&](auto wide, auto tpw) {
            constexpr int kTPW = decltype(tpw)::value;
            uint32_t t = 0;
            for (uint32_t m = 1; m <= (uint32_t)kMaxMips; ++m) {
                a.run_begin[m] = t;
                if (m < mips) t += (6u * spec_tile_geom<kTPW>(std::max(So >> m, 1u)).per_face + 7) / 8;
            }
            hipLaunchKernelGGL((specular_split_kernel<decltype(wide)::value, kTPW>), dim3(t * 8), dim3(256), 0, s, a);
        };
        uint32_t tiles = 0;
        for (uint32_t m = 1; m < mips && tiles <= kSpecFewTiles; ++m)
            tiles += 6u * spec_tile_geom<kSpecTPW>(std::max(So >> m, 1u)).per_face;
        const std::integral_constant<int, kSpecTPW> many;
        const std::integral_constant<int, 1> one;
        const bool few = spec_few(tiles, n);
        if (S > kNarrowFace) few ? run(std::true_type(), one) : run(std::true_type(), many);
        else few ? run(std::false_type(), one) : run(std::false_type(), many);
    }
    return hipGetLastError();
}

hipError_t launch_ggx_tables(uint32_t mips, uint32_t n, float4* table, hipStream_t s) {
    hipLaunchKernelGGL(ggx_table_kernel, dim3((mips * n + 255) / 256), dim3(256), 0, s, mips, n, table);
    return hipGetLastError();
}

hipError_t launch_probe_batch(const ProbeJob* d_jobs, const ProbeItem* d_items, const uint32_t* d_xcd_begin,
                              const float4* d_tables, uint32_t persistent_wgs, bool wide, bool one, uint32_t* d_queues,
                              hipStream_t s) {
    const uint32_t grid = std::max((persistent_wgs + 7) / 8, 1u) * 8;  // every XCD gets workgroups
    const auto kernel = wide ? (one ? probe_batch_kernel<true, 1> : probe_batch_kernel<true, kSpecTPW>)
                             : (one ? probe_batch_kernel<false, 1> : probe_batch_kernel<false, kSpecTPW>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, s, d_jobs, d_items, d_xcd_begin, d_tables, d_queues);
    return hipGetLastError();
}

}  // namespace hvx
