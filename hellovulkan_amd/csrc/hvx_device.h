// hvx_device.h — device-side vector algebra and software texture sampling.
//
// The evaluation order of every expression is fixed and matches the scalar
// definitions the path is specified by: dot(a,b) = (ax*bx + ay*by) + az*bz;
// mat*vec row r = ((m[0][r]*x + m[1][r]*y) + m[2][r]*z) + m[3][r]*w;
// normalize(v) = v * (1 / sqrt(dot(v, v))). All translation units that include
// this header are compiled with -ffp-contract=off, so nothing is fused unless a
// kernel asks for it explicitly.
//
// Texture sampling follows the Vulkan specification's texel filtering:
// LINEAR filter (u = s*W - 1/2, i0 = floor(u), alpha = frac(u)), REPEAT wrap
// for 2D images, cube face selection by major axis (ties X > Y > Z) and
// seamless cube edges (the texel across an edge is found by folding the face
// plane over the edge; a corner texel is the mean of its three neighbours).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hvx_math.h"

namespace hvx {

struct f3 {
    float x, y, z;
};

__device__ __forceinline__ f3 make3(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ f3 add3(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 sub3(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 mul3(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ float dot3(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ f3 cross3(f3 a, f3 b) {
    return {a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y};
}
__device__ __forceinline__ float length3(f3 a) { return sqrtf_(dot3(a, a)); }
__device__ __forceinline__ f3 normalize3(f3 a) {
    const float inv = 1.0f / sqrtf_(dot3(a, a));
    return mul3(a, inv);
}

// column-major 4x4 times (x, y, z, w)
__device__ __forceinline__ void matvec4(const float* m, float x, float y, float z, float w, float o[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        o[r] = ((m[r] * x + m[4 + r] * y) + m[8 + r] * z) + m[12 + r] * w;
    }
}

// ------------------------------------------- correctly rounded fast paths
// Correctly rounded square root of x in [2^-102, FLT_MAX]: Markstein's
// iteration from the hardware reciprocal square root y ~ 1/sqrt(x):
// s0 = rn(x y), then one correction s0 + (x - s0^2) (y/2) with the residual
// fused, so it is exact. Five operations where correcting the hardware square
// root by both neighbours' residuals takes nine. Verified equal to sqrtf on
// every float of [2^-102, 2^128) on gfx950 (tests/test_gpu_fastmath.py);
// below 2^-102 the residual is subnormal and the result can be an ulp off.
__device__ __forceinline__ float sqrt_rn_normal(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float s0 = x * y;
    const float r = __builtin_fmaf(-s0, s0, x);
    return __builtin_fmaf(r, 0.5f * y, s0);
}

// Correctly rounded reciprocal of a normal b with |b| in [2^-125, 2^125]:
// hardware estimate (within 1 ulp) plus one Newton-Raphson correction with
// fused multiply-add, y' = y + y (1 - b y): the fused residual is rounded
// once, so y' carries only an O(ulp^2) error before its single rounding.
// Verified equal to 1.0f / b on every float b with |b| in [2^-125, 2^125)
// on gfx950 (tests/test_gpu_fastmath.py).
__device__ __forceinline__ float rcp_rn_normal(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    const float e = __builtin_fmaf(-b, y, 1.0f);
    return __builtin_fmaf(e, y, y);
}

// 1.0f / sqrtf(q) (both correctly rounded) of a squared length q within 2048
// floats of 1, from its bit pattern alone. With q = 1 + d 2^-23, d >= 0, the
// square root 1 + d/2 2^-23 - O(d^2) 2^-46 rounds to 1 + floor(d/2) 2^-23 (a
// tie is broken downwards by the small term), whose reciprocal rounds to
// 1 - floor(d/2) 2^-23, twice as many of the floats below 1; with q = 1 +
// d 2^-24, d < 0, the root rounds to 1 - ceil(-d/2) 2^-24 and the reciprocal
// to 1 + ceil(ceil(-d/2)/2) 2^-23. Holds for -8190 <= d <= 2897 (every float
// checked, tests/test_gpu_unit_length.py). Eight integer operations for the 13 and
// two transcendental ones of rcp_rn_normal(sqrt_rn_normal(q)), to which other
// values fall back.
__host__ __device__ __forceinline__ uint32_t inv_unit_length_bits(int d) {
    const int one = 0x3f800000;
    return (uint32_t)(d >= 0 ? one - (d & ~1) : one + ((3 - d) >> 2));
}
__device__ __forceinline__ float inv_unit_length(float q) {
    const int d = (int)f2u(q) - 0x3f800000;
    if (__builtin_expect((uint32_t)(d + 2048) > 4096u, 0)) return rcp_rn_normal(sqrt_rn_normal(q));
    return u2f(inv_unit_length_bits(d));
}

// a / b correctly rounded where a, b, a / b and the residuals a - b q (down to
// about |a| 2^-24) are normal: the correctly rounded reciprocal, then two
// Newton steps of the quotient with fused residuals. The first leaves q within
// an ulp, and from there the second rounds correctly (Markstein). Without the
// scaling and special cases of the compiler's division.
__device__ __forceinline__ float div_by_normal(float a, float b, float y) {  // y = rcp_rn_normal(b)
    float q = a * y;
    q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float div_rn_normal(float a, float b) { return div_by_normal(a, b, rcp_rn_normal(b)); }

// atan2f_ and acosf_ of hvx_math.h to the bit, for finite arguments (acosf_:
// |x| < 1; others go to hvx_math.h). Those round a double whose error is a few
// of its ulps to float, so any value within 2^-42 of it whose float is the same
// at both ends of that range gives the same result. This one takes a single
// quotient with an unscaled reciprocal, fused Horner steps and no terms below
// 2^-46; about one argument in 10^5 lies too near the middle between two floats
// and takes the functions themselves.
__device__ __forceinline__ double atan2_near(double y, double x) {
    const double ax = __builtin_fabs(x), ay = __builtin_fabs(y);
    const double mn = __builtin_fmin(ax, ay), mx = __builtin_fmax(ax, ay);
    // t = mn / mx, or (t sqrt3 - 1) / (t + sqrt3) past tan(pi / 12)
    const bool far = mn > 0.2679491924311227 * mx;
    const double num = far ? __builtin_fma(mn, kSqrt3, -mx) : mn, den = far ? __builtin_fma(mx, kSqrt3, mn) : mx;
    double r = __builtin_amdgcn_rcp(den);
    r = __builtin_fma(__builtin_fma(-den, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-den, r, 1.0), r, r);
    const double t = num * r, t2 = t * t;
    double p = 1.0 / 21.0;
    p = __builtin_fma(p, t2, -1.0 / 19.0);
    p = __builtin_fma(p, t2, 1.0 / 17.0);
    p = __builtin_fma(p, t2, -1.0 / 15.0);
    p = __builtin_fma(p, t2, 1.0 / 13.0);
    p = __builtin_fma(p, t2, -1.0 / 11.0);
    p = __builtin_fma(p, t2, 1.0 / 9.0);
    p = __builtin_fma(p, t2, -1.0 / 7.0);
    p = __builtin_fma(p, t2, 1.0 / 5.0);
    p = __builtin_fma(p, t2, -1.0 / 3.0);
    double a = (far ? kPio6 : 0.0) + __builtin_fma(t * t2, p, t);
    a = ay > ax ? kPio2 - a : a;
    a = x < 0.0 ? kPiD - a : a;
    return __builtin_copysign(a, y);
}
// a's float if every value within 2^-42 of it has the same
__device__ __forceinline__ bool float_of_near(double a, float& f) {
    f = (float)(a * (1.0 + 0x1p-42));
    return f == (float)(a * (1.0 - 0x1p-42));
}
__device__ __forceinline__ float atan2f_rn(float y, float x) {
    float f;
    if (__builtin_expect(float_of_near(atan2_near((double)y, (double)x), f), 1)) return f;
    return atan2f_(y, x);
}
__device__ __forceinline__ float acosf_rn(float x) {
    // square root of z = (1 - x)(1 + x), at least 2^-24: two Newton steps from the hardware's estimate
    const double z = (1.0 - (double)x) * (1.0 + (double)x), r = __builtin_amdgcn_rsq(z);
    double g = z * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(g, __builtin_fma(-h, g, 0.5), g);
    float f;
    if (__builtin_expect(__builtin_fabsf(x) < 1.0f && float_of_near(atan2_near(g, (double)x), f), 1)) return f;
    return acosf_(x);
}

// normalize3 of a vector whose squared length is a float in [2^-102, FLT_MAX]
// (every near-unit vector): the same correctly rounded square root and
// reciprocal, by the fast paths above, so the result is bit-identical.
__device__ __forceinline__ f3 normalize3_rn(f3 a) { return mul3(a, rcp_rn_normal(sqrt_rn_normal(dot3(a, a)))); }

// normalize3, bit-identical, of a vector whose squared length is known to be
// within 2048 floats of 1 (a combination of an orthonormal frame with unit
// coefficients, a reflection of one unit vector about another: both within a
// few tens of floats).
__device__ __forceinline__ f3 normalize3_unit(f3 a) {
    return mul3(a, u2f(inv_unit_length_bits((int)f2u(dot3(a, a)) - 0x3f800000)));
}

// ------------------------------------------------------------ cube sampling
struct CubeCoord {
    int face;
    float s, t;
};

// Face and plane coordinates of direction r. Selects and sign flips instead of
// a branch per face: the lanes of a wave look all ways. UNIT: r has unit
// length up to rounding, so the divisions by the major component (at least
// 0.57) need no scaling; they share its reciprocal. (A numerator near zero
// whose residual is subnormal vanishes in the sum with 1.)
template <bool UNIT = false>
__device__ __forceinline__ CubeCoord cube_select(f3 r) {
    const float ax = absf(r.x), ay = absf(r.y), az = absf(r.z);
    const bool X = ax >= ay && ax >= az, Y = !X && ay >= az;
    const float ma = X ? ax : (Y ? ay : az);
    const bool neg = !((X ? r.x : (Y ? r.y : r.z)) >= 0.0f);
    const uint32_t flip = neg ? 0x80000000u : 0u;
    // sc: -z, z, x, x, x, -x and tc: -y, -y, z, -z, -y, -y of faces 0 .. 5
    const float sc = u2f(f2u(X ? -r.z : r.x) ^ (Y ? 0u : flip));
    const float tc = u2f(f2u(Y ? r.z : -r.y) ^ (Y ? flip : 0u));
    CubeCoord c;
    c.face = (X ? 0 : (Y ? 2 : 4)) + (neg ? 1 : 0);
    float qs, qt;
    if constexpr (UNIT) {
        const float y = rcp_rn_normal(ma);
        qs = div_by_normal(sc, ma, y);
        qt = div_by_normal(tc, ma, y);
    } else {
        qs = sc / ma;
        qt = tc / ma;
    }
    c.s = 0.5f * (qs + 1.0f);
    c.t = 0.5f * (qt + 1.0f);
    return c;
}

// Folds coordinate c (if |c| > S) onto the plane of the major coordinate mj:
// c -> sign(c) * S, mj -> sign(mj) * (2S - |c|).
__device__ __forceinline__ bool edge_fold(int& c, int& mj, int S) {
    const int ac = c < 0 ? -c : c;
    if (ac <= S) return false;
    mj = mj > 0 ? (2 * S - ac) : -(2 * S - ac);
    c = c > 0 ? S : -S;
    return true;
}

// Texel (face, i, j) with at most one of i, j one step outside [0, S):
// returns the linear texel index of the texel across the edge.
__device__ __forceinline__ int cube_edge_index_inl(int f, int i, int j, int S) {
    const int a = 2 * i + 1 - S, b = 2 * j + 1 - S;
    // 3D point (doubled-integer units) of the texel centre on face f's plane
    int p0, p1, p2;
    switch (f) {
        case 0: p0 = S; p1 = -b; p2 = -a; break;
        case 1: p0 = -S; p1 = -b; p2 = a; break;
        case 2: p0 = a; p1 = S; p2 = b; break;
        case 3: p0 = a; p1 = -S; p2 = -b; break;
        case 4: p0 = a; p1 = -b; p2 = S; break;
        default: p0 = -a; p1 = -b; p2 = -S; break;
    }
    // fold the out-of-range coordinate onto the neighbouring face
    switch (f >> 1) {
        case 0: if (!edge_fold(p1, p0, S)) edge_fold(p2, p0, S); break;
        case 1: if (!edge_fold(p0, p1, S)) edge_fold(p2, p1, S); break;
        default: if (!edge_fold(p0, p2, S)) edge_fold(p1, p2, S); break;
    }
    const int ax = p0 < 0 ? -p0 : p0, ay = p1 < 0 ? -p1 : p1, az = p2 < 0 ? -p2 : p2;
    int nf, na, nb;
    if (ax >= ay && ax >= az) {
        if (p0 > 0) { nf = 0; na = -p2; nb = -p1; }
        else { nf = 1; na = p2; nb = -p1; }
    } else if (ay >= az) {
        if (p1 > 0) { nf = 2; na = p0; nb = p2; }
        else { nf = 3; na = p0; nb = -p2; }
    } else {
        if (p2 > 0) { nf = 4; na = p0; nb = -p1; }
        else { nf = 5; na = -p0; nb = -p1; }
    }
    const int ni = (na + S - 1) >> 1, nj = (nb + S - 1) >> 1;
    return (nf * S + nj) * S + ni;
}
__device__ __noinline__ int cube_edge_index(int f, int i, int j, int S) { return cube_edge_index_inl(f, i, j, S); }

// RGB of texel (f, i, j) of a cube level with seamless edges.
__device__ __noinline__ f3 cube_texel_seamless(const float4* __restrict__ level, int S, int f, int i, int j) {
    // taps of a finite direction are within one texel of the face
    i = i < -1 ? -1 : (i > S ? S : i);
    j = j < -1 ? -1 : (j > S ? S : j);
    const bool iin = (unsigned)i < (unsigned)S, jin = (unsigned)j < (unsigned)S;
    if (iin && jin) {
        const float4 v = level[(f * S + j) * S + i];
        return {v.x, v.y, v.z};
    }
    if (iin || jin) {
        const float4 v = level[cube_edge_index(f, i, j, S)];
        return {v.x, v.y, v.z};
    }
    const int ci = i < 0 ? 0 : S - 1, cj = j < 0 ? 0 : S - 1;
    const float4 v0 = level[(f * S + cj) * S + ci];
    const float4 va = level[cube_edge_index(f, i, cj, S)];
    const float4 vb = level[cube_edge_index(f, ci, j, S)];
    return {((v0.x + va.x) + vb.x) / 3.0f, ((v0.y + va.y) + vb.y) / 3.0f, ((v0.z + va.z) + vb.z) / 3.0f};
}

// Bilinear seamless sample of one cube level (RGB).
__device__ __forceinline__ f3 sample_cube(const float4* __restrict__ level, int S, f3 dir) {
    const CubeCoord cc = cube_select(dir);
    const float u = cc.s * (float)S - 0.5f;
    const float v = cc.t * (float)S - 0.5f;
    const float fu = floorf_(u), fv = floorf_(v);
    const float a = u - fu, b = v - fv;
    const int i0 = (int)fu, j0 = (int)fv;
    const float w00 = (1.0f - a) * (1.0f - b), w10 = a * (1.0f - b);
    const float w01 = (1.0f - a) * b, w11 = a * b;
    f3 t00, t10, t01, t11;
    if (i0 >= 0 && j0 >= 0 && i0 + 1 < S && j0 + 1 < S) {
        const float4* row0 = level + (cc.face * S + j0) * S + i0;
        const float4 q00 = row0[0], q10 = row0[1], q01 = row0[S], q11 = row0[S + 1];
        t00 = {q00.x, q00.y, q00.z};
        t10 = {q10.x, q10.y, q10.z};
        t01 = {q01.x, q01.y, q01.z};
        t11 = {q11.x, q11.y, q11.z};
    } else {
        t00 = cube_texel_seamless(level, S, cc.face, i0, j0);
        t10 = cube_texel_seamless(level, S, cc.face, i0 + 1, j0);
        t01 = cube_texel_seamless(level, S, cc.face, i0, j0 + 1);
        t11 = cube_texel_seamless(level, S, cc.face, i0 + 1, j0 + 1);
    }
    return {((w00 * t00.x + w10 * t10.x) + w01 * t01.x) + w11 * t11.x,
            ((w00 * t00.y + w10 * t10.y) + w01 * t01.y) + w11 * t11.y,
            ((w00 * t00.z + w10 * t10.z) + w01 * t01.z) + w11 * t11.z};
}

// The same bilinear seamless sample in two steps, so the texel loads of one
// sample can be in flight while other work runs: cube_taps finds the four
// taps' texel indices and weights (and issues nothing), the caller loads the
// taps, cube_combine forms the sum exactly as sample_cube does. A tap at a
// cube corner (both coordinates off the face) is the mean of three texels;
// such samples are marked and cube_combine recomputes them with sample_cube.
struct CubeTaps {
    int idx[4];  // taps (i0,j0), (i0+1,j0), (i0,j0+1), (i0+1,j0+1); a corner tap holds 0
    float w00, w10, w01, w11;
    int face, i0, j0;  // the footprint's face and first texel
    bool interior;     // all four taps on face `face` (the usual case)
    bool corner;
};

// Linear texel index of tap (f, i, j), i and j at most one step off the
// face; -1 for a corner tap.
__device__ __forceinline__ int cube_tap_index(int S, int f, int i, int j) {
    i = i < -1 ? -1 : (i > S ? S : i);
    j = j < -1 ? -1 : (j > S ? S : j);
    const bool iin = (unsigned)i < (unsigned)S, jin = (unsigned)j < (unsigned)S;
    if (iin && jin) return (f * S + j) * S + i;
    if (iin || jin) return cube_edge_index_inl(f, i, j, S);
    return -1;
}

template <bool UNIT = false>
__device__ __forceinline__ CubeTaps cube_taps(int S, f3 dir) {
    const CubeCoord cc = cube_select<UNIT>(dir);
    const float u = cc.s * (float)S - 0.5f;
    const float v = cc.t * (float)S - 0.5f;
    const float fu = floorf_(u), fv = floorf_(v);
    const float a = u - fu, b = v - fv;
    const int i0 = (int)fu, j0 = (int)fv;
    CubeTaps t;
    t.w00 = (1.0f - a) * (1.0f - b);
    t.w10 = a * (1.0f - b);
    t.w01 = (1.0f - a) * b;
    t.w11 = a * b;
    t.corner = false;
    t.face = cc.face;
    t.i0 = i0;
    t.j0 = j0;
    t.interior = (uint32_t)i0 < (uint32_t)(S - 1) && (uint32_t)j0 < (uint32_t)(S - 1);
    if (t.interior) {
        const int base = (cc.face * S + j0) * S + i0;
        t.idx[0] = base;
        t.idx[1] = base + 1;
        t.idx[2] = base + S;
        t.idx[3] = base + S + 1;
    } else {
        const int di[4] = {0, 1, 0, 1}, dj[4] = {0, 0, 1, 1};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int id = cube_tap_index(S, cc.face, i0 + di[k], j0 + dj[k]);
            t.corner = t.corner || id < 0;
            t.idx[k] = id < 0 ? 0 : id;
        }
    }
    return t;
}

// The bilinear sum of loaded taps q (sample_cube's expression); a sample
// with a corner tap is resampled with sample_cube.
__device__ __forceinline__ f3 cube_combine(const float4* __restrict__ level, int S, f3 dir, const CubeTaps& t,
                                           const float4 q[4]) {
    if (t.corner) return sample_cube(level, S, dir);
    return {((t.w00 * q[0].x + t.w10 * q[1].x) + t.w01 * q[2].x) + t.w11 * q[3].x,
            ((t.w00 * q[0].y + t.w10 * q[1].y) + t.w01 * q[2].y) + t.w11 * q[3].y,
            ((t.w00 * q[0].z + t.w10 * q[1].z) + t.w01 * q[2].z) + t.w11 * q[3].z};
}

// ------------------------------------------------------------- 2D sampling
__device__ __forceinline__ int wrap_rep(int i, int n) {
    // within one period of the image without a division (35 instructions)
    int r = i < 0 ? i + n : (i >= n ? i - n : i);
    if (__builtin_expect((uint32_t)r >= (uint32_t)n, 0)) {
        r = i % n;
        if (r < 0) r += n;
    }
    return r;
}

// Bilinear REPEAT sample of an RGBA32F image (returns RGB).
__device__ __forceinline__ f3 sample_2d_rgba_repeat(const float4* __restrict__ img, int W, int H, float s, float t) {
    const float u = s * (float)W - 0.5f;
    const float v = t * (float)H - 0.5f;
    const float fu = floorf_(u), fv = floorf_(v);
    const float a = u - fu, b = v - fv;
    const int i0 = wrap_rep((int)fu, W), i1 = wrap_rep((int)fu + 1, W);
    const int j0 = wrap_rep((int)fv, H), j1 = wrap_rep((int)fv + 1, H);
    const float w00 = (1.0f - a) * (1.0f - b), w10 = a * (1.0f - b);
    const float w01 = (1.0f - a) * b, w11 = a * b;
    const float4 q00 = img[j0 * W + i0], q10 = img[j0 * W + i1], q01 = img[j1 * W + i0], q11 = img[j1 * W + i1];
    return {((w00 * q00.x + w10 * q10.x) + w01 * q01.x) + w11 * q11.x,
            ((w00 * q00.y + w10 * q10.y) + w01 * q01.y) + w11 * q11.y,
            ((w00 * q00.z + w10 * q10.z) + w01 * q01.z) + w11 * q11.z};
}

// Bilinear REPEAT sample of an RG32F image.
__device__ __forceinline__ float2 sample_2d_rg_repeat(const float2* __restrict__ img, int W, int H, float s, float t) {
    const float u = s * (float)W - 0.5f;
    const float v = t * (float)H - 0.5f;
    const float fu = floorf_(u), fv = floorf_(v);
    const float a = u - fu, b = v - fv;
    const int i0 = wrap_rep((int)fu, W), i1 = wrap_rep((int)fu + 1, W);
    const int j0 = wrap_rep((int)fv, H), j1 = wrap_rep((int)fv + 1, H);
    const float w00 = (1.0f - a) * (1.0f - b), w10 = a * (1.0f - b);
    const float w01 = (1.0f - a) * b, w11 = a * b;
    const float2 q00 = img[j0 * W + i0], q10 = img[j0 * W + i1], q01 = img[j1 * W + i0], q11 = img[j1 * W + i1];
    return {((w00 * q00.x + w10 * q10.x) + w01 * q01.x) + w11 * q11.x,
            ((w00 * q00.y + w10 * q10.y) + w01 * q01.y) + w11 * q11.y};
}

// IBL output-texel direction: texCoord = (x + .5)/D, uv = texCoord*2 - 1,
// normalize(UVToXYZ(face, uv)), then y = -y.
__device__ __forceinline__ f3 texel_dir(int face, int x, int y, int D) {
    const float rd = rcp_rn_normal((float)D);
    const float u = div_by_normal((float)x + 0.5f, (float)D, rd) * 2.0f - 1.0f;
    const float v = div_by_normal((float)y + 0.5f, (float)D, rd) * 2.0f - 1.0f;
    f3 p;
    switch (face) {
        case 0: p = {1.0f, v, -u}; break;
        case 1: p = {-1.0f, v, u}; break;
        case 2: p = {u, -1.0f, v}; break;
        case 3: p = {u, 1.0f, -v}; break;
        case 4: p = {u, v, 1.0f}; break;
        default: p = {-u, v, -1.0f}; break;
    }
    f3 d = normalize3_rn(p);  // squared length in [1, 3]
    d.y = -d.y;
    return d;
}

__host__ __device__ inline size_t cube_level_offset_floats(uint32_t S, uint32_t level) {
    size_t off = 0;
    for (uint32_t m = 0; m < level; ++m) {
        const size_t s = (S >> m) > 0 ? (S >> m) : 1;
        off += 6 * s * s * 4;
    }
    return off;
}

}  // namespace hvx
