// The pair force laws of the PP pair kernels (pp_tiled.hip, pp_newton.hip,
// pp_sparse.hip): the arithmetic of each mode is described at the head of pp_tiled.hip.
#pragma once
#include "common.h"
#include "pp_kernels.h"

namespace cube2 {

constexpr int kQ = 128;  // queue entries per wavefront
// A position farther from every particle than any range: its squared distance
// overflows to +inf, so a pair test with it fails without a bounds check.
constexpr float kFar = 1e30f;

// 1/x from an approximation y0: with e = 1 - x*y0 (one FMA, rounded once),
// 1/x = y0/(1-e) = y0 (1 + e + e^2 + e^3/(1-e)), so y0 + y0 (e + e^2) is
// within |e|^3 + 3*2^-53 (relative) of 1/x.  For |e| <= 2^-18 that is below
// 2^-51.
__device__ inline double recip_refine(double x, double y0) {
    const double e = fma(-x, y0, 1.0);
    return fma(fma(e, e, e), y0, y0);
}

__device__ inline float div_by(float a, double y) { return (float)((double)a * y); }

// RN(sqrt(x)) and an FP64 reciprocal of it from one v_rsq_f32, for normal
// positive finite x (pair distances: the positions are multiples of ratio_cs *
// 2^-16 apart).  With y =
// rsq(x), g = x y is within a few ulps of sqrt(x), its residual d = x - g^2 is
// exact in an FMA, and g + d y/2 differs from sqrt(x) by about 2^-45, so that
// its rounding could only err where sqrt(x) lies that close to a midpoint;
// no float does (the self-test compares every float of exponent in [-40, 40]
// with IEEE sqrtf).  y is within 2^-21 of 1/RN(sqrt(x)), so one cubic step
// (recip_refine) makes the reciprocal.  Against v_sqrt_f32 with a rounding
// test on both neighbours and v_rcp_f64: 5 instead of 10 instructions and
// one transcendental fewer.
__device__ inline float sqrt_recip(float x, double& inv) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float g = x * y;
    const float r = fmaf(fmaf(-g, g, x), 0.5f * y, g);
    inv = recip_refine((double)r, (double)y);
    return r;
}

// Wavefront-uniform copies (scalar registers) of values every lane holds.
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline float uni(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ inline double uni(double v) {
    return __hiloint2double(uni(__double2hiint(v)), uni(__double2loint(v)));
}

struct FraK {
    float a;        // softening diameter
    double inv_a;   // 1/a in FP64
    double two_inv_a;  // 2/a
    double half_a2;  // (a/2)^2 in FP64
    float c;        // (1/35)/(a*a), as basic_functions.f08:103 rounds it
    float r2max;    // a^2 (1 + 2^-17): for r^2 above it, RN(2r/a) > 2 for certain
};

__device__ inline FraK make_frak(float a) {
    FraK K;
    K.a = a;
    K.inv_a = a > 0.0f ? 1.0 / (double)a : 0.0;
    K.two_inv_a = 2.0 * K.inv_a;
    K.half_a2 = 0.25 * (double)a * (double)a;
    K.r2max = (float)((double)a * a * (1.0 + 0x1p-17));
    {
#pragma clang fp contract(off)
        K.c = 1.0f / 35.0f / (a * a);
    }
    return K;
}

__device__ inline FraK uni(const FraK& K) {
    return FraK{uni(K.a), uni(K.inv_a), uni(K.two_inv_a), uni(K.half_a2), uni(K.c), uni(K.r2max)};
}

// F_ra(r, a) of basic_functions.f08:95-109 with the reference's rounding, for
// ep = RN(2r/a) <= 2 (the caller handles a = 0 and ep > 2, where F_ra is
// 1/(r*r)).  Evaluated without divergence: the powers are shared, both
// polynomials are formed in the reference's operation order, and one is
// selected.  RN(12/e2) is 12 * (FP64 reciprocal), rounded once to float;
// the reciprocal refines y0 = (a/2)^2 (1/r)^2, which is within a few float
// roundings of 1/e2 (ep = RN(2r/a), e2 = RN(ep*ep)).
__device__ inline float fra_ref_poly(float ep, const FraK& K, double inv_r2) {
#pragma clang fp contract(off)
    const float e2 = ep * ep, e3 = e2 * ep, e4 = e3 * ep, e5 = e4 * ep, e6 = e5 * ep;
    const float t12 = (float)(12.0 * recip_refine((double)e2, K.half_a2 * inv_r2));
    const float hi = K.c * (t12 - 224.0f + 896.0f * ep - 840.0f * e2 + 224.0f * e3 + 70.0f * e4 -
                            48.0f * e5 + 7.0f * e6);
    const float lo = K.c * (224.0f * ep - 224.0f * e3 + 70.0f * e4 + 48.0f * e5 - 21.0f * e6);
    // (the reference's F_ra is 0 at ep = 0; pairs here have r^2 >= 2^-28, so
    // ep > 0)
    return ep > 1.0f ? hi : lo;
}

__device__ inline float fra_fast2(float ep, float ir2, float c) {
    if (ep > 2.0f) return ir2;
    const float hi = fmaf(3.0f / 35.0f, ir2,
                          c * fmaf(ep, fmaf(ep, fmaf(ep, fmaf(ep, fmaf(ep, fmaf(ep, 7.0f, -48.0f),
                                                                         70.0f), 224.0f), -840.0f),
                                            896.0f), -224.0f));
    const float e2 = ep * ep;
    const float lo = c * ep * fmaf(e2, fmaf(ep, fmaf(ep, fmaf(ep, -21.0f, 48.0f), 70.0f), -224.0f), 224.0f);
    return ep > 1.0f ? hi : lo;
}

enum { kModeRef = 0, kModeFast = 1, kModePrecise = 2, kModePlummer = 3 };

// 1/r^2 - F_ra(r, a) for r < a (ep = 2r/a in (0, 2]), cancellation-free.
__device__ inline float short_term(float ep, float ir2, float c) {
    const float t = 2.0f - ep, t2 = t * t;
    const float q = fmaf(ep, fmaf(ep, fmaf(ep, 7.0f, 22.0f), 10.0f), 4.0f);
    const float hi = t2 * t2 * t * q * ir2 * (1.0f / 140.0f);
    const float e2 = ep * ep;
    const float lo =
        ir2 - c * ep * fmaf(e2, fmaf(ep, fmaf(ep, fmaf(ep, -21.0f, 48.0f), 70.0f), -224.0f), 224.0f);
    return ep > 1.0f ? hi : lo;
}

// 1/r^2 - r / (r^2 + eps^2)^(3/2) (Plummer softening), cancellation-free:
// with u = eps^2/r^2 and w = (1 + u)^(-1/2) it is (1 - w^3)/r^2, and
// 1 - w = u w^2 / (1 + w), so (1/r^2) u w^2 (1 + w + w^2) / (1 + w).
__device__ inline float plummer_term(float ir2, float eps2) {
    const float u = eps2 * ir2;
    const float w = __frsqrt_rn(1.0f + u);
    const float w2 = w * w;
    return ir2 * u * w2 * (1.0f + w + w2) / (1.0f + w);
}

template <int kMode>
__device__ inline void pair_force(float4 e, const FraK& Ka, const FraK& Kr, float& fx, float& fy,
                                  float& fz) {
    if (kMode == kModeRef) {
#pragma clang fp contract(off)
        double inv_rm;
        const float rm = sqrt_recip(e.w, inv_rm);
        // RN(1/(r*r)): the reciprocal of RN(r*r) refined from (1/r)^2
        const double inv_rm2 = inv_rm * inv_rm;
        const float frr = (float)recip_refine((double)(rm * rm), inv_rm2);
        // range term: r < range, so ep <= 2 except by rounding at the cutoff
        // (RN(2 rm / a): doubling is exact on either side of the product)
        const float epr = div_by(rm, Kr.two_inv_a);
        const float fr = epr > 2.0f ? frr : fra_ref_poly(epr, Kr, inv_rm2);
        // softening term: 1/(r*r) unless r is within app; the polynomial runs
        // only when some lane of the wavefront needs it
        float fa = frr;
        if (Ka.a != 0.0f && __ballot(e.w <= Ka.r2max)) {
            const float epa = div_by(rm, Ka.two_inv_a);
            if (__ballot(epa <= 2.0f)) {
                const float pa = fra_ref_poly(epa, Ka, inv_rm2);
                if (epa <= 2.0f) fa = pa;
            }
        }
        const float fpp = fa - fr;
        fx = div_by(fpp * e.x, inv_rm);
        fy = div_by(fpp * e.y, inv_rm);
        fz = div_by(fpp * e.z, inv_rm);
    } else if (kMode == kModeFast) {
        const float ir = __frsqrt_rn(e.w);
        const float ir2 = ir * ir;
        const float r = e.w * ir;
        float fa = ir2;
        if (r <= Ka.a) fa = fra_fast2(r * (float)(2.0 * Ka.inv_a), ir2, Ka.c);
        const float f = (fa - fra_fast2(r * (float)(2.0 * Kr.inv_a), ir2, Kr.c)) * ir;
        fx = f * e.x;
        fy = f * e.y;
        fz = f * e.z;
    } else if (kMode == kModePlummer) {
        // pair = (1/r^2 - F_ra(r, range)) - (1/r^2 - r/(r^2 + app^2)^(3/2)),
        // each piece cancellation-free (softening length eps = app)
        const float r = sqrtf(e.w);
        const float ir = 1.0f / r;
        const float ir2 = ir * ir;
        float f = short_term(r * (float)(2.0 * Kr.inv_a), ir2, Kr.c);
        if (Ka.a > 0.0f) f -= plummer_term(ir2, Ka.a * Ka.a);
        f *= ir;
        fx = f * e.x;
        fy = f * e.y;
        fz = f * e.z;
    } else {
        // pair = (1/r^2 - F_ra(r, range)) - (1/r^2 - F_ra(r, app)), the second
        // term zero for r > app; each piece cancellation-free.
        const float r = sqrtf(e.w);
        const float ir = 1.0f / r;
        const float ir2 = ir * ir;
        float f = short_term(r * (float)(2.0 * Kr.inv_a), ir2, Kr.c);
        if (Ka.a > 0.0f && r < Ka.a) f -= short_term(r * (float)(2.0 * Ka.inv_a), ir2, Ka.c);
        f *= ir;
        fx = f * e.x;
        fy = f * e.y;
        fz = f * e.z;
    }
}

// Orders LDS accesses of the lanes of one wavefront.  LDS operations of a
// wavefront are performed in issue order, so a compiler barrier suffices (no
// block barrier: the wavefronts of a block run independent trip counts).
__device__ inline void wave_lds_sync() { __builtin_amdgcn_wave_barrier(); }

// Signed fixed point (value * scale, rounded to nearest) of a pairs-once
// partial sum, added to a particle's 64-bit accumulator: integer adds
// commute, so the totals do not depend on the order of the atomics.
__device__ inline unsigned long long to_fixed(double v, float scale) {
    return (unsigned long long)__double2ll_rn(v * (double)scale);
}
__device__ inline void fixed_add(unsigned long long* dst, double v, float scale) {
    if (v != 0.0) atomicAdd(dst, to_fixed(v, scale));
}

}  // namespace cube2
