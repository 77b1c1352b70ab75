// Arithmetic helpers shared by the FP32 and FP64 kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace ommhip {

template <class R>
struct Math;

// FP32 pair arithmetic.  erfc(x) = erfcx(x) * exp(-x^2) with erfcx fitted
// (this project's own weighted Chebyshev fit, converted to monomials) as a
// degree-8 polynomial in t = (x - 2.5)/(x + 2.5) on x in [0, 6]: relative error
// 1.2e-8 in exact arithmetic, 1.6e-7 evaluated in FP32.  exp(-x^2) reuses the
// hardware exp2; reciprocal and reciprocal square root are the hardware's
// (about 1 ulp), well inside the FP32 rounding of the force sums.
template <>
struct Math<float> {
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ float rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
    static __device__ __forceinline__ void erfc_exp(float x, float& erfc_v, float& ex) {
        float t = (x - 2.5f) * rcp(x + 2.5f);
        t = fminf(t, 0.41176470f);
        float p = 0.0003302688419353217f;
        p = fmaf(p, t, 0.0008612216333858669f);
        p = fmaf(p, t, -0.0026842965744435787f);
        p = fmaf(p, t, -0.003998667001724243f);
        p = fmaf(p, t, 0.039928220212459564f);
        p = fmaf(p, t, -0.12503232061862946f);
        p = fmaf(p, t, 0.2517129182815552f);
        p = fmaf(p, t, -0.3717367649078369f);
        p = fmaf(p, t, 0.21080636978149414f);
        ex = __builtin_amdgcn_exp2f(-(x * x) * 1.4426950408889634f);
        erfc_v = p * ex;
    }
    static __device__ __forceinline__ float round(float x) { return rintf(x); }
    static __device__ __forceinline__ float max(float a, float b) { return fmaxf(a, b); }
    // e^{-x} through the hardware exp2.
    static __device__ __forceinline__ float exp_neg(float x) { return __builtin_amdgcn_exp2f(-x * 1.4426950408889634f); }
};

template <>
struct Math<double> {
    static __device__ __forceinline__ double rcp(double x) { return 1.0 / x; }
    static __device__ __forceinline__ double rsqrt(double x) { return 1.0 / sqrt(x); }
    static __device__ __forceinline__ void erfc_exp(double x, double& erfc_v, double& ex) {
        erfc_v = erfc(x);
        ex = exp(-x * x);
    }
    static __device__ __forceinline__ double round(double x) { return rint(x); }
    static __device__ __forceinline__ double max(double a, double b) { return fmax(a, b); }
    static __device__ __forceinline__ double exp_neg(double x) { return exp(-x); }
};

// FP64 arithmetic of the mixed form's pair energies, branch-free where the
// device library's functions branch per lane (a wave then runs every branch).
//   1/sqrt(x): the hardware estimate and one third-order step.
//   e^{-y}: y = n ln 2 + r with ln 2 in two parts (Cody and Waite 1980), a degree-11
//     Chebyshev fit of e^{-r} (4e-18), scaled by 2^-n.
//   erfc(x) = erfcx(x) e^{-x^2}, the square's rounding carried into the
//     exponential; erfcx fitted as a degree-18 polynomial in
//     t = (x - 3.5)/(x + 3.5) on [0, 6] (5e-17; this project's own Chebyshev fit,
//     converted to monomials).  Against 113-bit values on [0, 6]: e^{-x^2} 1.6e-16 at
//     most, erfc 6.2e-16 at most and 1.3e-16 RMS (the library's: 3.6e-15 through
//     the rounded square, 5.6e-16 and 0.8e-16).  Past 6, where erfc is below
//     2.2e-17, erfcx keeps its value at 6.
struct PairF64 {
    static __device__ __forceinline__ double rsqrt(double x) {
        const double y = __builtin_amdgcn_rsq(x);
        const double e = __builtin_fma(-x * y, y, 1.0);
        return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
    }
    // e^{-(y + lo)}, lo far below y's last bit.
    static __device__ __forceinline__ double exp_neg2(double y, double lo) {
        const double n = ::rint(y * 1.4426950408889634);
        double r = __builtin_fma(n, -0.69314718048553913832, y);
        r = __builtin_fma(n, -7.4406171100123968474e-11, r) + lo;
        double p = -2.5110049204818658e-08;
        p = __builtin_fma(p, r, 2.763265472252779e-07);
        p = __builtin_fma(p, r, -2.7557240887229869e-06);
        p = __builtin_fma(p, r, 2.4801485441561313e-05);
        p = __builtin_fma(p, r, -0.00019841269890076403);
        p = __builtin_fma(p, r, 0.0013888888952352863);
        p = __builtin_fma(p, r, -0.008333333333319589);
        p = __builtin_fma(p, r, 0.041666666666487953);
        p = __builtin_fma(p, r, -0.1666666666666668);
        p = __builtin_fma(p, r, 0.50000000000000189);
        p = __builtin_fma(p, r, -1.0);
        p = __builtin_fma(p, r, 1.0);
        return __builtin_amdgcn_ldexp(p, -(int)n);
    }
    static __device__ __forceinline__ void erfc_exp(double x, double& erfc_v, double& ex) {
        const double d = x + 3.5;
        double inv = __builtin_amdgcn_rcp(d);
        const double e = __builtin_fma(-d, inv, 1.0);
        inv = __builtin_fma(inv, __builtin_fma(e, e, e), inv);
        const double t = fmin((x - 3.5) * inv, 2.5 / 9.5);
        double p = 6.5345122623739597e-09;
        p = __builtin_fma(p, t, 1.0367848021253531e-07);
        p = __builtin_fma(p, t, 4.9889072559661435e-07);
        p = __builtin_fma(p, t, 6.8808222316898235e-07);
        p = __builtin_fma(p, t, -1.3338186652105755e-06);
        p = __builtin_fma(p, t, -1.586264817894677e-06);
        p = __builtin_fma(p, t, 1.3329551953514485e-05);
        p = __builtin_fma(p, t, -4.6877789129044389e-06);
        p = __builtin_fma(p, t, -0.00010808726785738658);
        p = __builtin_fma(p, t, 0.00028855604152742221);
        p = __builtin_fma(p, t, 0.00026738544806297868);
        p = __builtin_fma(p, t, -0.0042422386037449271);
        p = __builtin_fma(p, t, 0.016976760915254154);
        p = __builtin_fma(p, t, -0.045436761184877404);
        p = __builtin_fma(p, t, 0.094427806909503698);
        p = __builtin_fma(p, t, -0.16133852476447774);
        p = __builtin_fma(p, t, 0.23313048160024843);
        p = __builtin_fma(p, t, -0.28926504483276755);
        p = __builtin_fma(p, t, 0.1552936556088943);
        const double y = fmin(x * x, 1000.0);
        ex = exp_neg2(y, y < 1000.0 ? __builtin_fma(x, x, -y) : 0.0);
        erfc_v = p * ex;
    }
};

}  // namespace ommhip
