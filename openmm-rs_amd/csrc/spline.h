// Order-5 cardinal B-splines of smooth PME on the device: the weights and
// derivatives of one fractional coordinate and the stencil of a position.
#pragma once

#include "common.h"

namespace ommhip {

// x / 3, correctly rounded (P. Markstein, IA-64 and Elementary Functions, 2000:
// a quotient within an ulp, corrected by its exact remainder times the rounded
// reciprocal), in three instructions instead of the general division's ten.
template <class R>
__device__ __forceinline__ R third(R x) {
    const R r = (R)1 / (R)3, q = x * r;
    return fma(fma(q, (R)-3, x), r, q);
}

// Order-5 cardinal B-spline weights and derivatives (pme.rs:151-174).  Which
// products are fused is written out: the spreads' kernels have to agree in
// every bit, and the compiler's own choice varies from kernel to kernel.
template <class R>
__device__ __forceinline__ void spline5(R f, R w[5], R dw[5]) {
#pragma clang fp contract(off)
    w[0] = (R)1 - f;
    w[1] = f;
    w[2] = f * w[1] / (R)2;
    w[1] = fma(f + (R)1, w[0], ((R)2 - f) * w[1]) / (R)2;
    w[0] *= ((R)1 - f) / (R)2;
    w[3] = third(f * w[2]);
    w[2] = third(fma(f + (R)1, w[1], ((R)3 - f) * w[2]));
    w[1] = third(fma(f + (R)2, w[0], ((R)2 - f) * w[1]));
    w[0] *= third((R)1 - f);
    dw[0] = -w[0];
    dw[1] = w[0] - w[1];
    dw[2] = w[1] - w[2];
    dw[3] = w[2] - w[3];
    dw[4] = w[3];
    w[4] = f * w[3] / (R)4;
    w[3] = fma(f + (R)1, w[2], ((R)4 - f) * w[3]) / (R)4;
    w[2] = fma(f + (R)2, w[1], ((R)3 - f) * w[2]) / (R)4;
    w[1] = fma(f + (R)3, w[0], ((R)2 - f) * w[1]) / (R)4;
    w[0] *= ((R)1 - f) / (R)4;
}

// w[i] for an i known at run time, without an indexed register.
template <class R>
__device__ __forceinline__ R pick(const R w[5], int i) {
    return i == 0 ? w[0] : (i == 1 ? w[1] : (i == 2 ? w[2] : (i == 3 ? w[3] : w[4])));
}

// The base index alone, as stencil_axis takes it.
__device__ __forceinline__ int stencil_base(const double p[3], const Box& b, int d, int n) {
#pragma clang fp contract(off)
    const double f = fma(p[2], b.recip[d * 3 + 2], fma(p[1], b.recip[d * 3 + 1], p[0] * b.recip[d * 3]));
    const int i = (int)floor((f - floor(f)) * (double)n);
    return i < n ? i : 0;
}

// pme.rs:201-218: base index and spline of the fractional grid coordinate along
// axis d of a grid of n points.
template <class R>
__device__ __forceinline__ int stencil_axis(const double p[3], const Box& b, int d, int n, R w[5], R dw[5]) {
#pragma clang fp contract(off)
    const double f = fma(p[2], b.recip[d * 3 + 2], fma(p[1], b.recip[d * 3 + 1], p[0] * b.recip[d * 3]));
    const double part = f - floor(f), c = part * (double)n;
    const double fl = floor(c);
    spline5<R>((R)fma(part, (double)n, -fl), w, dw);
    const int i = (int)fl;  // in [0, n], n where f - floor(f) rounds to one
    return i < n ? i : 0;
}

template <class R>
__device__ __forceinline__ void stencil(const double* p, const Box& b, const int dims[3], int idx[3], R w[3][5],
                                        R dw[3][5]) {
    for (int a = 0; a < 3; ++a) idx[a] = stencil_axis<R>(p, b, a, dims[a], w[a], dw[a]);
}

}  // namespace ommhip
