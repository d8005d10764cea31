// Divisions of the plain kernels with the reciprocal shared between quotients.
//
// The plain kernels divide where the reference divides, and every quotient has to be
// rounded as IEEE division rounds it.  The compiler's FP64 division is 11 instructions
// (two of them the scaling of extreme exponents, one a quarter-rate reciprocal); most
// quotients of a kernel share their denominator (ρ, p, J, 2ρ) or divide by 3, 5 or 7.
// With y = 1/b refined by Newton steps, q = a·y, r = a - b·q (exact in an fma) and
// q + r·y rounded once is the correctly rounded quotient (P. Markstein, IBM J. Res. Dev.
// 34 (1990) 111-119; the compiler's sequence is the same one between its scaling steps), so
// a quotient by a known reciprocal is 3 instructions and a constant one as well.
// div_fixup restores the quotients of zeros, infinities and NaN.  Without the scaling,
// results lose their last bits only where the denominator or the quotient's residual leaves
// the normal range (FP64: magnitudes beyond 1e±290; FP32: beyond 1e±30).
//
// Measured with the plain kernels' other work unchanged, same bits: five ORK256 steps of the
// 2-D hybrid form (2175 elements, N=5, limiter and CFL control) 2652 -> 2253 us, ten steps of
// the Sod tube with matrix dissipation 499 -> 450 us, an SSPRK33 step of the 3-D strong form
// in FP32 (7182 elements, N=4) 123 -> 116 us.
//
// Types other than double and float (the dual numbers of the adjoint) divide.
#pragma once

#include <hip/hip_runtime.h>

namespace flouhip {

template <typename T>
struct Recip {
    T b;
    __device__ explicit Recip(T b_) : b(b_) {}
    __device__ T div(T a) const { return a / b; }                   // a / b
    __device__ T div2(T a) const { return a / (T(2) * b); }         // a / (2b)
    __device__ T fin(T a) const { return a / b; }                   // a / b, b finite and not 0, a finite
    __device__ T fix(T q, T a) const { return q; }                  // div(a) from q = fin(a)
};

template <>
struct Recip<double> {
    double b, y;
    __device__ explicit Recip(double b_) : b(b_) {
        // v_rcp_f64 is good to 2^-24; one step of third order leaves only the last rounding
        const double y0 = __builtin_amdgcn_rcp(b);
        const double e = __builtin_fma(-b, y0, 1.0);
        y = __builtin_fma(y0, __builtin_fma(e, e, e), y0);
    }
    __device__ static double quot(double a, double b, double y) {
        const double q = a * y;
        return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), y, q), b, a);
    }
    __device__ double fix(double q, double a) const { return __builtin_amdgcn_div_fixup(q, b, a); }
    __device__ double div(double a) const { return quot(a, b, y); }
    __device__ double div2(double a) const { return quot(a, 2.0 * b, 0.5 * y); }
    __device__ double fin(double a) const {
        const double q = a * y;
        return __builtin_fma(__builtin_fma(-b, q, a), y, q);
    }
};

template <>
struct Recip<float> {
    float b, y;
    __device__ explicit Recip(float b_) : b(b_) {
        const float y0 = __builtin_amdgcn_rcpf(b);
        y = __builtin_fmaf(__builtin_fmaf(-b, y0, 1.0f), y0, y0);
    }
    __device__ static float quot(float a, float b, float y) {
        const float q = a * y;
        return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-b, q, a), y, q), b, a);
    }
    __device__ float fix(float q, float a) const { return __builtin_amdgcn_div_fixupf(q, b, a); }
    __device__ float div(float a) const { return quot(a, b, y); }
    __device__ float div2(float a) const { return quot(a, 2.0f * b, 0.5f * y); }
    __device__ float fin(float a) const {
        const float q = a * y;
        return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
    }
};

// a / b
template <typename T>
__device__ inline T xdiv(T a, T b) {
    return Recip<T>(b).div(a);
}

// a / b for finite a and b, b not 0 (elsewhere NaN, where the quotient would be infinite or 0)
template <typename T>
__device__ inline T fdiv(T a, T b) {
    return Recip<T>(b).fin(a);
}

// a / C for a finite a and a small whole number C (1/C rounded at compile time)
template <int C, typename T>
__device__ inline T cdiv(T a) {
    return a / T(C);
}
template <int C>
__device__ inline double cdiv(double a) {
    constexpr double y = 1.0 / C;
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-(double)C, q, a), y, q);
}
template <int C>
__device__ inline float cdiv(float a) {
    constexpr float y = 1.0f / C;
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-(float)C, q, a), y, q);
}

}  // namespace flouhip
