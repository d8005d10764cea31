// Two-point flux along a mean metric: the pairs of the FP64 split form on curved elements.
//
// The flux along n̄ is formed directly (ρ̂ ū·n̄ first) instead of every component's contraction, with
// sums by fused multiply-adds and quotients that share their reciprocals but are rounded as divisions.
// Its rms error against extended precision is at most the reference order's, from 0.8 of it
// (products with reciprocals good to an ulp, without the last correction: up to 1.4 of it where the
// logarithm's branch begins).
#pragma once

#include "common.hpp"
#include "physics_plain.hpp"

namespace flouhip {
namespace split {

// F of the logarithmic mean, see plain::logmean_factor; is: 1/(a + b).  The series' argument
// (a - b)/(a + b) is formed directly.  Where u could be 0.01 to rounding or more, the reference's quotients
// decide (the branches are 1e-9 apart there: 5 % of the pairs with values as 11 to 9 took the other one), and
// the logarithm and its divisor share the rounding of a/b, which their quotient then hardly feels.
__device__ __forceinline__ double mean_factor(double a, double b, double is, int* err) {
    const double f = (a - b) * is, u = f * f;
    if (u < 0.01 * (1 - 1e-12)) {
        const double s = __builtin_fma(u, 1.0 / 7, 1.0 / 5);
        return __builtin_fma(u, __builtin_fma(u, s, 1.0 / 3), 1.0);
    }
    return plain::logmean_factor(a, b, err);
}

// Flux input slots: plain::put_slots and, for Chandrasekhar, |u|²/4.
template <int ND, int TP>
constexpr int curved_slots() {
    return plain::tp_slots<ND, TP>() + (TP == TP_CHANDRASEKHAR ? 1 : 0);
}

// The slots of a node with primitives P in an array of stride S; ir: the reciprocal of ρ.
template <int ND, int TP, int S>
__device__ __forceinline__ void curved_node(double* s, const double* q, const double* P, const Recip<double>& ir) {
    plain::put_slots<double, ND, TP, S>(s, q, P, ir);
    if constexpr (TP == TP_CHANDRASEKHAR) {
        double uu = P[1] * P[1];
#pragma unroll
        for (int k = 1; k < ND; ++k) uu = __builtin_fma(P[1 + k], P[1 + k], uu);
        s[(ND + 2) * S] = 0.25 * uu;
    }
}

// Velocity k of a node, from its slots.
template <int TP, int S>
__device__ __forceinline__ double curved_velocity(const double* s, int k) {
    return TP == TP_STDAVG ? s[k * S] : 2 * s[(1 + k) * S];
}

// Two-point flux along the mean metric n of two nodes.
template <int ND, int TP>
__device__ __forceinline__ void pair_flux_along(const double* A, const double* B, const double* n, double ig1, int* err,
                                                double* F) {
    if constexpr (TP == TP_STDAVG) {
        double w[2], m = (A[ND + 1] + B[ND + 1]) * n[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) m = __builtin_fma(A[ND + 1 + k] + B[ND + 1 + k], n[k], m);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const double* X = s ? B : A;
            w[s] = X[0] * n[0];
#pragma unroll
            for (int k = 1; k < ND; ++k) w[s] = __builtin_fma(X[k], n[k], w[s]);
        }
        const double p = A[ND] + B[ND];
        F[0] = m;
#pragma unroll
        for (int c = 0; c < ND; ++c)
            F[1 + c] = __builtin_fma(A[ND + 1 + c], w[0], __builtin_fma(B[ND + 1 + c], w[1], p * n[c]));
        F[ND + 1] = __builtin_fma(A[2 * ND + 1] + A[ND], w[0], (B[2 * ND + 1] + B[ND]) * w[1]);
    } else {
        double u[ND];
#pragma unroll
        for (int k = 0; k < ND; ++k) u[k] = A[1 + k] + B[1 + k];
        double un = u[0] * n[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) un = __builtin_fma(u[k], n[k], un);
        const double hs = A[0] + B[0];
        double mass, p, e;
        if constexpr (TP == TP_CHANDRASEKHAR) {
            const double sb = A[ND + 1] + B[ND + 1];
            const Recip<double> ihs(hs), isb(sb);
            const double fr = mean_factor(A[0], B[0], ihs.y, err), fb = mean_factor(A[ND + 1], B[ND + 1], isb.y, err);
            mass = fdiv(hs, fr) * un;
            p = isb.div(hs);  // 0 where a node has no pressure, see plain::pair_flux
            // 1/(2β̂(γ-1)) + p/ρ̂ = (F_β/(γ-1) + F_ρ)/(β1 + β2), + |ū|² - (|u1|² + |u2|²)/4
            e = isb.fin(__builtin_fma(fb, ig1, fr)) - (A[ND + 2] + B[ND + 2]);
#pragma unroll
            for (int k = 0; k < ND; ++k) e = __builtin_fma(u[k], u[k], e);
            F[ND + 1] = mass * e;
        } else {
            p = A[ND + 1] + B[ND + 1];
            e = A[ND + 2] + B[ND + 2];
            mass = hs * un;
            F[ND + 1] = __builtin_fma(mass, e, p * un);
        }
        F[0] = mass;
#pragma unroll
        for (int c = 0; c < ND; ++c) F[1 + c] = __builtin_fma(mass, u[c], p * n[c]);
    }
}

}  // namespace split
}  // namespace flouhip
