// Reverse products of the FP64 line adjoint (vjp_split.hip): the node inputs of a pair's flux, the pair, and
// the pull-back of the inputs' cotangents to (ρ, m, E).
//
// Held against extended precision they are no less exact than the general adjoint's (adjoint.hpp,
// twopoint_vjp2p): rms errors 0.7 to 1.0 of its.  That takes quotients rounded as divisions in the logarithm's
// branch, where the mean's slope amplifies the error of a/b (by reciprocals good to an ulp: 1.3 times the
// general adjoint's where the branch begins), and in a node's inputs, each formed once.
#pragma once

#include "common.hpp"
#include "adjoint.hpp"
#include "exact_div.hpp"

namespace flouhip {
namespace svjp {

using adj::rcp;

// The inputs of a node with state q in an array of stride S: Chandrasekhar (ρ/2, u/2.., β), Kennedy-Gruber (ρ/2,
// u/2.., p/2, E/(2ρ)), StdAverage (u.., H, |u|²).
template <int ND, int TP, int S>
__device__ __forceinline__ void node_inputs(double* s, const double* q, double gm1) {
    constexpr int NV = ND + 2;
    const Recip<double> iq(q[0]);
    const double ir = iq.y;
    double u[ND], mu = 0;
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        u[k] = iq.fin(q[1 + k]);
        mu = fma(q[1 + k], u[k], mu);
    }
    const double p = gm1 * fma(-0.5, mu, q[NV - 1]);
    if constexpr (TP == TP_STDAVG) {
#pragma unroll
        for (int k = 0; k < ND; ++k) s[k * S] = u[k];
        s[ND * S] = fdiv(q[NV - 1] + p, q[0]);
        s[(ND + 1) * S] = mu * ir;
    } else {
        s[0] = 0.5 * q[0];
#pragma unroll
        for (int k = 0; k < ND; ++k) s[(1 + k) * S] = 0.5 * u[k];
        if constexpr (TP == TP_CHANDRASEKHAR) {
            s[(ND + 1) * S] = fdiv(0.5 * q[0], p);
        } else {
            s[(ND + 1) * S] = 0.5 * p;
            s[(ND + 2) * S] = 0.5 * q[NV - 1] * ir;
        }
    }
}

// F = atanh(f)/f of a logarithmic mean and dF/du at u = f² on the forward's branch
// (Utilities.jl:34-44); a, b: the two values.  SERIES: the caller knows that u < 0.01.  Both
// forms are evaluated and selected otherwise: a branch per pair in the unrolled line took every
// register and spilled.
template <bool SERIES>
__device__ __forceinline__ void lm_factor(double u, double f, double a, double b, double& F, double& dF) {
    F = fma(u, fma(u, fma(u, 1.0 / 7, 1.0 / 5), 1.0 / 3), 1.0);
    dF = fma(u, fma(u, 3.0 / 7, 2.0 / 5), 1.0 / 3);
    if constexpr (!SERIES) {
        const double Fl = 0.5 * fdiv(log(fdiv(a, b)), f);
        const double dl = 0.5 * (rcp(1 - u) - Fl) * rcp(u);
        F = u < 0.01 ? F : Fl;
        dF = u < 0.01 ? dF : dl;
    }
}

// Reverse product of component n (the first velocity) of the two-point flux for the cotangent
// G = (ρ, n, t.., E), scaled by s, added to the cotangents gi and gj of the nodes' inputs:
// Chandrasekhar (ρ/2, u/2.., β), Kennedy-Gruber (ρ/2, u/2.., p/2, E/(2ρ)).
// CURV: of the flux along n, the mean metric, instead.
template <int ND, int TP, bool SERIES, bool CURV>
__device__ __forceinline__ void pair_vjp(const double* P, const double* Q, const double* G, const double* n, double s,
                                         double ig1, double* gi, double* gj) {
    constexpr int NV = ND + 2;
    double gn = G[1];
    if constexpr (CURV) {
        gn = G[1] * n[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) gn = fma(G[1 + k], n[k], gn);
    }
    if constexpr (TP == TP_STDAVG) {  // (u.., H, |u|²; only for CURV, see line_phase); s: with the mean's ½
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const double* X = side ? Q : P;
            double* g = side ? gj : gi;
            double un = X[0] * n[0], U = G[1] * X[0];
#pragma unroll
            for (int k = 1; k < ND; ++k) {
                un = fma(X[k], n[k], un);
                U = fma(G[1 + k], X[k], U);
            }
            U = fma(G[NV - 1], X[ND], U);
            const double g1 = 1 / ig1, pg = g1 * fma(G[NV - 1], un, gn), gU = G[0] + U;
            g[0] = fma(s, fma(-U, un, 0.5 * pg * X[ND + 1]), g[0]);
#pragma unroll
            for (int k = 0; k < ND; ++k)
                g[1 + k] = fma(s, fma(G[1 + k], un, fma(-pg, X[k], gU * n[k])), g[1 + k]);
            g[NV - 1] = fma(s, fma(G[NV - 1], un, pg), g[NV - 1]);
        }
        return;
    }
    double ub[ND];
#pragma unroll
    for (int k = 0; k < ND; ++k) ub[k] = P[1 + k] + Q[1 + k];
    double un = ub[0];
    if constexpr (CURV) {
        un = ub[0] * n[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) un = fma(ub[k], n[k], un);
    }
    double gu = G[1] * ub[0];
#pragma unroll
    for (int k = 1; k < ND; ++k) gu = fma(G[1 + k], ub[k], gu);
    const double ge = G[NV - 1];
    if constexpr (TP == TP_KENNEDY_GRUBER) {
        // f = (m, m ū + p̄ n, m ē + p̄ ū_n), m = ρ̄ ū_n: every input enters as the sum
        const double rho = P[0] + Q[0], p = P[ND + 1] + Q[ND + 1], e = P[ND + 2] + Q[ND + 2];
        const double m = rho * un;
        const double mb = fma(ge, e, G[0] + gu);
        const double unb = fma(mb, rho, ge * p);
        double t[NV + 1];
        t[0] = mb * un;
#pragma unroll
        for (int k = 0; k < ND; ++k) t[1 + k] = CURV ? fma(m, G[1 + k], unb * n[k]) : (k == 0 ? fma(m, gn, unb) : m * G[1 + k]);
        t[ND + 1] = fma(ge, un, gn);
        t[ND + 2] = ge * m;
#pragma unroll
        for (int c = 0; c < NV + 1; ++c) {
            gi[c] = fma(s, t[c], gi[c]);
            gj[c] = fma(s, t[c], gj[c]);
        }
    } else {
        // ρ̂ = (a_i + a_j)/F_ρ, p̄ = (a_i + a_j)/(β_i + β_j), m = ρ̂ ū_n,
        // h = (F_β/(γ-1) + F_ρ)/(β_i + β_j) + 2 v_i·v_j, f = (m, m ū + p̄ n, m h)
        double dot = P[1] * Q[1];
#pragma unroll
        for (int k = 1; k < ND; ++k) dot = fma(P[1 + k], Q[1 + k], dot);
        const double hs = P[0] + Q[0], dA = P[0] - Q[0], sb = P[ND + 1] + Q[ND + 1], db = P[ND + 1] - Q[ND + 1];
        const double rb = rcp(sb), ihs = rcp(hs);
        const double fr = dA * ihs, ur = fr * fr, fb = db * rb, u2 = fb * fb;
        double Fr, dFr, Fb, dFb;
        if (!SERIES) __builtin_amdgcn_sched_barrier(0);  // one logarithm's registers at a time
        lm_factor<SERIES>(ur, fr, P[0], Q[0], Fr, dFr);
        if (!SERIES) __builtin_amdgcn_sched_barrier(0);
        lm_factor<SERIES>(u2, fb, P[ND + 1], Q[ND + 1], Fb, dFb);
        if (!SERIES) __builtin_amdgcn_sched_barrier(0);
        const double iFr = rcp(Fr);
        const double rho = hs * iFr;
        const double m = rho * un;
        const double Xf = fma(Fb, ig1, Fr);
        const double h = fma(rb, Xf, 2 * dot);
        const double hb = ge * m;                     // h̄
        const double mb = fma(ge, h, G[0] + gu);      // m̄
        const double mbr = mb * rho;                  // of ū_n
        const double rhob = mb * un;                  // of ρ̂
        const double t = hb * rb;
        double rbb = fma(hb, Xf, gn * hs);            // of 1/(β_i + β_j), through h and p̄
        const double Frb = fma(-rhob * rho, iFr, t);  // of F_ρ, through ρ̂ and h
        double hsb = fma(gn, rb, rhob * iFr);         // of a_i + a_j, through p̄ and ρ̂
        const double dAb = (2 * fr) * (Frb * dFr) * ihs;
        hsb = fma(-dAb, fr, hsb);
        const double fbb = (2 * fb) * (t * ig1) * dFb;
        const double dbb = fbb * rb;
        rbb = fma(fbb, db, rbb);
        const double sbb = -rbb * rb * rb;
        const double dotb = 2 * hb;
        gi[0] = fma(s, hsb + dAb, gi[0]);
        gj[0] = fma(s, hsb - dAb, gj[0]);
        gi[NV - 1] = fma(s, sbb + dbb, gi[NV - 1]);
        gj[NV - 1] = fma(s, sbb - dbb, gj[NV - 1]);
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const double ubb = CURV ? fma(m, G[1 + k], mbr * n[k]) : (k == 0 ? fma(m, gn, mbr) : m * G[1 + k]);
            gi[1 + k] = fma(s, fma(dotb, Q[1 + k], ubb), gi[1 + k]);
            gj[1 + k] = fma(s, fma(dotb, P[1 + k], ubb), gj[1 + k]);
        }
    }
}

// The state's cotangent V from the inputs s (stride S) and their cotangents t; StdAverage's are the state's.
template <int ND, int TP, int S>
__device__ __forceinline__ void node_pullback(const double* s, const double* t, double gm1, double* V) {
    constexpr int NV = ND + 2;
    if constexpr (TP == TP_STDAVG) {
#pragma unroll
        for (int v = 0; v < NV; ++v) V[v] = t[v];
    } else {
        const double rho = 2 * s[0], ir = rcp(rho);
        double u[ND], uu = 0, ubu = 0;
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            u[k] = 2 * s[(1 + k) * S];
            uu = fma(u[k], u[k], uu);
        }
        double rb, pg, eb;  // of ρ at fixed (u, p, E), (γ-1) × of p, of E at fixed ρ
        if constexpr (TP == TP_CHANDRASEKHAR) {
            const double b = s[(ND + 1) * S], ip = fdiv(2 * b, rho);  // 1/p = 2β/ρ
            rb = 0.5 * fma(t[NV - 1], ip, t[0]);
            pg = -gm1 * t[NV - 1] * (b * ip);
            eb = 0;
        } else {
            eb = 0.5 * t[ND + 2] * ir;
            rb = fma(-eb, 2 * s[(ND + 2) * S], 0.5 * t[0]);
            pg = 0.5 * gm1 * t[ND + 1];
        }
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const double ubk = 0.5 * t[1 + k];
            ubu = fma(ubk, u[k], ubu);
            V[1 + k] = fma(ubk, ir, -pg * u[k]);
        }
        V[0] = fma(-ubu, ir, fma(0.5 * pg, uu, rb));
        V[NV - 1] = pg + eb;
    }
}

}  // namespace svjp
}  // namespace flouhip
