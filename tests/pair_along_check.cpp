// CPU check of the curved elements' two-point flux (flou.jl_amd/csrc/pair_along.hpp) against extended
// precision: the device functions compiled for the host, the hardware's reciprocal (good to 2^-24) and
// quotient fixup stood in for.  Prints, per flux, dimension, metric and spread of the two states, the
// rms error of the mass, momentum and energy components over that of the reference's own FP64
// arithmetic on the same pairs (both against long double), and the largest deviation from
// that arithmetic where the densities or β lie at the log-mean's branch point; built and run by
// tests/test_pair_along.py.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>

inline double __builtin_amdgcn_rcp(double x) { return (double)(float)(1.0 / x); }
inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }
inline double __builtin_amdgcn_div_fixup(double q, double b, double a) { return std::isfinite(q) ? q : a / b; }
inline float __builtin_amdgcn_div_fixupf(float q, float b, float a) { return std::isfinite(q) ? q : a / b; }
inline int atomicOr(int* p, int b) { const int o = *p; *p |= b; return o; }
using std::fabs; using std::log; using std::sqrt; using std::exp; using std::pow;
#include "pair_along.hpp"

using LD = long double;
static const double GAM = 1.4;

template <class T> T logmean(T a, T b) {
    const T xi = a / b, f = (xi - T(1)) / (xi + T(1)), u = f * f;
    const T F = u < T(0.01) ? ((T(1) + u / T(3)) + (u * u) / T(5)) + ((u * u) * u) / T(7) : std::log(xi) / (T(2) * f);
    return (a + b) / (T(2) * F);
}

template <class T, int ND> void prim(const T* Q, T* P) {
    T s = Q[1] * Q[1];
    for (int k = 1; k < ND; ++k) s = s + Q[1 + k] * Q[1 + k];
    P[0] = Q[0];
    for (int k = 0; k < ND; ++k) P[1 + k] = Q[1 + k] / Q[0];
    P[ND + 1] = (T(GAM) - T(1)) * (Q[ND + 1] - s / (T(2) * Q[0]));
}

// The reference's flux and its contraction with the mean metric, in its order.
template <class T, int ND, int TP> void reference(const double* q1, const double* q2, const double* n1, const double* n2, T* F) {
    T Q1[5], Q2[5], P1[5], P2[5], n[3], f[5][3], um[3];
    for (int v = 0; v < ND + 2; ++v) { Q1[v] = q1[v]; Q2[v] = q2[v]; }
    for (int k = 0; k < ND; ++k) n[k] = (T(n1[k]) + T(n2[k])) / T(2);
    prim<T, ND>(Q1, P1);
    prim<T, ND>(Q2, P2);
    const T p1 = P1[ND + 1], p2 = P2[ND + 1];
    for (int k = 0; k < ND; ++k) um[k] = (P1[1 + k] + P2[1 + k]) / T(2);
    if (TP == flouhip::TP_STDAVG) {
        for (int k = 0; k < ND; ++k) {
            f[0][k] = (Q1[1 + k] + Q2[1 + k]) / T(2);
            for (int c = 0; c < ND; ++c) {
                T s = Q1[1 + c] * P1[1 + k];
                if (c == k) s = s + p1;
                s = s + Q2[1 + c] * P2[1 + k];
                if (c == k) s = s + p2;
                f[1 + c][k] = s / T(2);
            }
            f[ND + 1][k] = ((Q1[ND + 1] + p1) * P1[1 + k] + (Q2[ND + 1] + p2) * P2[1 + k]) / T(2);
        }
    } else if (TP == flouhip::TP_CHANDRASEKHAR) {
        const T b1 = P1[0] / (T(2) * p1), b2 = P2[0] / (T(2) * p2);
        const T rho = logmean(P1[0], P2[0]), p = (P1[0] + P2[0]) / (T(2) * (b1 + b2)), beta = logmean(b1, b2);
        T sq = P1[1] * P1[1];
        for (int k = 1; k < ND; ++k) sq = sq + P1[1 + k] * P1[1 + k];
        for (int k = 0; k < ND; ++k) sq = sq + P2[1 + k] * P2[1 + k];
        T h = T(1) / ((T(2) * beta) * (T(GAM) - T(1))) - sq / T(4);
        h = h + p / rho;
        for (int k = 0; k < ND; ++k) h = h + um[k] * um[k];
        for (int k = 0; k < ND; ++k) {
            f[0][k] = rho * um[k];
            for (int c = 0; c < ND; ++c)
                f[1 + c][k] = c == k ? rho * (um[k] * um[k]) + p : (rho * um[std::min(c, k)]) * um[std::max(c, k)];
            f[ND + 1][k] = (rho * um[k]) * h;
        }
    } else {
        const T rho = (P1[0] + P2[0]) / T(2), p = (p1 + p2) / T(2), e = (Q1[ND + 1] / Q1[0] + Q2[ND + 1] / Q2[0]) / T(2);
        for (int k = 0; k < ND; ++k) {
            const T m = rho * um[k];
            f[0][k] = m;
            for (int c = 0; c < ND; ++c) f[1 + c][k] = c == k ? m * um[c] + p : m * um[c];
            f[ND + 1][k] = m * e + p * um[k];
        }
    }
    for (int v = 0; v < ND + 2; ++v) {
        T s = f[v][0] * n[0];
        for (int k = 1; k < ND; ++k) s = s + f[v][k] * n[k];
        F[v] = s;
    }
}

// The kernel's: node slots as it stages them, half metrics, the pair flux.
template <int ND, int TP> void kernel(const double* q1, const double* q2, const double* n1, const double* n2, double* F) {
    constexpr int NS = flouhip::split::curved_slots<ND, TP>();
    double S[2][NS], n[ND], P[ND + 2];
    int err = 0;
    for (int s = 0; s < 2; ++s) {
        const double* q = s ? q2 : q1;
        const flouhip::Recip<double> ir(q[0]);
        flouhip::plain::cons2prim<double, ND>(q, GAM, P, ir);
        flouhip::split::curved_node<ND, TP, 1>(S[s], q, P, ir);
    }
    for (int k = 0; k < ND; ++k) n[k] = 0.5 * n1[k] + 0.5 * n2[k];
    flouhip::split::pair_flux_along<ND, TP>(S[0], S[1], n, 1.0 / (GAM - 1.0), &err, F);
}

static std::mt19937_64 rng(7);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }

template <int ND> void state(double* Q, double rho, double p) {
    double k = 0;
    Q[0] = rho;
    for (int i = 0; i < ND; ++i) {
        const double u = U(-1, 1) * std::sqrt(p / rho);
        Q[1 + i] = rho * u;
        k += u * u;
    }
    Q[ND + 1] = p / (GAM - 1) + 0.5 * rho * k;
}

template <int ND, int TP> void errors() {
    const double lo[4] = {1, 1.25, 2.5, 10}, hi[4] = {1.1, 2.2, 7.5, 1000};
    for (int metric = 0; metric < 2; ++metric)
        for (int ratio = 0; ratio < 4; ++ratio)
            for (int inverse = 0; inverse < 2; ++inverse) {
                double so[3] = {0}, sk[3] = {0};
                for (int it = 0; it < 100000; ++it) {
                    double q1[5], q2[5], n1[3], n2[3], O[5], K[5];
                    LD X[5];
                    const double r = 1 / U(1 / hi[ratio], 1 / lo[ratio]), s1 = U(1, 10), s2 = U(0.1, 10);
                    double r1 = s1 * U(0.99, 1.01), r2 = s1 * r * U(0.99, 1.01);
                    double p1 = s2 * U(0.99, 1.01), p2 = s2 * (inverse ? 1 / r : r) * U(0.99, 1.01);
                    if (U(0, 1) < 0.5) { std::swap(r1, r2); std::swap(p1, p2); }
                    state<ND>(q1, r1, p1);
                    state<ND>(q2, r2, p2);
                    for (int k = 0; k < ND; ++k) {  // a line's own direction dominates its metric, or does not
                        n1[k] = metric == 0 ? U(-1, 1) : (k == 0 ? U(0.9, 1.1) : 0.05 * U(-1, 1));
                        n2[k] = n1[k] * U(0.9, 1.1);
                    }
                    reference<LD, ND, TP>(q1, q2, n1, n2, X);
                    reference<double, ND, TP>(q1, q2, n1, n2, O);
                    kernel<ND, TP>(q1, q2, n1, n2, K);
                    const double m = std::sqrt(std::max(r1 * p1, r2 * p2)), p = std::max(p1, p2);
                    const double e = p * std::sqrt(std::max(p1 / r1, p2 / r2));
                    for (int v = 0; v < ND + 2; ++v) {
                        const int c = v == 0 ? 0 : (v <= ND ? 1 : 2);
                        const double scale = c == 0 ? m : (c == 1 ? p : e);
                        const double eo = (double)((O[v] - X[v]) / scale), ek = (double)((K[v] - X[v]) / scale);
                        so[c] += eo * eo;
                        sk[c] += ek * ek;
                    }
                }
                std::printf("error %d %d %d %g-%g %d %.4f %.4f %.4f\n", ND, TP, metric, lo[ratio], hi[ratio], inverse,
                            std::sqrt(sk[0] / so[0]), std::sqrt(sk[1] / so[1]), std::sqrt(sk[2] / so[2]));
            }
}

// Densities (or β) whose quotient is 11/9 to rounding, where f² = 0.01.
template <int ND> void branch() {
    double worst = 0;
    for (int i = 1; i <= 4000; ++i)
        for (int beta = 0; beta < 2; ++beta) {
            double q1[5], q2[5], n[3] = {1, 0.1, -0.2}, O[5], K[5];
            const double a = i * 11 / 100.0, b = i * 9 / 100.0;
            state<ND>(q1, a, beta ? 0.5 : a);
            state<ND>(q2, b, beta ? 0.5 : b);
            reference<double, ND, flouhip::TP_CHANDRASEKHAR>(q1, q2, n, n, O);
            kernel<ND, flouhip::TP_CHANDRASEKHAR>(q1, q2, n, n, K);
            double big = 0;
            for (int v = 0; v < ND + 2; ++v) big = std::max(big, std::fabs(O[v]));
            for (int v = 0; v < ND + 2; ++v) worst = std::max(worst, std::fabs(K[v] - O[v]) / big);
        }
    std::printf("branch %d %.3e\n", ND, worst);
}

template <int ND> void all() {
    errors<ND, flouhip::TP_STDAVG>();
    errors<ND, flouhip::TP_CHANDRASEKHAR>();
    errors<ND, flouhip::TP_KENNEDY_GRUBER>();
    branch<ND>();
}

int main() {
    all<2>();
    all<3>();
}
