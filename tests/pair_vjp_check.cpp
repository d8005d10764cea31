// CPU check of the line adjoint's reverse products (flou.jl_amd/csrc/pair_vjp.hpp) against extended
// precision: the device functions compiled for the host, the hardware's instructions stood in for.  Prints, per
// flux, dimension, metric and spread of the two states, the rms error of the ρ, momentum and energy cotangents over
// that of the general adjoint (twopoint_vjp2p of adjoint.hpp in FP64) on the same pairs, both against
// twopoint_vjp2p in long double; built and run by tests/test_pair_vjp.py.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>

inline double __builtin_amdgcn_rcp(double x) { return (double)(float)(1.0 / x); }
inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }
inline double __builtin_amdgcn_div_fixup(double q, double b, double a) { return std::isfinite(q) ? q : a / b; }
inline float __builtin_amdgcn_div_fixupf(float q, float b, float a) { return std::isfinite(q) ? q : a / b; }
inline void __builtin_amdgcn_sched_barrier(int) {}
using std::fabs; using std::fma; using std::log; using std::sqrt;
#include "pair_vjp.hpp"

using LD = long double;
static const double GAM = 1.4;
static std::mt19937_64 rng(7);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }

template <class T, int ND, int TP>
void general(const double* q1, const double* q2, const double* n1, const double* n2, const double* G, T (*b)[5]) {
    T Q[2][5], R[2][8], n[3], g[5];
    for (int v = 0; v < ND + 2; ++v) { Q[0][v] = q1[v]; Q[1][v] = q2[v]; g[v] = G[v]; b[0][v] = b[1][v] = T(0); }
    for (int k = 0; k < ND; ++k) n[k] = (T(n1[k]) + T(n2[k])) / T(2);
    for (int s = 0; s < 2; ++s) flouhip::adj::node_prims<T, ND>(Q[s], T(GAM), R[s]);
    flouhip::adj::twopoint_vjp2p<T, ND, TP>(Q[0], R[0], Q[1], R[1], n, T(GAM), T(1) / (T(GAM) - T(1)), g, b[0], b[1]);
}

template <int ND, int TP>
void line(const double* q1, const double* q2, const double* n1, const double* n2, const double* G, double (*b)[5]) {
    constexpr int NA = TP == flouhip::TP_KENNEDY_GRUBER ? ND + 3 : ND + 2;
    const double gm1 = GAM - 1;
    double P[2][NA], t[2][NA] = {{0}}, n[ND];
    flouhip::svjp::node_inputs<ND, TP, 1>(P[0], q1, gm1);
    flouhip::svjp::node_inputs<ND, TP, 1>(P[1], q2, gm1);
    for (int k = 0; k < ND; ++k) n[k] = 0.5 * n1[k] + 0.5 * n2[k];
    const double da = P[0][0] - P[1][0], sa = P[0][0] + P[1][0];
    const double db = P[0][ND + 1] - P[1][ND + 1], sb = P[0][ND + 1] + P[1][ND + 1];
    const double w = TP == flouhip::TP_STDAVG ? 0.5 : 1.0;
    if (TP != flouhip::TP_CHANDRASEKHAR || (da * da < 0.0099 * sa * sa && db * db < 0.0099 * sb * sb))
        flouhip::svjp::pair_vjp<ND, TP, true, true>(P[0], P[1], G, n, w, 1 / gm1, t[0], t[1]);
    else
        flouhip::svjp::pair_vjp<ND, TP, false, true>(P[0], P[1], G, n, w, 1 / gm1, t[0], t[1]);
    for (int s = 0; s < 2; ++s) flouhip::svjp::node_pullback<ND, TP, 1>(P[s], t[s], gm1, b[s]);
}

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
    const double lo[5] = {1, 1.25, 1.5, 2.5, 10}, hi[5] = {1.1, 1.4, 2.2, 7.5, 100};
    for (int metric = 0; metric < 2; ++metric)
        for (int ratio = 0; ratio < 5; ++ratio)
            for (int inverse = 0; inverse < 2; ++inverse) {
                double so[3] = {0}, sk[3] = {0};
                for (int it = 0; it < 60000; ++it) {
                    double q1[5], q2[5], n1[3], n2[3], G[5], O[2][5], K[2][5];
                    LD X[2][5];
                    const double r = 1 / U(1 / hi[ratio], 1 / lo[ratio]), s1 = U(1, 10), s2 = U(0.1, 10);
                    double r1 = s1 * U(0.99, 1.01), r2 = s1 * r * U(0.99, 1.01);
                    double p1 = s2 * U(0.99, 1.01), p2 = s2 * (inverse ? 1 / r : r) * U(0.99, 1.01);
                    if (U(0, 1) < 0.5) { std::swap(r1, r2); std::swap(p1, p2); }
                    state<ND>(q1, r1, p1);
                    state<ND>(q2, r2, p2);
                    for (int k = 0; k < ND; ++k) {  // any direction, or the line's own dominates its metric
                        n1[k] = metric == 0 ? U(-1, 1) : (k == 0 ? U(0.9, 1.1) : 0.05 * U(-1, 1));
                        n2[k] = n1[k] * U(0.9, 1.1);
                    }
                    const double u = std::sqrt(std::max(p1 / r1, p2 / r2));
                    G[0] = U(-1, 1);
                    for (int k = 0; k < ND; ++k) G[1 + k] = U(-1, 1) / u;
                    G[ND + 1] = U(-1, 1) / (u * u);
                    general<LD, ND, TP>(q1, q2, n1, n2, G, X);
                    general<double, ND, TP>(q1, q2, n1, n2, G, O);
                    line<ND, TP>(q1, q2, n1, n2, G, K);
                    for (int s = 0; s < 2; ++s)
                        for (int v = 0; v < ND + 2; ++v) {
                            const int c = v == 0 ? 0 : (v <= ND ? 1 : 2);
                            const double scale = c == 0 ? u : (c == 1 ? 1 : 1 / u);
                            const double eo = (double)((O[s][v] - X[s][v]) / scale);
                            const double ek = (double)((K[s][v] - X[s][v]) / scale);
                            so[c] += eo * eo;
                            sk[c] += ek * ek;
                        }
                }
                std::printf("%d %d %d %g-%g %d %.4f %.4f %.4f\n", ND, TP, metric, lo[ratio], hi[ratio], inverse,
                            std::sqrt(sk[0] / so[0]), std::sqrt(sk[1] / so[1]), std::sqrt(sk[2] / so[2]));
            }
}

int main() {
    errors<2, flouhip::TP_STDAVG>();
    errors<2, flouhip::TP_CHANDRASEKHAR>();
    errors<2, flouhip::TP_KENNEDY_GRUBER>();
    errors<3, flouhip::TP_STDAVG>();
    errors<3, flouhip::TP_CHANDRASEKHAR>();
    errors<3, flouhip::TP_KENNEDY_GRUBER>();
}
