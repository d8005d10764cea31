// FP64 adjoint of the split-form Euler rhs on axis-aligned affine and curved elements (GLL nodes,
// Chandrasekhar, Kennedy-Gruber or StdAverage two-point flux, StdAverage or LxF(StdAverage)
// surface flux), 2-D and 3-D, with the reverse RK stage epilogue: VjpArgs of common.hpp, the
// products of k_vjp (vjp_plain.hip) up to rounding.
//
// What bounds it: FP64 arithmetic and, on small states, HBM.  k_vjp gives a thread to every
// node; it differentiates pairs along full metric vectors and hands the partner's side over
// through an LDS table (1859 VALU per wave of 64 nodes at 2-D N=5).  Here a thread takes a line:
//   * each pair of the line is recomputed and differentiated once, both sides accumulated in
//     registers; no table, and one wave runs lines of one direction, so that the direction, the
//     LDS strides and the line frame (normal velocity first) are compile-time constants;
//   * off the (zero) diagonal S_ij = ω_i D♯_ij is antisymmetric (SBP), so the cotangent of the
//     pair flux F♯(i, j), -D♯_ij w_i - D♯_ji w_j, is S_ij (w_j/ω_j - w_i/ω_i);
//   * the metric Ja_dd scales the line's result, not every pair's normal;
//   * cotangents are those of the halved node inputs, pulled back to (ρ, m, E) once per node;
//   * the face flux is differentiated with respect to the own trace only, by the line that
//     ends there.
// Curved elements (CURV): the pair's flux along the mean metric, which lies in LDS for all
// directions, in physical components; normals per face node.
// LDS: the node inputs and w = c·Y/J; the rows of the directions are added, one direction after
// the other, over w.  Measured, Chandrasekhar, rhs_vjp: 2-D N=5, 0.59 M nodes: 55 -> 40 us;
// 3-D N=5, 1.7 M nodes: 271 -> 184 us; 3-D N=7, 0.5 M nodes: 238 -> 72 us;
// curved 3-D N=6, 0.6 M nodes: 146 -> 87 us.
// Compile with -DFLOUHIP_ND=2|3.
#include "common.hpp"
#include "adjoint.hpp"
#include "pair_vjp.hpp"
#include "stage.hpp"
#include <type_traits>

namespace flouhip {
namespace svjp {

using adj::rcp;

// Elements per block: the lines of one direction fill whole waves (3-D N=6 of 7 nodes: 49 of
// 64 lanes, N=5: 108 of 128); 2-D N=7 leaves 8 lanes for a third block per CU (Kennedy-Gruber, 4624
// elements: 27.6 -> 18.7 us).
template <int ND, int N, bool CURV>
constexpr int epb() {
    if (CURV && ND == 3) return N == 4 ? 4 : (N == 5 ? 2 : 1);  // nine metric values per node beside them
    return ND == 2 ? (N == 8 ? 7 : 64 / N) : (N == 4 ? 4 : (N == 5 ? 5 : (N == 6 ? 3 : 1)));
}

// LDS rows are padded where lines of N nodes pile up on few banks (2-D, 16384 elements,
// Kennedy-Gruber, rhs_vjp without and with: lines of 4 nodes 14.1 and 11.8 us, of 8 79.3 and
// 59.2); lines of 6 nodes lose more by the block per CU that the padding costs (32.6 and 37.4).
template <int ND, int N>
using Nodes = NodeLds<ND, N, N == 4 || N == 8>;

template <int ND, int N, int TP, bool CURV>
struct LCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND, NV = ND + 2;
    static constexpr int EPB = epb<ND, N, CURV>();
    static constexpr int NN = EPB * Nodes<ND, N>::ES;  // LDS nodes per block
    static constexpr int NL = EPB * NPF;                 // lines per block and direction
    static constexpr int WPD = (NL + 63) / 64;           // waves per direction
    // a fourth wave for the node phases where the lines fill their three (3-D N=3, 2 M nodes: 157 ->
    // 150 us, N=7: 277 -> 261; not N=6, 49 of 64 lanes: 205 -> 209)
    static constexpr int TPB = (ND * WPD == 3 && NL % 64 == 0 ? 4 : ND * WPD) * 64;
    static constexpr int NA = TP == TP_KENNEDY_GRUBER ? ND + 3 : ND + 2;  // node inputs = line rows
};

// One side of the face flux along n (CURV; else along the first axis of the state's frame): its
// state with what the products need.
template <int ND, bool CURV>
struct Side {
    double ir, u[ND], uu, un, p, c, a;
    __device__ __forceinline__ Side(const double* R, const double* n, double gamma) {
        ir = rcp(R[0]);
        uu = 0;
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            u[k] = R[1 + k] * ir;
            uu = fma(u[k], u[k], uu);
        }
        p = (gamma - 1) * fma(-0.5 * R[0], uu, R[ND + 1]);
        c = sqrt(gamma * p * ir);
        un = u[0];
        if constexpr (CURV) {
            un = u[0] * n[0];
#pragma unroll
            for (int k = 1; k < ND; ++k) un = fma(u[k], n[k], un);
        }
        a = fabs(un) + c;
    }
    // Adds to b the product of f(R)·n for the cotangent G and lb times the gradient of a.
    __device__ __forceinline__ void add(const double* R, const double* G, const double* n, double gamma, double lb,
                                        double* b) const {
        constexpr int NV = ND + 2;
        const double g1 = gamma - 1;
        double gn = G[1];
        if constexpr (CURV) {
            gn = G[1] * n[0];
#pragma unroll
            for (int k = 1; k < ND; ++k) gn = fma(G[1 + k], n[k], gn);
        }
        double unb = G[NV - 1] * (R[NV - 1] + p);
#pragma unroll
        for (int k = 0; k < ND; ++k) unb = fma(G[1 + k], R[1 + k], unb);
        unb += lb * (un > 0 ? 1.0 : (un < 0 ? -1.0 : 0.0));
        const double cb = lb == 0 ? 0.0 : 0.5 * lb * rcp(c);  // of c²
        const double pg = g1 * (fma(G[NV - 1], un, gn) + cb * gamma * ir);
        const double uir = unb * ir;
        b[0] += -uir * un + 0.5 * pg * uu - cb * c * c * ir;
#pragma unroll
        for (int k = 0; k < ND; ++k)
            b[1 + k] += fma(G[1 + k], un, fma(-pg, u[k], CURV ? (G[0] + uir) * n[k] : (k == 0 ? G[0] + uir : 0.0)));
        b[NV - 1] += fma(G[NV - 1], un, pg);
    }
};

// The momentum m with its normal part reversed.
template <int ND, bool CURV>
__device__ __forceinline__ void mirror(double* m, const double* n) {
    if constexpr (CURV) {
        double mn = m[0] * n[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) mn = fma(m[k], n[k], mn);
#pragma unroll
        for (int k = 0; k < ND; ++k) m[k] = fma(-2 * mn, n[k], m[k]);
    } else {
        m[0] = -m[0];
    }
}

// A wave's lines of direction DIR.  Component k of a vector in the line frame is physical
// component (DIR + k) % ND; on curved elements (sM: half the metric rows) it is k.
template <int ND, int N, int TP, bool CURV, int DIR>
__device__ __forceinline__ void line_phase(const VjpArgs<double>& A, const double* sP, const double* sM, double* sW,
                                           double* sT, const double* sS, const double* siw, int e0, int nel, int l,
                                           double (&acc)[N][LCfg<ND, N, TP, CURV>::NA]) {
    using C = LCfg<ND, N, TP, CURV>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, NN = C::NN, NA = C::NA;
    using M = Nodes<ND, N>;
    constexpr int ST = M::template step<DIR>();
    constexpr int GST = DIR == 0 ? 1 : (DIR == 1 ? N : N * N);  // step along the line in the state
    const RhsArgs<double>& a = A.r;
    const bool task = l < C::NL && l / NPF < nel;
    const int le = task ? l / NPF : 0, f = l % NPF;
    const int base = le * M::ES + M::template line<DIR>(f);
    const double ja = CURV ? 1.0 : a.egeom[(int64_t)(e0 + le) * a.egeom_stride + DIR * (ND + 1)];
    const double gamma = a.gamma, ig1 = 1 / (gamma - 1);
    int vo[ND];  // physical variable of line-frame momentum k
#pragma unroll
    for (int k = 0; k < ND; ++k) vo[k] = CURV ? 1 + k : 1 + (DIR + k) % ND;

    // ---- faces at the two line ends: cotangent of the own trace ------------------------
    if (task) {
#pragma unroll
        for (int sd = 0; sd < 2; ++sd) {
            const int slot = (e0 + le) * NF + 2 * DIR + sd;
            const int info = a.finfo[slot], nb = a.nb[slot];
            const double* g = a.fgeom + ((int64_t)a.fgi[slot] * (CURV ? NPF : 1) +
                                         (CURV ? face_master_node<ND, N>(f, info) : 0)) * (3 * ND + 1);
            const bool slave = finfo_side(info);
            const double so = slave ? -g[DIR] : g[DIR];   // own outward normal along the axis
            double n[ND];                                 // CURV: the own outward normal
#pragma unroll
            for (int k = 0; k < ND; ++k) n[k] = slave ? -g[k] : g[k];
            const int64_t on = (int64_t)(e0 + le) * NPE + line_node<ND, N>(DIR, f, 0) + (sd ? (N - 1) * GST : 0);
            double o[NV], x[NV], G[NV], ob[NV], xb[NV];
            o[0] = a.Q[on];
            o[NV - 1] = a.Q[(NV - 1) * a.ndofs + on];
#pragma unroll
            for (int k = 0; k < ND; ++k) o[1 + k] = a.Q[vo[k] * a.ndofs + on];
            // S̄ = ½·jac·(-∂g_own w_own + ∂g_nb w_nb), of (f_o + f_x)·n + λ·diss·(o - x)
            const double h = 0.5 * g[3 * ND];
            const double co = h * (sd ? a.ops[ops_gp(N) + N - 1] : a.ops[ops_gm(N)]);
            const int ol = base + (sd ? (N - 1) * ST : 0);
            G[0] = -co * sW[ol];
            G[NV - 1] = -co * sW[(NV - 1) * NN + ol];
#pragma unroll
            for (int k = 0; k < ND; ++k) G[1 + k] = -co * sW[vo[k] * NN + ol];
            int type = -1;
            if (nb >= 0) {
                const int kp = finfo_nbpos(info);
                const int64_t nn = (int64_t)nb * NPE +
                                   line_node<ND, N>(CURV ? kp >> 1 : DIR, CURV ? face_nb_node<ND, N>(f, info) : f,
                                                    (kp & 1) ? N - 1 : 0);
                const double cn = h * ((kp & 1) ? a.ops[ops_gp(N) + N - 1] : a.ops[ops_gm(N)]) *
                                  (A.c / (CURV ? a.ngeom[ND * ND * a.ndofs + nn]
                                               : a.egeom[(int64_t)nb * a.egeom_stride + ND * ND]));
                x[0] = a.Q[nn];
                x[NV - 1] = a.Q[(NV - 1) * a.ndofs + nn];
                G[0] = fma(cn, A.Y[nn], G[0]);
                G[NV - 1] = fma(cn, A.Y[(NV - 1) * a.ndofs + nn], G[NV - 1]);
#pragma unroll
                for (int k = 0; k < ND; ++k) {
                    x[1 + k] = a.Q[vo[k] * a.ndofs + nn];
                    G[1 + k] = fma(cn, A.Y[vo[k] * a.ndofs + nn], G[1 + k]);
                }
            } else {
                const int bd = finfo_bd(info);
                type = a.bctype[bd];
                const double* src = type == BC_DIRICHLET ? a.bcstate + ((int64_t)a.fid[slot] * NPF + f) * NV
                                                         : a.bcconst + bd * NV;
                const bool given = type == BC_DIRICHLET || type == BC_INFLOW;
                x[0] = given ? src[0] : o[0];
                x[NV - 1] = given ? src[NV - 1] : o[NV - 1];
#pragma unroll
                for (int k = 0; k < ND; ++k) x[1 + k] = given ? src[vo[k]] : o[1 + k];
                if (type == BC_SLIP) mirror<ND, CURV>(x + 1, n);
            }
            if constexpr (!CURV) {  // frame of the own outward normal
                o[1] *= so;
                x[1] *= so;
                G[1] *= so;
            }
            const Side<ND, CURV> S(o, n, gamma), X(x, n, gamma);
            double lo = 0, lx = 0, dl = 0;
#pragma unroll
            for (int v = 0; v < NV; ++v) ob[v] = xb[v] = 0;
            if (a.sdiss == DISS_LXF) {
                // λ's derivative goes to the side that the forward's maximum keeps, the master on ties
                const bool mine = slave ? X.a < S.a : !(S.a < X.a);
                const double lam = (mine ? S.a : X.a) * a.intensity;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    ob[v] = lam * G[v];
                    xb[v] = -lam * G[v];
                    dl = fma(o[v] - x[v], G[v], dl);
                }
                dl *= a.intensity;
                lo = mine ? dl : 0;
                lx = mine ? 0 : dl;
            }
            S.add(o, G, n, gamma, lo, ob);
            if (type == BC_OUTFLOW || type == BC_SLIP) {  // the exterior state follows the own trace
                X.add(x, G, n, gamma, lx, xb);
                if (type == BC_SLIP) mirror<ND, CURV>(xb + 1, n);
#pragma unroll
                for (int v = 0; v < NV; ++v) ob[v] += xb[v];
            }
            if constexpr (!CURV) ob[1] *= so;
            double* t = sT + ((le * NF + 2 * DIR + sd) * NV) * NPF + f;
            t[0] = ob[0];
            t[(NV - 1) * NPF] = ob[NV - 1];
#pragma unroll
            for (int k = 0; k < ND; ++k) t[vo[k] * NPF] = ob[1 + k];
        }
    }

    // ---- the line's pairs ----------------------------------------------------------------
    auto load = [&](int base, int p, double* P, double* W) {
        const double* s = sP + base + p * ST;
        const double* w = sW + base + p * ST;
        if constexpr (TP == TP_STDAVG) {  // u.., H, |u|²
#pragma unroll
            for (int k = 0; k < ND; ++k) P[k] = s[(vo[k] - 1) * NN];
            P[ND] = s[ND * NN];
            P[ND + 1] = s[(ND + 1) * NN];
        } else {
            P[0] = s[0];
#pragma unroll
            for (int k = 0; k < ND; ++k) P[1 + k] = s[vo[k] * NN];
#pragma unroll
            for (int c = ND + 1; c < NA; ++c) P[c] = s[c * NN];
        }
        W[0] = w[0];
#pragma unroll
        for (int k = 0; k < ND; ++k) W[1 + k] = w[vo[k] * NN];
        W[NV - 1] = w[(NV - 1) * NN];
    };
    auto metric = [&](int base, int p, double* n) {
        const double* s = sM + base + p * ST;
#pragma unroll
        for (int k = 0; k < ND; ++k) n[k] = s[(ND * DIR + k) * NN];
    };
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int c = 0; c < NA; ++c) acc[p][c] = 0;
    if constexpr (TP == TP_STDAVG && !CURV) {
        // the flux is a sum of node terms: each node takes the reverse product of ½ f(Q)·n̄ for
        // Σ_j S_ij (w_j/ω_j - w_i/ω_i)
#pragma unroll
        for (int i = 0; i < N; ++i) {
            double P[NA], wi[NV];
            load(base, i, P, wi);
#pragma unroll
            for (int v = 0; v < NV; ++v) wi[v] *= siw[i];
#pragma unroll
            for (int j = i + 1; j < N; ++j) {
                const double* w = sW + base + j * ST;
                const double s = sS[i * N + j], iw = siw[j];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const int pv = v == 0 || v == NV - 1 ? v : vo[v >= 1 && v <= ND ? v - 1 : 0];
                    const double g = fma(w[pv * NN], iw, -wi[v]);
                    acc[i][v] = fma(s, g, acc[i][v]);
                    acc[j][v] = fma(s, g, acc[j][v]);
                }
            }
        }
        const double h = 0.5 * ja;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            double P[NA], w[NV], G[NV];
            load(base, i, P, w);
#pragma unroll
            for (int v = 0; v < NV; ++v) G[v] = h * acc[i][v];
            double U = G[1] * P[0];
#pragma unroll
            for (int k = 1; k < ND; ++k) U = fma(G[1 + k], P[k], U);
            U = fma(G[NV - 1], P[ND], U);
            const double un = P[0], pg = (gamma - 1) * fma(G[NV - 1], un, G[1]);
            acc[i][0] = fma(-U, un, 0.5 * pg * P[ND + 1]);
#pragma unroll
            for (int k = 0; k < ND; ++k) acc[i][1 + k] = fma(G[1 + k], un, fma(-pg, P[k], k == 0 ? G[0] + U : 0.0));
            acc[i][NV - 1] = fma(G[NV - 1], un, pg);
        }
    } else {
        auto pairs = [&, base0 = base](auto series) {
            // The address is opaque from here, so that the two forms of the pairs share no loads (their
            // values stayed live over the whole line: 256 registers and a wave per SIMD at 3-D N=7, 4096
            // elements 257 -> 168 us; curved 3-D N=6 likewise)
            int base = base0;
            if constexpr (TP == TP_CHANDRASEKHAR) asm volatile("" : "+v"(base));
#pragma unroll
            for (int i = 0; i < N; ++i) {
                double P[NA], wi[NV], ni[ND];
                load(base, i, P, wi);
                if constexpr (CURV) metric(base, i, ni);
#pragma unroll
                for (int v = 0; v < NV; ++v) wi[v] *= siw[i];
#pragma unroll
                for (int j = i + 1; j < N; ++j) {
                    double Q[NA], G[NV], n[ND];
                    load(base, j, Q, G);
                    if constexpr (CURV) {
                        metric(base, j, n);
#pragma unroll
                        for (int k = 0; k < ND; ++k) n[k] += ni[k];
                    }
                    const double iw = siw[j];
#pragma unroll
                    for (int v = 0; v < NV; ++v) G[v] = fma(G[v], iw, -wi[v]);
                    pair_vjp<ND, TP, decltype(series)::value, CURV>(P, Q, G, n,
                                                                    sS[i * N + j] * (TP == TP_STDAVG ? 0.5 : ja), ig1,
                                                                    acc[i], acc[j]);
                    // one pair's loads and arithmetic at a time: the registers hold the rows,
                    // node i and one pair
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        if constexpr (TP == TP_CHANDRASEKHAR) {
            // the series for every pair of the wave's lines when the spreads of ρ and β along
            // each line allow it (u of its extreme values below 0.01), else the general form
            double amax = sP[base], amin = amax, bmax = sP[(ND + 1) * NN + base], bmin = bmax;
#pragma unroll
            for (int p = 1; p < N; ++p) {
                const double x = sP[base + p * ST], y = sP[(ND + 1) * NN + base + p * ST];
                amax = fmax(amax, x); amin = fmin(amin, x);
                bmax = fmax(bmax, y); bmin = fmin(bmin, y);
            }
            const double da = amax - amin, sa = amax + amin, db = bmax - bmin, sb = bmax + bmin;
            const bool near = da * da < 0.01 * (1 - 1e-12) * sa * sa && db * db < 0.01 * (1 - 1e-12) * sb * sb;
            if (__all(!task || near)) pairs(std::true_type());
            else pairs(std::false_type());
        } else {
            pairs(std::true_type());
        }
    }
    // (the rows are pinned here: their use below is conditional, and the pairs would sink into it)
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int c = 0; c < NA; ++c) asm volatile("" : "+v"(acc[p][c]));
}

// Adds (direction 0: writes) a line's rows to the nodes' sums, in physical component order.
template <int ND, int N, int TP, bool CURV, int DIR>
__device__ __forceinline__ void add_rows(double* sR, int nel, int l, const double (&acc)[N][LCfg<ND, N, TP, CURV>::NA]) {
    using C = LCfg<ND, N, TP, CURV>;
    using M = Nodes<ND, N>;
    constexpr int ST = M::template step<DIR>();
    if (l >= C::NL || l / C::NPF >= nel) return;
    double* r = sR + (l / C::NPF) * M::ES + M::template line<DIR>(l % C::NPF);
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int c = 0; c < C::NA; ++c) {
            const int pc = !CURV && c >= 1 && c <= ND ? 1 + (DIR + c - 1) % ND : c;
            double* x = r + pc * C::NN + p * ST;
            *x = DIR == 0 ? acc[p][c] : *x + acc[p][c];
        }
}

template <int ND, int N, int TP, bool CURV>
__global__ void __launch_bounds__((LCfg<ND, N, TP, CURV>::TPB)) k_svjp(const VjpArgs<double> A) {
    using C = LCfg<ND, N, TP, CURV>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN, NA = C::NA;
    __shared__ double sP[NA * NN];                       // node inputs
    __shared__ double sW[(NA > NV ? NA : NV) * NN];      // w = c·Y/J, then the sums of the rows
    __shared__ double sT[EPB * NF * NV * NPF];           // cotangents of the own traces
    __shared__ double sM[CURV ? ND * ND * NN : 1];       // CURV: half the metric, component-major
    __shared__ double sS[N * N], siw[N];
    const RhsArgs<double>& a = A.r;
    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs, g0 = (int64_t)e0 * NPE;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const int nnb = nel * NPE;
    const double gamma = a.gamma, gm1 = a.gamma - 1;

    // The loads of all the thread's nodes come first (BATCH; spare threads load the block's first
    // node): 2-D N=7, 40,000 elements, Chandrasekhar 141 -> 134 us; 3-D N=5, 4096 elements 103.5 -> 105.8,
    // where they come node by node.
    constexpr int NPT = (EPB * NPE + TPB - 1) / TPB;
    constexpr bool BATCH = ND == 2 || N >= 7;
    constexpr int NB = BATCH ? NPT : 1;
    double q_[NB][NV], y_[NB][NV], j_[NB], m_[CURV ? NB : 1][CURV ? ND * ND : 1];
    auto state = [&](int t, int b) {
        const int j = tid + t * TPB < nnb ? tid + t * TPB : 0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            q_[b][v] = (a.Q + (v * Nd + g0))[j];
            y_[b][v] = (A.Y + (v * Nd + g0))[j];
        }
        j_[b] = CURV ? (a.ngeom + (ND * ND * Nd + g0))[j] : a.egeom[(int64_t)(e0 + j / NPE) * a.egeom_stride + ND * ND];
        if constexpr (CURV) {
#pragma unroll
            for (int c = 0; c < ND * ND; ++c) m_[b][c] = (a.ngeom + (c * Nd + g0))[j];
        }
    };
    if constexpr (BATCH) {
#pragma unroll
        for (int t = 0; t < NPT; ++t) state(t, t);
    }
    for (int i = tid; i < N * N; i += TPB) {
        const int r = i / N, c = i - r * N;
        const double* w = a.ops + ops_w(N);
        const double* D = a.ops + ops_Dsh(N);
        sS[i] = 0.5 * (w[r] * D[i] - w[c] * D[c * N + r]);
    }
    for (int i = tid; i < N; i += TPB) siw[i] = 1 / a.ops[ops_w(N) + i];
#pragma unroll
    for (int t = 0; t < NPT; ++t) {
        const int j = tid + t * TPB;
        if (j >= nnb) break;
        const int jj = Nodes<ND, N>::node(j);
        const int b = BATCH ? t : 0;
        if constexpr (!BATCH) state(t, 0);
        const double* const q = q_[b];
        const double* const y = y_[b];
        const double cj = A.c / j_[b];
        if constexpr (CURV) {
#pragma unroll
            for (int c = 0; c < ND * ND; ++c) sM[c * NN + jj] = 0.5 * m_[b][c];
        }
        node_inputs<ND, TP, NN>(sP + jj, q, gm1);
#pragma unroll
        for (int v = 0; v < NV; ++v) sW[v * NN + jj] = cj * y[v];
    }
    __syncthreads();

    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int dir = wave / C::WPD;
    const int l = dir < ND ? (wave - dir * C::WPD) * 64 + (tid & 63) : C::NL;
    double acc[N][NA];
    if (dir == 0) line_phase<ND, N, TP, CURV, 0>(A, sP, sM, sW, sT, sS, siw, e0, nel, l, acc);
    else if (ND == 2 || dir == 1) line_phase<ND, N, TP, CURV, 1>(A, sP, sM, sW, sT, sS, siw, e0, nel, l, acc);
    else if (dir == ND - 1) line_phase<ND, N, TP, CURV, ND - 1>(A, sP, sM, sW, sT, sS, siw, e0, nel, l, acc);
    __syncthreads();  // w has been read
    if (dir == 0) add_rows<ND, N, TP, CURV, 0>(sW, nel, l, acc);
    __syncthreads();
    if (dir == 1) add_rows<ND, N, TP, CURV, 1>(sW, nel, l, acc);
    __syncthreads();
    if constexpr (ND == 3) {
        if (dir == 2) add_rows<ND, N, TP, CURV, 2>(sW, nel, l, acc);
        __syncthreads();
    }

    // ---- per node: pullback of the inputs, face terms, epilogue (its operands first) ------------
    double p_[3][NB][NV];
    auto operands = [&](int t, int b) {
        const int j = tid + t * TPB < nnb ? tid + t * TPB : 0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            p_[0][b][v] = A.P0 ? (A.P0 + (v * Nd + g0))[j] : 0.0;
            p_[1][b][v] = A.P1 ? (A.P1 + (v * Nd + g0))[j] : 0.0;
            p_[2][b][v] = A.P2 ? (A.P2 + (v * Nd + g0))[j] : 0.0;
        }
    };
    if constexpr (BATCH) {
#pragma unroll
        for (int t = 0; t < NPT; ++t) operands(t, t);
    }
#pragma unroll
    for (int it = 0; it < NPT; ++it) {
        const int j = tid + it * TPB;
        if (j >= nnb) break;
        const int jj = Nodes<ND, N>::node(j);
        double t[NA], V[NV];
#pragma unroll
        for (int c = 0; c < NA; ++c) t[c] = sW[c * NN + jj];
        node_pullback<ND, TP, NN>(sP + jj, t, gm1, V);
        const int le = j / NPE, node = j - le * NPE;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            int f, pos;
            node_line<ND, N>(node, d, f, pos);
            if (pos == 0 || pos == N - 1) {
                const double* F = sT + ((le * NF + 2 * d + (pos == 0 ? 0 : 1)) * NV) * NPF + f;
#pragma unroll
                for (int v = 0; v < NV; ++v) V[v] += F[v * NPF];
            }
        }
        const int b = BATCH ? it : 0;
        if constexpr (!BATCH) operands(it, 0);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t i = v * Nd + g0 + j;
            const double o = V[v] + A.a0 * p_[0][b][v] + A.a1 * p_[1][b][v];
            if (A.o1) A.o1[i] = A.b0 * o + A.b1 * p_[1][b][v] + A.b2 * p_[2][b][v];
            A.o0[i] = o;
        }
    }
}

template <int ND, int N, int TP, bool CURV>
static hipError_t launch(const VjpArgs<double>& a, hipStream_t s) {
    using C = LCfg<ND, N, TP, CURV>;
    hipLaunchKernelGGL((k_svjp<ND, N, TP, CURV>), dim3((a.r.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

// (curved 2-D: not where the general kernel is as fast, see flou_hip_create)
template <int ND, int N, bool CURV>
static VjpLauncherF64 pick_tp(int tp) {
    if constexpr (CURV && ND == 2 && N == 8) {
        return nullptr;
    } else {
        switch (tp) {
            case TP_STDAVG: return &launch<ND, N, TP_STDAVG, CURV>;
            case TP_CHANDRASEKHAR: return &launch<ND, N, TP_CHANDRASEKHAR, CURV>;
            case TP_KENNEDY_GRUBER:
                if constexpr (CURV && ND == 2 && (N == 5 || N == 7)) return nullptr;
                else return &launch<ND, N, TP_KENNEDY_GRUBER, CURV>;
            default: return nullptr;
        }
    }
}

}  // namespace svjp

#define FLOUHIP_CAT_(a, b) a##b
#define FLOUHIP_CAT(a, b) FLOUHIP_CAT_(a, b)

VjpLauncherF64 FLOUHIP_CAT(split_vjp_f64_, FLOUHIP_ND)(int n, int tp, bool curved) {
    switch (n) {
        case 4: return curved ? svjp::pick_tp<FLOUHIP_ND, 4, true>(tp) : svjp::pick_tp<FLOUHIP_ND, 4, false>(tp);
        case 5: return curved ? svjp::pick_tp<FLOUHIP_ND, 5, true>(tp) : svjp::pick_tp<FLOUHIP_ND, 5, false>(tp);
        case 6: return curved ? svjp::pick_tp<FLOUHIP_ND, 6, true>(tp) : svjp::pick_tp<FLOUHIP_ND, 6, false>(tp);
        case 7: return curved ? svjp::pick_tp<FLOUHIP_ND, 7, true>(tp) : svjp::pick_tp<FLOUHIP_ND, 7, false>(tp);
        case 8: return curved ? svjp::pick_tp<FLOUHIP_ND, 8, true>(tp) : svjp::pick_tp<FLOUHIP_ND, 8, false>(tp);
        default: return nullptr;
    }
}

}  // namespace flouhip
