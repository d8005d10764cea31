// FP64 split-form Euler rhs on axis-aligned affine elements (Flou's CartesianMesh), GLL
// nodes, StdAverage or LxF(StdAverage) surface flux, with the RK stage epilogue: the plain
// kernel's arithmetic (rhs_plain.hip, reference order, every value rounded where the
// reference rounds it) without the work that this geometry makes void.
//
// What bounds it: FP64 arithmetic, by issue (90 % of busy cycles) and by the clock the power
// limit leaves under it (1.8 to 2.0 of 2.4 GHz).  k_plain<double, 3, 6, ..> spends about 4000
// VALU slots per node, most of them on divisions, on the two components of every flux that a
// diagonal metric multiplies by zero, and on rotations by 0 and ±1.  Measured against it (same
// bits): 3-D N=5, 10.5 M nodes, Chandrasekhar: 1.65 -> 0.90 ms per CK2N54 stage; 2-D N=5, 0.59 M
// nodes: 66 -> 40 us.  With the same results:
//   * only the flux component along the line's direction is formed: f·n̄ has one term, the
//     others are exact zeros.  The direction is a compile-time constant of each phase;
//   * flux inputs are staged halved, so that means are one addition (pair_flux);
//   * a node's own contravariant flux goes into the same table as the pairs, so that its row
//     reads N entries without a case for the diagonal, at offsets that advance by constants
//     (2504 -> 2186 VALU per wave at 3-D N=5 with the above, 2084 with all that follows);
//   * face states are read in the order of the face frame by index (faces.hpp);
//   * quotients share reciprocals (exact_div.hpp), the node's contravariant flux reuses its
//     primitives, the lift touches the end nodes only (∂g is exactly zero elsewhere);
//   * loads are unconditional, spare lanes and boundary faces loading something valid (branches
//     around each load: 3-D 4 nodes per line 80.9 -> 74.7 us, 2-D 8 nodes 26.8 -> 25.8);
//   * the face fluxes come last and lie over the dead table (39 KB of LDS at 3-D N=5, 4 waves
//     per SIMD); their neighbour traces are loaded before the last direction's rows.
// One thread per node (blocks rounded up to whole waves, the spare lanes take pairs), pairs
// pair-major: consecutive lanes evaluate the same pair of consecutive lines, so node reads
// and table writes are conflict-light and the pair's positions nearly uniform.
// Compile with -DFLOUHIP_ND=1|2|3.
#include "common.hpp"
#include "faces.hpp"
#include "pair_along.hpp"
#include "physics_plain.hpp"
#include "stage.hpp"

namespace flouhip {
namespace split {

// LDS rows are padded where lines of N nodes pile up on few banks (Kennedy-Gruber, 0.6 M nodes in
// 2-D, 1 M in 3-D, without and with: 2-D lines of 4 nodes 25.8 and 22.0 us, of 6 31.7 and 26.2, of
// 8 48.8 and 28.5; 3-D of 4 62 and 60, of 8 127 and 100); not for 2 nodes, nor 6 in 3-D (no gain).
template <int ND, int N>
using Nodes = NodeLds<ND, N, N == 4 || N == 8 || (ND == 2 && N == 6)>;

template <int ND, int N>
struct SCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND, NV = ND + 2;
    // Elements per block: two waves where their nodes and pairs fill whole waves (2-D N=4: 5
    // elements of 25 nodes against 10: CFL run of 2623 elements 289 -> 259 us; more, smaller
    // blocks wait less at barriers and spread evenly over the CUs), else the count up to 256
    // threads that does (2-D N=5: 7; 5 elements: gradient 1360 -> 1374 us).  3-D N=5 runs one
    // element (216 of 256 lanes; two, 432 of 448: CK2N54 step 4698 -> 5145 us).
    static constexpr int EPB = NPE > 128 ? 1 : (ND == 2 && N == 6 ? 7 : (ND == 2 && N == 7 ? 5 : 128 / NPE));
    static constexpr int NN = EPB * NPE;                 // nodes per block
    static constexpr int TPB = block_threads(NN);        // threads per block
    static constexpr int NPAIR = N * (N - 1) / 2;
    static constexpr int NPR = EPB * NPF * NPAIR;        // pairs per block and direction
    static constexpr int NL = EPB * NPF;                 // lines per block and direction
    static constexpr int SN = EPB * Nodes<ND, N>::ES;  // LDS nodes per block
    // The table: pair fluxes of line l at pr·NLP + l, then the nodes' own; entry k, variable v at
    // k·KS + v·VS.  2-D (4 variables) keeps a plane per variable with an odd line count, so that
    // neither the pairs' writes nor the rows' reads pile up on few banks.
    static constexpr int NLP = ND == 2 ? NL | 1 : NL;
    static constexpr int TAB = NPAIR * NLP + NN;
    static constexpr int KS = ND == 2 ? 1 : NV, VS = ND == 2 ? TAB : 1;
};

// One direction: every pair flux and every node's contravariant flux (the diagonal entry of
// F♯) into the table, then after a barrier (before which LOADS may issue global loads) every
// node's D♯ row over it in the order j = 0..N-1.
template <int ND, int N, int TP, int DIR, typename LOADS>
__device__ __forceinline__ void direction(const RhsArgs<double>& a, const double* sS, double* sTab, const double* sD,
                                          const double* sG, int nel, int tid, int le, int node, bool valid,
                                          const double (&q)[ND + 2], const double (&u)[ND], double p, LOADS loads,
                                          double (&acc)[ND + 2]) {
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, SN = C::SN, NL = C::NL, NS = plain::tp_slots<ND, TP>();
    constexpr int KS = C::KS, VS = C::VS, DIAG = C::NPAIR * C::NLP;
    using M = Nodes<ND, N>;
    const double gm1 = a.gamma - 1.0;
    int lf, ii;
    node_line<ND, N>(node, DIR, lf, ii);
    if (valid) {
        // contravariant flux along DIR (plain::contravariant_flux, diagonal metric)
        const double ja = sG[le * (ND + 1) + DIR];
        double* t = sTab + (DIAG + tid) * KS;
        t[0] = q[1 + DIR] * ja;
#pragma unroll
        for (int c = 0; c < ND; ++c) t[(1 + c) * VS] = (c == DIR ? q[1 + DIR] * u[c] + p : q[1 + DIR] * u[c]) * ja;
        t[(NV - 1) * VS] = ((q[NV - 1] + p) * u[DIR]) * ja;
    }
#pragma unroll 1
    for (int k = tid; k < C::NPR; k += C::TPB) {
        const int pr = k / NL, l = k - pr * NL;
        const int le2 = C::EPB == 1 ? 0 : l / NPF, f = l - le2 * NPF;
        if (le2 >= nel) continue;
        const int ab = pair_ab<N>(pr);
        const int base = le2 * M::ES + M::template line<DIR>(f);
        constexpr int ST = M::template step<DIR>();
        const double* pa = sS + base + (ab >> 3) * ST;
        const double* pb = sS + base + (ab & 7) * ST;
        double A[NS], B[NS], F[NV];
#pragma unroll
        for (int c = 0; c < NS; ++c) { A[c] = pa[c * SN]; B[c] = pb[c * SN]; }
        plain::pair_flux<double, ND, TP, DIR>(A, B, sG[le2 * (ND + 1) + DIR], gm1, a.errflag, F);
#pragma unroll
        for (int v = 0; v < NV; ++v) sTab[(pr * C::NLP + l) * KS + v * VS] = F[v];
    }
    loads();
    __syncthreads();
    if (valid) {
        // pair (j, ii) or (ii, j) of the node's line: pair index ii - 1 at j = 0, then N - j - 2
        // further for each j < ii and 1 further from there (the place of j = ii is skipped over)
        const int diag = (DIAG + tid) * KS;
        int off = ((ii - 1) * C::NLP + le * NPF + lf) * KS;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double* t = sTab + (j == ii ? diag : off);
            const double Dij = sD[ii * N + j];
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = acc[v] - Dij * t[v * VS];
            off += (j < ii ? N - j - 2 : 1) * (C::NLP * KS);
        }
    }
    __syncthreads();  // the table has been read
}

template <int ND, int N, int TP>
__global__ void __launch_bounds__((SCfg<ND, N>::TPB)) k_split(const RhsArgs<double> a) {
    using T = double;
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN;
    constexpr int NS = plain::tp_slots<ND, TP>();
    constexpr int NFN = EPB * NF * NPF;  // face nodes of the block
    constexpr int TAB = C::TAB, FACE = NN + NFN;
    __shared__ T sS[NS * C::SN];                       // two-point flux inputs, [slot][node]
    __shared__ T sTab[NV * (TAB > FACE ? TAB : FACE)];  // pair and node fluxes of one direction, then
                                                       // conservative states [v][node] and face fluxes
    __shared__ T sD[N * N];
    __shared__ T sG[EPB * (ND + 1)];                   // Ja_dd and J per element

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const T gamma = a.gamma;

    // ---- own node, face tables, operators -----------------------------------------------
    const int fe = tid / (NF * NPF), fk = (tid - fe * (NF * NPF)) / NPF, ff = tid % NPF;
    const bool pf = tid < NFN && fe < nel;
    // (spare lanes load something valid instead of branching)
    const int pslot = e0 * NF + (pf ? fe * NF + fk : 0);
    const int pinfo = a.finfo[pslot], pnb = a.nb[pslot], pfgi = a.fgi[pslot];
    const bool valid = tid < nel * NPE;
    const int tn = valid ? tid : 0;
    const int le = tid / NPE, node = tid - le * NPE;
    const int64_t g0 = (int64_t)e0 * NPE;
    T q[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = (a.Q + (v * Nd + g0))[tn];
    static_assert(N * N <= TPB && EPB * (ND + 1) <= TPB, "one operator and geometry entry per thread");
    const T Dv = a.ops[ops_Dsh(N) + (tid < N * N ? tid : 0)];
    const int ge = tid / (ND + 1), gc = tid - ge * (ND + 1);
    const T Gv = a.egeom[(int64_t)(e0 + (ge < nel ? ge : 0)) * a.egeom_stride + (gc < ND ? gc * (ND + 1) : ND * ND)];
    T u[ND], p;
    {
        T P[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, gamma, P, ir);
#pragma unroll
        for (int k = 0; k < ND; ++k) u[k] = P[1 + k];
        p = P[ND + 1];
        if (valid) plain::put_slots<T, ND, TP, C::SN>(sS + Nodes<ND, N>::node(tid), q, P, ir);
    }
    if (tid < N * N) sD[tid] = Dv;
    if (tid < EPB * (ND + 1)) sG[tid] = Gv;
    __syncthreads();

    // ---- volume terms, direction by direction ---------------------------------------------
    // The first face node's neighbour trace (in the order ρ, normal and transverse momenta, E)
    // and face data and the epilogue's operand are loaded before the last direction's rows.
    T acc[NV], pext[NV], xv[NV], pn = T(0), pj = T(0);
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    const T* aux = stage_aux(a);
    auto none = []() {};
    auto prefetch = [&]() {
        const int kp = pnb >= 0 ? finfo_nbpos(pinfo) : 0, dir = fk >> 1;
        load_trace<T, ND, NV>(a.Q + (int64_t)(pnb >= 0 ? pnb : e0) * NPE +
                                  line_node<ND, N>(kp >> 1, ff, (kp & 1) ? N - 1 : 0),
                              Nd, dir, pext);
        const T* g = a.fgeom + (int64_t)pfgi * (3 * ND + 1);
        pn = g[dir];
        pj = g[3 * ND];
        if (aux) {
#pragma unroll
            for (int v = 0; v < NV; ++v) xv[v] = (aux + (v * Nd + g0))[tn];
        }
    };
    if constexpr (ND == 1) {
        direction<ND, N, TP, 0>(a, sS, sTab, sD, sG, nel, tid, le, node, valid, q, u, p, prefetch, acc);
    } else {
        direction<ND, N, TP, 0>(a, sS, sTab, sD, sG, nel, tid, le, node, valid, q, u, p, none, acc);
        if constexpr (ND == 3)
            direction<ND, N, TP, 1>(a, sS, sTab, sD, sG, nel, tid, le, node, valid, q, u, p, none, acc);
        direction<ND, N, TP, ND - 1>(a, sS, sTab, sD, sG, nel, tid, le, node, valid, q, u, p, prefetch, acc);
    }

    // ---- numerical fluxes on the element's faces --------------------------------------------
    T* const sU = sTab;
    T* const sFn = sTab + NV * NN;
    if (valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sU[v * NN + tid] = q[v];
    }
    __syncthreads();
    for (int it = tid; it < NFN; it += TPB) {
        const bool first = it == tid;
        const int le2 = it / (NF * NPF), r = it - le2 * (NF * NPF);
        const int k = r / NPF, f = r - k * NPF;
        if (le2 >= nel) continue;
        const int dir = k >> 1;
        const int slot = (e0 + le2) * NF + k;
        const int info = first ? pinfo : a.finfo[slot];
        const int nbe = first ? pnb : a.nb[slot];
        const int on = le2 * NPE + line_node<ND, N>(dir, f, (k & 1) ? N - 1 : 0);
        T own[NV], ext[NV], Fn[NV];
        own[0] = sU[on];
#pragma unroll
        for (int c = 0; c < ND; ++c) own[1 + c] = sU[face_mom<ND>(dir, c) * NN + on];
        own[NV - 1] = sU[(NV - 1) * NN + on];
        T sn = pn, jac = pj;
        if (!first) {
            const T* g = a.fgeom + (int64_t)a.fgi[slot] * (3 * ND + 1);
            sn = g[dir];
            jac = g[3 * ND];
        }
        if (nbe >= 0) {
            if (first) {
#pragma unroll
                for (int v = 0; v < NV; ++v) ext[v] = pext[v];
            } else {
                const int kp = finfo_nbpos(info);
                load_trace<T, ND, NV>(a.Q + (int64_t)nbe * NPE + line_node<ND, N>(kp >> 1, f, (kp & 1) ? N - 1 : 0),
                                      Nd, dir, ext);
            }
        } else {
            boundary_trace<T, ND, NPF, NV>(a, info, slot, f, dir, own, ext);
        }
        axis_flux<T, ND>(own, ext, sn, jac, finfo_side(info), a.sdiss, gamma, a.intensity, a.errflag, Fn);
        T* o = sFn + ((le2 * NF + k) * NV) * NPF + f;
        o[0] = Fn[0];
#pragma unroll
        for (int c = 0; c < ND; ++c) o[face_mom<ND>(dir, c) * NPF] = Fn[1 + c];
        o[(NV - 1) * NPF] = Fn[NV - 1];
    }
    __syncthreads();
    if (!valid) return;

    // ---- FR lift on the end nodes, mass matrix and stage epilogue -----------------------------
    const T gm0 = a.ops[ops_gm(N)], gpn = a.ops[ops_gp(N) + N - 1];
#pragma unroll
    for (int dir = 0; dir < ND; ++dir) {
        int f, ii;
        node_line<ND, N>(node, dir, f, ii);
        if (ii == 0 || ii == N - 1) {
            const T* s = sFn + ((le * NF + 2 * dir + (ii ? 1 : 0)) * NV) * NPF + f;
            const T c = ii ? gpn : gm0;
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = acc[v] - c * s[v * NPF];
        }
    }
    const Recip<T> iJ(sG[le * (ND + 1) + ND]);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

// ---- 1-D ----------------------------------------------------------------------------------------
//
// Meshes of a few dozen to some ten thousand nodes: bound by the chain of dependent operations,
// not by any rate.  Two waves take the nodes and pairs and two the faces, which read their traces from
// memory and wait for nothing: the surface flux (any of the framework's) runs beside the pairs.
// Measured, ORK256 steps of 20 elements, N=3, Chandrasekhar and
// MatrixDissipation: 8.3 -> 7.3 us per stage.
template <int N>
struct ECfg {
    static constexpr int G = 128, TPB = 2 * G;
    static constexpr int NPAIR = N * (N - 1) / 2;
    static constexpr int EPB = N == 2 ? 64 : G / NPAIR;  // a pair per thread
    static constexpr int NN = EPB * N;
};

template <int N, int TP>
__global__ void __launch_bounds__((ECfg<N>::TPB)) k_split_1d(const RhsArgs<double> a) {
    using T = double;
    using C = ECfg<N>;
    constexpr int NV = 3, EPB = C::EPB, NN = C::NN, NS = plain::tp_slots<1, TP>(), NPAIR = C::NPAIR;
    __shared__ T sS[NS * NN];            // two-point flux inputs
    __shared__ T sTab[NV][EPB * NPAIR];  // pair fluxes
    __shared__ T sFn[NV][2 * EPB];       // face fluxes
    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs, g0 = (int64_t)e0 * N;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    if (tid >= C::G) {
        const int it = tid - C::G, le = it >> 1, k = it & 1;
        const bool task = le < nel;
        T own[NV], ext[NV], F[NV];
        if (task) {
            const int slot = (e0 + le) * 2 + k;
            const int info = a.finfo[slot], nbe = a.nb[slot];
            const T* g = a.fgeom + (int64_t)a.fgi[slot] * 4;
            load_trace<T, 1, NV>(a.Q + (int64_t)(e0 + le) * N + (k ? N - 1 : 0), Nd, 0, own);
            const T sn = g[0], jac = g[3];
            if (nbe >= 0)
                load_trace<T, 1, NV>(a.Q + (int64_t)nbe * N + ((finfo_nbpos(info) & 1) ? N - 1 : 0), Nd, 0, ext);
            else
                boundary_trace<T, 1, 1, NV>(a, info, slot, 0, 0, own, ext);
            own[1] = sn * own[1];
            ext[1] = sn * ext[1];
            const bool slave = finfo_side(info);
            T L[NV], R[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                L[v] = slave ? ext[v] : own[v];
                R[v] = slave ? own[v] : ext[v];
            }
            plain::euler_numericalflux<T, 1>(L, R, a.savg, a.sdiss, a.typo, a.intensity, a.gamma, a.errflag, F);
            F[1] = sn * F[1];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const T x = F[v] * jac;
                sFn[v][it] = slave ? -x : x;
            }
        }
        __syncthreads();
        __syncthreads();
        return;
    }
    const bool valid = tid < nel * N;
    const int le = tid / N, ii = tid - le * N;
    const T ja = a.egeom[0 + (int64_t)(valid ? e0 + le : e0) * a.egeom_stride];
    const T J = a.egeom[1 + (int64_t)(valid ? e0 + le : e0) * a.egeom_stride];
    T q[NV], xv[NV], D[N];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    const T* aux = stage_aux(a);
    if (aux && valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
    }
#pragma unroll
    for (int j = 0; j < N; ++j) D[j] = a.ops[ops_Dsh(N) + ii * N + j];
    const T gm0 = a.ops[ops_gm(N)], gpn = a.ops[ops_gp(N) + N - 1];
    T own[NV];  // the node's contravariant flux
    {
        T P[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, 1>(q, a.gamma, P, ir);
        if (valid) plain::put_slots<T, 1, TP, NN>(sS + tid, q, P, ir);
        own[0] = q[1] * ja;
        own[1] = (q[1] * P[1] + P[2]) * ja;
        own[2] = ((q[2] + P[2]) * P[1]) * ja;
    }
    __syncthreads();
    {
        const int pr = tid / EPB, l = tid - pr * EPB;
        if (pr < NPAIR && l < nel) {
            const int ab = pair_ab<N>(pr);
            const T* sa = sS + l * N + (ab >> 3);
            const T* sb = sS + l * N + (ab & 7);
            T A[NS], B[NS], F[NV];
#pragma unroll
            for (int c = 0; c < NS; ++c) { A[c] = sa[c * NN]; B[c] = sb[c * NN]; }
            const T jl = a.egeom[(int64_t)(e0 + l) * a.egeom_stride];
            plain::pair_flux<T, 1, TP, 0>(A, B, jl, a.gamma - T(1), a.errflag, F);
#pragma unroll
            for (int v = 0; v < NV; ++v) sTab[v][tid] = F[v];
        }
    }
    __syncthreads();
    if (!valid) return;
    T acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    int off = (ii - 1) * EPB + le;  // as in direction()
#pragma unroll
    for (int j = 0; j < N; ++j) {
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = acc[v] - D[j] * (j == ii ? own[v] : sTab[v][j == ii ? 0 : off]);
        off += (j < ii ? N - j - 2 : 1) * EPB;
    }
    if (ii == 0 || ii == N - 1) {
        const T c = ii ? gpn : gm0;
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = acc[v] - c * sFn[v][2 * le + (ii ? 1 : 0)];
    }
    const Recip<T> iJ(J);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

template <int ND, int N, int TP>
static hipError_t launch(const RhsArgs<double>& a, hipStream_t s) {
    using C = SCfg<ND, N>;
    hipLaunchKernelGGL((k_split<ND, N, TP>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

template <int N, int TP>
static hipError_t launch_1d(const RhsArgs<double>& a, hipStream_t s) {
    using C = ECfg<N>;
    hipLaunchKernelGGL((k_split_1d<N, TP>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

// While all blocks run at once.  Against the general kernel (lxf false: the other surface fluxes) that is
// up to 1024 blocks at every node count (512 to 1024 blocks, N nodes per line: 1.0 to 1.2 times as fast at 2 and
// 3, 1.1 to 1.4 from 4; N=8, 6250 blocks 15.3 us against 29.5).  k_split, which LxF and StdAverage have instead,
// does without the second half of the block: 5 nodes and more up to 768 blocks (1.0 to 1.3; 8 nodes and StdAverage,
// 896 blocks 5.16 us against 5.37); 2 and 3 nodes 0.88 to 1.0 from 128 blocks, 4 nodes 0.91 to 1.08.
template <int N>
static RhsLauncherF64 pick_1d(int tp, int64_t ne, bool lxf) {
    const int64_t nb = (ne + ECfg<N>::EPB - 1) / ECfg<N>::EPB;
    if (lxf ? N < 5 || nb > 768 : nb > 1024) return nullptr;
    switch (tp) {
        case TP_STDAVG: return &launch_1d<N, TP_STDAVG>;
        case TP_CHANDRASEKHAR: return &launch_1d<N, TP_CHANDRASEKHAR>;
        case TP_KENNEDY_GRUBER: return &launch_1d<N, TP_KENNEDY_GRUBER>;
        default: return nullptr;
    }
}

template <int ND, int N>
static RhsLauncherF64 pick_tp(int tp) {
    switch (tp) {
        case TP_STDAVG: return &launch<ND, N, TP_STDAVG>;
        case TP_CHANDRASEKHAR: return &launch<ND, N, TP_CHANDRASEKHAR>;
        case TP_KENNEDY_GRUBER: return &launch<ND, N, TP_KENNEDY_GRUBER>;
        default: return nullptr;
    }
}

// ---- curved elements --------------------------------------------------------------------------
//
// The same form with a metric per node.  The general kernel forms every component of a pair's
// flux and contracts them with the mean metric n̄, with IEEE quotients throughout, and reads
// metrics from memory once per pair.  Here the flux along n̄ is formed directly (pair_along.hpp), sums
// by fused multiply-adds, so results agree with the general kernel's up to rounding and are no
// less exact; a direction's metric rows lie in LDS beside the flux inputs.  Eight-wave blocks run two
// to a CU up to 128 registers: they read a node's velocities from its slots again for each direction (3-D
// N=6, held in registers: 133, one block per CU, 84 us against 61 at 0.6 M nodes).  Faces: the flux along n from the master's frame; every sum over the two sides
// commutes and is rounded the same way on both, so that the sides' fluxes are opposite bit for bit.
// What bounds it: waits between the barriers at two or three blocks per CU.  A stage at 11.2 M nodes needs
// 2.1 GB (187 bytes per node) and moves 1.75 GB (FETCH_SIZE 1.30, WRITE_SIZE 0.45: part of the rest comes from the
// cache behind the L2s), 0.37 ms at a copy's rate.  Measured, Chandrasekhar, SSPRK33 steps: 3-D N=6,
// 11.2 M nodes: 9.1 -> 3.1 ms; N=5, 7.1 M nodes: 3.6 -> 1.8 ms.

// One direction: pairs and the nodes' own fluxes into the table, then (LOADS between) the
// nodes' D♯ rows over it.  m: the metric row of the own node.
template <int ND, int N, int TP, int DIR, typename LOADS>
__device__ __forceinline__ void curved_direction(const RhsArgs<double>& a, const double* sS, const double* sM, double* sTab,
                                                 const double* sD, int nel, int tid, int le, int node, bool valid,
                                                 const double (&q)[ND + 2], const double (&u)[ND], double p,
                                                 const double (&m)[ND], LOADS loads, double (&acc)[ND + 2]) {
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPF = C::NPF, SN = C::SN, NL = C::NL, NS = curved_slots<ND, TP>();
    constexpr int KS = C::KS, VS = C::VS, DIAG = C::NPAIR * C::NLP;
    using M = Nodes<ND, N>;
    const double ig1 = 1.0 / (a.gamma - 1.0);
    int lf, ii;
    node_line<ND, N>(node, DIR, lf, ii);
    if (valid) {
        double* t = sTab + (DIAG + tid) * KS;
        const double* s = sS + M::node(tid);
        auto vel = [&](int k) { return C::TPB > 256 ? curved_velocity<TP, SN>(s, k) : u[k]; };
        double w = vel(0) * m[0], mass = q[1] * m[0];
#pragma unroll
        for (int k = 1; k < ND; ++k) {
            w = __builtin_fma(vel(k), m[k], w);
            mass = __builtin_fma(q[1 + k], m[k], mass);
        }
        t[0] = mass;
#pragma unroll
        for (int c = 0; c < ND; ++c) t[(1 + c) * VS] = __builtin_fma(q[1 + c], w, p * m[c]);
        t[(NV - 1) * VS] = (q[NV - 1] + p) * w;
    }
#pragma unroll 1
    for (int k = tid; k < C::NPR; k += C::TPB) {
        const int pr = k / NL, l = k - pr * NL;
        const int le2 = C::EPB == 1 ? 0 : l / NPF, f = l - le2 * NPF;
        if (le2 >= nel) continue;
        const int ab = pair_ab<N>(pr);
        const int base = le2 * M::ES + M::template line<DIR>(f);
        constexpr int ST = M::template step<DIR>();
        const int ia = base + (ab >> 3) * ST, ib = base + (ab & 7) * ST;
        double A[NS], B[NS], n[ND], F[NV];
#pragma unroll
        for (int c = 0; c < NS; ++c) { A[c] = sS[c * SN + ia]; B[c] = sS[c * SN + ib]; }
#pragma unroll
        for (int c = 0; c < ND; ++c) n[c] = sM[c * SN + ia] + sM[c * SN + ib];
        pair_flux_along<ND, TP>(A, B, n, ig1, a.errflag, F);
#pragma unroll
        for (int v = 0; v < NV; ++v) sTab[(pr * C::NLP + l) * KS + v * VS] = F[v];
    }
    loads();
    __syncthreads();
    if (valid) {
        const int diag = (DIAG + tid) * KS;
        int off = ((ii - 1) * C::NLP + le * NPF + lf) * KS;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double* t = sTab + (j == ii ? diag : off);
            const double Dij = sD[ii * N + j];
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = __builtin_fma(-Dij, t[v * VS], acc[v]);
            off += (j < ii ? N - j - 2 : 1) * (C::NLP * KS);
        }
    }
}

template <int ND, int N, int TP>
__global__ void __launch_bounds__((SCfg<ND, N>::TPB)) k_split_curved(const RhsArgs<double> a) {
    using T = double;
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN, SN = C::SN;
    constexpr int NS = curved_slots<ND, TP>(), FG = 3 * ND + 1;
    constexpr int NFN = EPB * NF * NPF;  // face nodes of the block
    constexpr int TAB = C::TAB, FACE = NN + NFN;
    __shared__ T sS[NS * SN];                           // two-point flux inputs, [slot][node]
    __shared__ T sM[ND * SN];                           // half the metric row of the direction, [component][node]
    __shared__ T sTab[NV * (TAB > FACE ? TAB : FACE)];  // as in k_split
    __shared__ T sD[N * N];

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const T gamma = a.gamma;

    // ---- own node, face tables, operators -----------------------------------------------
    const int fe = tid / (NF * NPF), fk = (tid - fe * (NF * NPF)) / NPF, ff = tid % NPF;
    const bool pf = tid < NFN && fe < nel;
    int pinfo = 0, pnb = -1, pfgi = 0;
    if (pf) {
        const int slot = (e0 + fe) * NF + fk;
        pinfo = a.finfo[slot];
        pnb = a.nb[slot];
        pfgi = a.fgi[slot];
    }
    const bool valid = tid < nel * NPE;
    const int le = tid / NPE, node = tid - le * NPE;
    const int64_t g0 = (int64_t)e0 * NPE;
    const int jj = Nodes<ND, N>::node(tid);
    T q[NV], m[ND];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    auto metric = [&](int dir) {  // the own node's metric row, on its way to LDS
#pragma unroll
        for (int c = 0; c < ND; ++c) m[c] = valid ? a.ngeom[(c + ND * dir) * Nd + g0 + tid] : T(0);
    };
    auto put_metric = [&]() {
        if (valid) {
#pragma unroll
            for (int c = 0; c < ND; ++c) sM[c * SN + jj] = T(0.5) * m[c];
        }
    };
    metric(0);
    for (int i = tid; i < N * N; i += TPB) sD[i] = a.ops[ops_Dsh(N) + i];
    T u[ND], p;
    {
        T P[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, gamma, P, ir);
#pragma unroll
        for (int k = 0; k < ND; ++k) u[k] = P[1 + k];
        p = P[ND + 1];
        if (valid) curved_node<ND, TP, SN>(sS + jj, q, P, ir);
    }
    put_metric();
    __syncthreads();

    // ---- volume terms, direction by direction ---------------------------------------------
    T acc[NV], pext[NV], xv[NV], pg[ND + 1], J = T(1);
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    const T* aux = stage_aux(a);
    auto trace = [&](int info, int nbe, int f, T* ext) {
        const int kp = finfo_nbpos(info);
        const T* Qn = a.Q + (int64_t)nbe * NPE +
                      line_node<ND, N>(kp >> 1, face_nb_node<ND, N>(f, info), (kp & 1) ? N - 1 : 0);
#pragma unroll
        for (int v = 0; v < NV; ++v) ext[v] = Qn[v * Nd];
    };
    auto frame = [&](int info, int fgi, int f, T* g) {  // the master's normal, surface J
        const T* s = a.fgeom + ((int64_t)fgi * NPF + face_master_node<ND, N>(f, info)) * FG;
#pragma unroll
        for (int c = 0; c < ND; ++c) g[c] = s[c];
        g[ND] = s[3 * ND];
    };
    auto prefetch = [&]() {
        if (pf && pnb >= 0) trace(pinfo, pnb, ff, pext);
        if (pf) frame(pinfo, pfgi, ff, pg);
        if (valid) {
            J = a.ngeom[ND * ND * Nd + g0 + tid];
            if (aux) {
#pragma unroll
                for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
            }
        }
    };
    curved_direction<ND, N, TP, 0>(a, sS, sM, sTab, sD, nel, tid, le, node, valid, q, u, p, m, [&]() { metric(1); }, acc);
    put_metric();
    __syncthreads();
    if constexpr (ND == 3) {
        curved_direction<ND, N, TP, 1>(a, sS, sM, sTab, sD, nel, tid, le, node, valid, q, u, p, m, [&]() { metric(2); }, acc);
        put_metric();
        __syncthreads();
    }
    curved_direction<ND, N, TP, ND - 1>(a, sS, sM, sTab, sD, nel, tid, le, node, valid, q, u, p, m, prefetch, acc);
    __syncthreads();

    // ---- numerical fluxes on the element's faces --------------------------------------------
    T* const sU = sTab;
    T* const sFn = sTab + NV * NN;
    if (valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sU[v * NN + tid] = q[v];
    }
    __syncthreads();
    for (int it = tid; it < NFN; it += TPB) {
        const bool first = it == tid;
        const int le2 = it / (NF * NPF), r = it - le2 * (NF * NPF);
        const int k = r / NPF, f = r - k * NPF;
        if (le2 >= nel) continue;
        const int slot = (e0 + le2) * NF + k;
        const int info = first ? pinfo : a.finfo[slot];
        const int nbe = first ? pnb : a.nb[slot];
        const T* own0 = sU + le2 * NPE + line_node<ND, N>(k >> 1, f, (k & 1) ? N - 1 : 0);
        T own[NV], ext[NV], g[ND + 1];
#pragma unroll
        for (int v = 0; v < NV; ++v) own[v] = own0[v * NN];
        if (first) {
#pragma unroll
            for (int c = 0; c <= ND; ++c) g[c] = pg[c];
        } else {
            frame(info, a.fgi[slot], f, g);
        }
        if (nbe >= 0) {
            if (first) {
#pragma unroll
                for (int v = 0; v < NV; ++v) ext[v] = pext[v];
            } else {
                trace(info, nbe, f, ext);
            }
        } else {
            const int bd = finfo_bd(info);
            const int type = a.bctype[bd];
            if (type == BC_DIRICHLET || type == BC_INFLOW) {
                const T* src = type == BC_DIRICHLET ? a.bcstate + ((int64_t)a.fid[slot] * NPF + f) * NV
                                                    : a.bcconst + bd * NV;
#pragma unroll
                for (int v = 0; v < NV; ++v) ext[v] = src[v];
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) ext[v] = own[v];
                if (type == BC_SLIP) {
                    T mn = own[1] * g[0];
#pragma unroll
                    for (int c = 1; c < ND; ++c) mn = mn + own[1 + c] * g[c];
#pragma unroll
                    for (int c = 0; c < ND; ++c) ext[1 + c] = own[1 + c] - (T(2) * mn) * g[c];
                }
            }
        }
        T mo = own[1] * g[0], mx = ext[1] * g[0];
#pragma unroll
        for (int c = 1; c < ND; ++c) {
            mo = mo + own[1 + c] * g[c];
            mx = mx + ext[1 + c] * g[c];
        }
        const Recip<T> iro(own[0]), irx(ext[0]);
        const T po = plain::pressure<T, ND>(own, gamma, iro), px = plain::pressure<T, ND>(ext, gamma, irx);
        const T uo = iro.div(mo), ux = irx.div(mx);
        const bool slave = finfo_side(info);
        T Fn[NV];
        Fn[0] = (mo + mx) / T(2);
#pragma unroll
        for (int c = 0; c < ND; ++c) Fn[1 + c] = ((own[1 + c] * uo + ext[1 + c] * ux) + (po + px) * g[c]) / T(2);
        Fn[NV - 1] = ((own[NV - 1] + po) * uo + (ext[NV - 1] + px) * ux) / T(2);
        const T sg = slave ? T(-1) : T(1);
        if (a.sdiss == DISS_LXF) {
            const T lo = fabs(uo) + plain::dsqrt(iro.div(gamma * po), a.errflag);
            const T lx = fabs(ux) + plain::dsqrt(irx.div(gamma * px), a.errflag);
            // the larger speed, the master's where they do not compare
            const T lam = sg * (slave ? ((lx < lo) ? lo : lx) : ((lo < lx) ? lx : lo));
#pragma unroll
            for (int v = 0; v < NV; ++v) Fn[v] = Fn[v] + ((lam * (own[v] - ext[v])) / T(2)) * a.intensity;
        }
        T* o = sFn + ((le2 * NF + k) * NV) * NPF + f;
        const T js = sg * g[ND];
#pragma unroll
        for (int v = 0; v < NV; ++v) o[v * NPF] = Fn[v] * js;
    }
    __syncthreads();
    if (!valid) return;

    // ---- FR lift on the end nodes, mass matrix and stage epilogue -----------------------------
    const T gm0 = a.ops[ops_gm(N)], gpn = a.ops[ops_gp(N) + N - 1];
#pragma unroll
    for (int dir = 0; dir < ND; ++dir) {
        int f, ii;
        node_line<ND, N>(node, dir, f, ii);
        if (ii == 0 || ii == N - 1) {
            const T* s = sFn + ((le * NF + 2 * dir + (ii ? 1 : 0)) * NV) * NPF + f;
            const T c = ii ? gpn : gm0;
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = acc[v] - c * s[v * NPF];
        }
    }
    const Recip<T> iJ(J);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

template <int ND, int N, int TP>
static hipError_t launch_curved(const RhsArgs<double>& a, hipStream_t s) {
    using C = SCfg<ND, N>;
    hipLaunchKernelGGL((k_split_curved<ND, N, TP>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

template <int ND, int N>
static RhsLauncherF64 pick_curved(int tp) {
    switch (tp) {
        case TP_STDAVG: return &launch_curved<ND, N, TP_STDAVG>;
        case TP_CHANDRASEKHAR: return &launch_curved<ND, N, TP_CHANDRASEKHAR>;
        case TP_KENNEDY_GRUBER: return &launch_curved<ND, N, TP_KENNEDY_GRUBER>;
        default: return nullptr;
    }
}

}  // namespace split

#define FLOUHIP_CAT_(a, b) a##b
#define FLOUHIP_CAT(a, b) FLOUHIP_CAT_(a, b)

RhsLauncherF64 FLOUHIP_CAT(split_f64_, FLOUHIP_ND)(int n, int tp) {
    switch (n) {
        case 2: return split::pick_tp<FLOUHIP_ND, 2>(tp);
        case 3: return split::pick_tp<FLOUHIP_ND, 3>(tp);
        case 4: return split::pick_tp<FLOUHIP_ND, 4>(tp);
        case 5: return split::pick_tp<FLOUHIP_ND, 5>(tp);
        case 6: return split::pick_tp<FLOUHIP_ND, 6>(tp);
        case 7: return split::pick_tp<FLOUHIP_ND, 7>(tp);
        case 8: return split::pick_tp<FLOUHIP_ND, 8>(tp);
        default: return nullptr;
    }
}

#if FLOUHIP_ND == 1
RhsLauncherF64 split_f64_1_small(int n, int tp, int64_t ne, bool lxf) {
    switch (n) {
        case 2: return split::pick_1d<2>(tp, ne, lxf);
        case 3: return split::pick_1d<3>(tp, ne, lxf);
        case 4: return split::pick_1d<4>(tp, ne, lxf);
        case 5: return split::pick_1d<5>(tp, ne, lxf);
        case 6: return split::pick_1d<6>(tp, ne, lxf);
        case 7: return split::pick_1d<7>(tp, ne, lxf);
        case 8: return split::pick_1d<8>(tp, ne, lxf);
        default: return nullptr;
    }
}
#else
RhsLauncherF64 FLOUHIP_CAT(split_curved_f64_, FLOUHIP_ND)(int n, int tp) {
    switch (n) {
        case 2: return split::pick_curved<FLOUHIP_ND, 2>(tp);
        case 3: return split::pick_curved<FLOUHIP_ND, 3>(tp);
        case 4: return split::pick_curved<FLOUHIP_ND, 4>(tp);
        case 5: return split::pick_curved<FLOUHIP_ND, 5>(tp);
        case 6: return split::pick_curved<FLOUHIP_ND, 6>(tp);
        case 7: return split::pick_curved<FLOUHIP_ND, 7>(tp);
        case 8: return split::pick_curved<FLOUHIP_ND, 8>(tp);
        default: return nullptr;
    }
}
#endif

}  // namespace flouhip
