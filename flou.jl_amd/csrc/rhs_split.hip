// FP64 split-form Euler rhs on axis-aligned affine elements (Flou's CartesianMesh), GLL
// nodes, StdAverage or LxF(StdAverage) surface flux, with the RK stage epilogue: the plain
// kernel's arithmetic (rhs_plain.hip, reference order, every value rounded where the
// reference rounds it) without the work that this geometry makes void.
//
// What bounds it: FP64 arithmetic, by issue (90 % of busy cycles) and by the clock the power
// limit leaves under it (1.8 to 2.0 of 2.4 GHz).  k_plain<double, 3, 6, ..> spends about 4000
// VALU slots per node, most of them on divisions, on the two components of every flux that a
// diagonal metric multiplies by zero, and on rotations by 0 and ±1.  Measured against it (same
// bits): 3-D N=5, 10.5 M nodes, Chandrasekhar: 1.65 -> 0.96 ms per CK2N54 stage; 2-D N=5, 0.59 M
// nodes: 66 -> 43 us.  With the same results:
//   * only the flux component along the line's direction is formed: f·n̄ has one term, the
//     others are exact zeros.  The direction is a compile-time constant of each phase;
//   * flux inputs are staged halved, so that means are one addition (pair_flux);
//   * a node's own contravariant flux goes into the same table as the pairs, so that its row
//     reads N entries without a case for the diagonal, at offsets that advance by constants
//     (2504 -> 2186 VALU per wave at 3-D N=5 with the above, 0.99 -> 0.96 ms);
//   * face states are read in the order of the face frame by index (faces.hpp);
//   * quotients share reciprocals (exact_div.hpp), the node's contravariant flux reuses its
//     primitives, the lift touches the end nodes only (∂g is exactly zero elsewhere);
//   * the face fluxes come last and lie over the dead table (39 KB of LDS at 3-D N=5, 4 waves
//     per SIMD); their neighbour traces are loaded before the last direction's rows.
// One thread per node (blocks rounded up to whole waves, the spare lanes take pairs), pairs
// pair-major: consecutive lanes evaluate the same pair of consecutive lines, so node reads
// and table writes are conflict-light and the pair's positions nearly uniform.
// Compile with -DFLOUHIP_ND=1|2|3.
#include "common.hpp"
#include "faces.hpp"
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
    static constexpr int TPB = ((NN + 63) / 64) * 64;    // threads per block
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
    T q[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    for (int i = tid; i < N * N; i += TPB) sD[i] = a.ops[ops_Dsh(N) + i];
    for (int i = tid; i < EPB * (ND + 1); i += TPB) {
        const int e = i / (ND + 1), c = i - e * (ND + 1);
        if (e < nel) sG[i] = a.egeom[(int64_t)(e0 + e) * a.egeom_stride + (c < ND ? c * (ND + 1) : ND * ND)];
    }
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
        if (pf && pnb >= 0) {
            const int kp = finfo_nbpos(pinfo), dir = fk >> 1;
            load_trace<T, ND, NV>(a.Q + (int64_t)pnb * NPE + line_node<ND, N>(kp >> 1, ff, (kp & 1) ? N - 1 : 0), Nd,
                                  dir, pext);
        }
        if (pf) {
            const T* g = a.fgeom + (int64_t)pfgi * (3 * ND + 1);
            pn = g[fk >> 1];
            pj = g[3 * ND];
        }
        if (aux && valid) {
#pragma unroll
            for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
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

template <int ND, int N, int TP>
static hipError_t launch(const RhsArgs<double>& a, hipStream_t s) {
    using C = SCfg<ND, N>;
    hipLaunchKernelGGL((k_split<ND, N, TP>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
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

}  // namespace flouhip
