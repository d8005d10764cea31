// FP64 split-form Euler rhs on axis-aligned affine elements (Flou's CartesianMesh), GLL
// nodes, StdAverage or LxF(StdAverage) surface flux, with the RK stage epilogue: the plain
// kernel's arithmetic (rhs_plain.hip, reference order, every value rounded where the
// reference rounds it) without the work that this geometry makes void.
//
// What bounds it: FP64 VALU issue.  k_plain<double, 3, 6, ..> spends about 4000 VALU slots
// per node, most of them on divisions, on the two components of every flux that a diagonal
// metric multiplies by zero, and on rotations by 0 and ±1.  Measured against it (same bits):
// 3-D N=5, 10.5 M nodes, Chandrasekhar: 1.65 -> 0.99 ms per CK2N54 stage (0.97 -> 1.6 TB/s of
// algorithmic bytes); 2-D N=5, 0.59 M nodes: 66 -> 47 us.  With the same results:
//   * only the flux component along the line's direction is formed: f·n̄ has one term, the
//     others are exact zeros.  The direction is a compile-time constant of each phase;
//   * face states are read in the order (normal, transverse..) of the face frame by index,
//     n = ±e_d, t = ±e_{d+1}, b = ±e_{d+2}: signs of the transverse axes commute with every
//     rounding of the LxF and StdAverage fluxes, so they need not be applied;
//   * quotients share reciprocals (exact_div.hpp), the diagonal contravariant flux reuses
//     the staged primitives, the lift touches the end nodes only (∂g is exactly zero
//     elsewhere);
//   * the pair table of one direction lies over the staged conservative states, which are
//     dead after the face fluxes; a thread keeps its own node's state in registers.
// One thread per node (blocks rounded up to whole waves, the spare lanes take pairs), pairs
// pair-major: consecutive lanes evaluate the same pair of consecutive lines, so node reads
// and table writes are conflict-light and the pair's positions nearly uniform.
// Compile with -DFLOUHIP_ND=1|2|3.
#include "common.hpp"
#include "physics_plain.hpp"
#include "stage.hpp"

namespace flouhip {
namespace split {

template <int ND, int N>
struct SCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND, NV = ND + 2;
    static constexpr int EPB = Cfg<ND, N>::EPB;
    static constexpr int NN = EPB * NPE;                 // nodes per block
    static constexpr int TPB = ((NN + 63) / 64) * 64;    // threads per block
    static constexpr int NPAIR = N * (N - 1) / 2;
    static constexpr int NPR = EPB * NPF * NPAIR;        // pairs per block and direction
    static constexpr int NL = EPB * NPF;                 // lines per block and direction
};

// One direction: the pair table, then every node's D♯ row over it in the order j = 0..N-1
// (diagonal: the contravariant flux), then this node's face terms are left to the caller.
template <int ND, int N, int TP, int DIR>
__device__ __forceinline__ void direction(const RhsArgs<double>& a, const double* sS, double* sPair, const double* sD,
                                          const double* sG, int nel, int tid, int le, int node, bool valid,
                                          const double (&q)[ND + 2], const double (&u)[ND], double p,
                                          double (&acc)[ND + 2]) {
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NN = C::NN, NS = plain::tp_slots<ND, TP>();
    const double gm1 = a.gamma - 1.0;
    __syncthreads();  // the table's memory has been read (the previous direction, or the own traces)
#pragma unroll 1
    for (int k = tid; k < C::NPR; k += C::TPB) {
        const int pr = k / C::NL, l = k - pr * C::NL;
        const int le2 = C::EPB == 1 ? 0 : l / NPF, f = l - le2 * NPF;
        if (le2 >= nel) continue;
        const int ab = pair_ab<N>(pr);
        const int base = le2 * NPE + line_node<ND, N>(DIR, f, 0);
        constexpr int ST = DIR == 0 ? 1 : (DIR == 1 ? N : N * N);
        const double* pa = sS + base + (ab >> 3) * ST;
        const double* pb = sS + base + (ab & 7) * ST;
        double A[NS], B[NS], F[NV];
#pragma unroll
        for (int c = 0; c < NS; ++c) { A[c] = pa[c * NN]; B[c] = pb[c * NN]; }
        plain::pair_flux<double, ND, TP, DIR>(A, B, sG[le2 * (ND + 1) + DIR], gm1, a.errflag, F);
#pragma unroll
        for (int v = 0; v < NV; ++v) sPair[k * NV + v] = F[v];
    }
    __syncthreads();
    if (valid) {
        int f, ii;
        node_line<ND, N>(node, DIR, f, ii);
        const double ja = sG[le * (ND + 1) + DIR];
        // contravariant flux of the node along DIR (plain::contravariant_flux, diagonal metric)
        double Fd[NV];
        Fd[0] = q[1 + DIR] * ja;
#pragma unroll
        for (int c = 0; c < ND; ++c) Fd[1 + c] = (c == DIR ? q[1 + DIR] * u[c] + p : q[1 + DIR] * u[c]) * ja;
        Fd[NV - 1] = ((q[NV - 1] + p) * u[DIR]) * ja;
        const int l = le * NPF + f;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double Dij = sD[ii * N + j];
            const int lo = j < ii ? j : ii, hi = j < ii ? ii : j;
            const int pr = j == ii ? 0 : lo * (2 * N - lo - 1) / 2 + (hi - lo - 1);
            const double* t = sPair + (pr * C::NL + l) * NV;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double F = j == ii ? Fd[v] : t[v];
                acc[v] = acc[v] - Dij * F;
            }
        }
    }
}

template <int ND, int N, int TP>
__global__ void __launch_bounds__((SCfg<ND, N>::TPB)) k_split(const RhsArgs<double> a) {
    using T = double;
    using C = SCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN;
    constexpr int NS = plain::tp_slots<ND, TP>();
    constexpr int UN = NV * (NN > C::NPR ? NN : C::NPR);
    __shared__ T sS[NS * NN];          // two-point flux inputs, [slot][node]
    __shared__ T sU[UN];               // conservative states [v][node], then the pair table
    __shared__ T sFn[EPB * NF * NV * NPF];
    __shared__ T sD[N * N];
    __shared__ T sG[EPB * (ND + 1)];   // Ja_dd and J per element

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const int nnb = nel * NPE;         // nodes of this block
    const T gamma = a.gamma, gm1 = a.gamma - 1.0;

    // ---- loads: face tables, own node, neighbour trace, epilogue operand, tables ----------
    constexpr int NFN = EPB * NF * NPF;
    const int fe = tid / (NF * NPF), fk = (tid - fe * (NF * NPF)) / NPF, ff = tid % NPF;
    const bool pf = tid < NFN && fe < nel;
    int pinfo = 0, pnb = -1, pfgi = 0;
    if (pf) {
        const int slot = (e0 + fe) * NF + fk;
        pinfo = a.finfo[slot];
        pnb = a.nb[slot];
        pfgi = a.fgi[slot];
    }
    const bool valid = tid < nnb;
    const int le = tid / NPE, node = tid - le * NPE;
    const int64_t g0 = (int64_t)e0 * NPE;
    T q[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    // a face node's states are read in the order ρ, normal and transverse momenta, E
    T pext[NV];
    if (pf && pnb >= 0) {
        const int kp = finfo_nbpos(pinfo), dir = fk >> 1;
        const T* Qn = a.Q + (int64_t)pnb * NPE + line_node<ND, N>(kp >> 1, ff, (kp & 1) ? N - 1 : 0);
        pext[0] = Qn[0];
#pragma unroll
        for (int c = 0; c < ND; ++c) pext[1 + c] = Qn[(1 + (dir + c) % ND) * Nd];
        pext[NV - 1] = Qn[(NV - 1) * Nd];
    }
    T pn = T(0), pj = T(0);
    if (pf) {
        const T* g = a.fgeom + (int64_t)pfgi * (3 * ND + 1);
        pn = g[fk >> 1];
        pj = g[3 * ND];
    }
    const T* aux = stage_aux(a);
    T xv[NV];
    if (aux && valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
    }
    for (int i = tid; i < N * N; i += TPB) sD[i] = a.ops[ops_Dsh(N) + i];
    for (int i = tid; i < EPB * (ND + 1); i += TPB) {
        const int e = i / (ND + 1), c = i - e * (ND + 1);
        if (e < nel) sG[i] = a.egeom[(int64_t)(e0 + e) * a.egeom_stride + (c < ND ? c * (ND + 1) : ND * ND)];
    }

    // ---- staging --------------------------------------------------------------------------
    T u[ND], p;
    {
        T P[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, gamma, P, ir);
#pragma unroll
        for (int k = 0; k < ND; ++k) u[k] = P[1 + k];
        p = P[ND + 1];
        if (valid) {
#pragma unroll
            for (int v = 0; v < NV; ++v) sU[v * NN + tid] = q[v];
            plain::put_slots<T, ND, TP, NN>(sS + tid, q, P, ir);
        }
    }
    __syncthreads();

    // ---- numerical fluxes on the element's faces -------------------------------------------
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
        int vo[ND];  // physical variable of each face-frame momentum
#pragma unroll
        for (int c = 0; c < ND; ++c) vo[c] = 1 + (dir + c) % ND;
        T own[NV], ext[NV];
        own[0] = sU[on];
#pragma unroll
        for (int c = 0; c < ND; ++c) own[1 + c] = sU[vo[c] * NN + on];
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
                const T* Qn = a.Q + (int64_t)nbe * NPE + line_node<ND, N>(kp >> 1, f, (kp & 1) ? N - 1 : 0);
                ext[0] = Qn[0];
#pragma unroll
                for (int c = 0; c < ND; ++c) ext[1 + c] = Qn[vo[c] * Nd];
                ext[NV - 1] = Qn[(NV - 1) * Nd];
            }
        } else {
            const int bd = finfo_bd(info);
            const int type = a.bctype[bd];
            if (type == BC_DIRICHLET || type == BC_INFLOW) {
                const T* src = type == BC_DIRICHLET ? a.bcstate + ((int64_t)a.fid[slot] * NPF + f) * NV
                                                    : a.bcconst + bd * NV;
                ext[0] = src[0];
#pragma unroll
                for (int c = 0; c < ND; ++c) ext[1 + c] = src[vo[c]];
                ext[NV - 1] = src[NV - 1];
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) ext[v] = own[v];
                if (type == BC_SLIP) ext[1] = -ext[1];
            }
        }
        // face frame: the momentum along the master's normal ±e_dir
        own[1] = sn * own[1];
        ext[1] = sn * ext[1];
        const bool slave = finfo_side(info);
        T Ql[NV], Qr[NV], Fn[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            Ql[v] = slave ? ext[v] : own[v];
            Qr[v] = slave ? own[v] : ext[v];
        }
        const Recip<T> irl(Ql[0]), irr(Qr[0]);
        const T pl = plain::pressure<T, ND>(Ql, gamma, irl), pr = plain::pressure<T, ND>(Qr, gamma, irr);
        const T ul = irl.div(Ql[1]), ur = irr.div(Qr[1]);
        Fn[0] = (Ql[1] + Qr[1]) / T(2);
        Fn[1] = (((Ql[1] * ul + pl) + Qr[1] * ur) + pr) / T(2);
#pragma unroll
        for (int c = 1; c < ND; ++c) Fn[1 + c] = (Ql[1 + c] * ul + Qr[1 + c] * ur) / T(2);
        Fn[NV - 1] = ((Ql[NV - 1] + pl) * ul + (Qr[NV - 1] + pr) * ur) / T(2);
        if (a.sdiss == DISS_LXF) {
            const T al = plain::dsqrt(irl.div(gamma * pl), a.errflag);
            const T ar = plain::dsqrt(irr.div(gamma * pr), a.errflag);
            const T la = fabs(ul) + al, lb = fabs(ur) + ar;
            const T lam = (la < lb) ? lb : la;
#pragma unroll
            for (int v = 0; v < NV; ++v) Fn[v] = Fn[v] + ((lam * (Ql[v] - Qr[v])) / T(2)) * a.intensity;
        }
        Fn[1] = sn * Fn[1];
        T* o = sFn + ((le2 * NF + k) * NV) * NPF + f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const T x = Fn[v] * jac;
            const int vv = (v == 0 || v == NV - 1) ? v : vo[v >= 1 && v <= ND ? v - 1 : 0];
            o[vv * NPF] = slave ? -x : x;
        }
    }

    // ---- volume terms, direction by direction ------------------------------------------------
    T acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    direction<ND, N, TP, 0>(a, sS, sU, sD, sG, nel, tid, le, node, valid, q, u, p, acc);
    if constexpr (ND >= 2) direction<ND, N, TP, 1>(a, sS, sU, sD, sG, nel, tid, le, node, valid, q, u, p, acc);
    if constexpr (ND >= 3) direction<ND, N, TP, 2>(a, sS, sU, sD, sG, nel, tid, le, node, valid, q, u, p, acc);
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
