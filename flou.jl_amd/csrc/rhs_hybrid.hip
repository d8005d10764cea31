// HybridDivOperator on GLL nodes (OpDivergence.jl:441-620, 781-801; Cartesian elements,
// Euler) with the numerical flux, the FR lift, 1/J and the RK stage epilogue, in the
// reference's order (every value rounded where the reference rounds it).
//
// Per direction: F̄_s = Σ_{k >= s} Σ_{l < s} (2ω_l D_lk) f♯(Q_l, Q_k) on the interface between
// line positions s-1 and s, blended with the surface flux of those two nodes by the entropy
// production of F̄, then dQ_i += (F̄_i - F̄_{i+1})/ω_i.
//
// What bounds it: FP64 VALU issue.  The form that evaluated each interface's sum and flux by
// itself computed the N(N-1)/2 pair fluxes of a line Σ_s s(N-s) times in all (35 instead of 15
// at N=6) and every node's entropy variables (two logarithms) twice per interface.  Here the
// block computes
//   * every pair of a direction once, into an LDS table, with the one flux component that a
//     diagonal metric keeps (DIAG; pair_flux);
//   * the entropy variables once per node, read for the blending and, in 1-D and 2-D, where
//     the face frame is a relabelling that keeps every rounding, for MatrixDissipation;
//   * the interface sums from the table, one thread per (line, interface), interface-major so
//     that the lanes of a wave run the same sum; the interface fluxes then replace the table.
// Blocks of at most 192 threads in 2-D: small meshes then spread evenly over the CUs (7
// elements per block at N=5 left 55 of 256 CUs with twice the others' work on 2175 elements).
// Measured: 2-D N=5, 2175 elements, Chandrasekhar and MatrixDissipation: 57 -> 25.5 us per stage.
// Compile with -DFLOUHIP_PREC_F64 or -DFLOUHIP_PREC_F32 and -DFLOUHIP_ND=1|2|3.
#include "common.hpp"
#include "faces.hpp"
#include "physics_plain.hpp"
#include "stage.hpp"

namespace flouhip {
namespace hybrid {

// LDS rows padded for lines of 4 and 8 nodes (MatrixDissipation, 0.6 M nodes in 2-D, 1 M in 3-D,
// without and with: 2-D of 8 nodes 109.7 and 105.8 us, 3-D of 4 258 and 254; 2-D of 6 89.6 and 92.2).
template <int ND, int N>
using Nodes = NodeLds<ND, N, N == 4 || N == 8>;

template <int ND, int N>
struct HCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND, NV = ND + 2;
    static constexpr int EPB = ND == 2 ? (N == 7 ? 5 : 192 / NPE) : Cfg<ND, N>::EPB;
    static constexpr int NN = EPB * NPE;
    static constexpr int TPB = block_threads(NN);
    static constexpr int NL = EPB * NPF;                 // lines per block and direction
    static constexpr int NPAIR = N * (N - 1) / 2;
    static constexpr int NPR = NL * NPAIR;
    static constexpr int SN = EPB * Nodes<ND, N>::ES;  // LDS nodes per block
};

// Flux input slots held beside the conservative states.
template <int ND, int TP>
constexpr int lds_slots() {
    return TP == TP_STDAVG ? ND + 1 : plain::tp_slots<ND, TP>();
}

// Both sides' states (and entropy variables) of an interface of direction DIR in the
// subcell frame, n = e_DIR, t and b the next axes: signs of t and b commute with every
// rounding of the surface fluxes.
template <typename T, int ND, int DIR>
__device__ __forceinline__ void to_frame(const T* x, T* r) {
    r[0] = x[0];
#pragma unroll
    for (int c = 0; c < ND; ++c) r[1 + c] = x[1 + (DIR + c) % ND];
    r[ND + 1] = x[ND + 1];
}

template <typename T, int ND, int N, int TP, bool DIAG, int DIR>
__device__ __forceinline__ void direction(const RhsArgs<T>& a, const T* sS, const T* sQ, const T* sW, T* sTab,
                                          const T* sC, const T* sw, const T* sM, int nel, int tid, int le, int node,
                                          bool valid, T (&acc)[ND + 2]) {
    using C = HCfg<ND, N>;
    constexpr int NV = C::NV, NPF = C::NPF, SN = C::SN, NL = C::NL;
    constexpr int NS = plain::tp_slots<ND, TP>(), NSL = lds_slots<ND, TP>();
    using M = Nodes<ND, N>;
    constexpr int ST = M::template step<DIR>();
    const T gm1 = a.gamma - T(1);
    const T avel[3] = {T(0), T(0), T(0)};
    // pair fluxes, each once
#pragma unroll 1
    for (int k = tid; k < C::NPR; k += C::TPB) {
        const int pr = k / NL, l = k - pr * NL;
        const int le2 = C::EPB == 1 ? 0 : l / NPF, f = l - le2 * NPF;
        if (le2 >= nel) continue;
        const int ab = pair_ab<N>(pr);
        const int base = le2 * M::ES + M::template line<DIR>(f);
        const T* pa = sS + base + (ab >> 3) * ST;
        const T* pb = sS + base + (ab & 7) * ST;
        T A[NS], B[NS], F[NV];
#pragma unroll
        for (int c = 0; c < NS; ++c) {  // StdAverage's conservative slots lie in sQ
            A[c] = c < NSL ? pa[c * SN] : T(0.5) * sQ[(pa - sS) + (1 + c - NSL) * SN];
            B[c] = c < NSL ? pb[c * SN] : T(0.5) * sQ[(pb - sS) + (1 + c - NSL) * SN];
        }
        if constexpr (DIAG) {
            plain::pair_flux<T, ND, TP, DIR>(A, B, sM[DIR * (ND + 1)], gm1, a.errflag, F);
        } else {
            // the general form takes conservative and primitive states (whole, not halved)
            T qa[NV], qb[NV], Pa[NV], Pb[NV];
            const T* ca = sQ + (pa - sS);
            const T* cb = sQ + (pb - sS);
            constexpr bool SD = TP == TP_STDAVG;
            constexpr int SC = TP == TP_KENNEDY_GRUBER ? ND + 2 : ND + 1;
            const T sa = TP == TP_KENNEDY_GRUBER ? T(2) * A[SC] : A[SC], sb = TP == TP_KENNEDY_GRUBER ? T(2) * B[SC] : B[SC];
#pragma unroll
            for (int v = 0; v < NV; ++v) { qa[v] = ca[v * SN]; qb[v] = cb[v * SN]; }
            Pa[0] = qa[0];
            Pb[0] = qb[0];
#pragma unroll
            for (int k = 0; k < ND; ++k) {
                Pa[1 + k] = SD ? A[k] : T(2) * A[1 + k];
                Pb[1 + k] = SD ? B[k] : T(2) * B[1 + k];
            }
            Pa[ND + 1] = T(2) * (SD ? A[ND] : A[ND + 1]);  // p (Chandrasekhar: unread)
            Pb[ND + 1] = T(2) * (SD ? B[ND] : B[ND + 1]);
            plain::twopointflux<T, ND, EQ_EULER, TP>(qa, qb, Pa, Pb, sa, sb, sM + ND * DIR, sM + ND * DIR, a.gamma,
                                                     avel, a.errflag, F);
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) sTab[v * C::NPR + k] = F[v];
    }
    __syncthreads();
    // interface fluxes: at most one per thread (NL (N-1) <= NN)
    const int s = 1 + tid / NL, l = tid % NL;
    const bool item = s < N && l / NPF < nel;
    T Fx[NV];
    if (item) {
        T Fb[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) Fb[v] = T(0);
        for (int ik = s; ik < N; ++ik)
            for (int il = 0; il < s; ++il) {
                const int pr = il * (2 * N - il - 1) / 2 + (ik - il - 1);
                const T* t = sTab + pr * NL + l;
                const T c = sC[il * N + ik];
#pragma unroll
                for (int v = 0; v < NV; ++v) Fb[v] = Fb[v] + c * t[v * C::NPR];
            }
        const int nr = (l / NPF) * M::ES + M::template line<DIR>(l % NPF) + s * ST, nl = nr - ST;
        T Ql[NV], Qr[NV], Wl[NV], Wr[NV], Rl[NV], Rr[NV], Vl[NV], Vr[NV], Fr[NV], Fv[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            Ql[v] = sQ[v * SN + nl]; Qr[v] = sQ[v * SN + nr];
            Wl[v] = sW[v * SN + nl]; Wr[v] = sW[v * SN + nr];
        }
        to_frame<T, ND, DIR>(Ql, Rl);
        to_frame<T, ND, DIR>(Qr, Rr);
        to_frame<T, ND, DIR>(Wl, Vl);
        to_frame<T, ND, DIR>(Wr, Vr);
        plain::euler_numericalflux<T, ND>(Rl, Rr, a.savg, a.sdiss, a.typo, a.intensity, a.gamma, a.errflag, Fr,
                                          ND <= 2 ? Vl : nullptr, ND <= 2 ? Vr : nullptr);
        Fv[0] = Fr[0];
#pragma unroll
        for (int c = 0; c < ND; ++c) Fv[1 + (DIR + c) % ND] = Fr[1 + c];
        Fv[NV - 1] = Fr[NV - 1];
#pragma unroll
        for (int v = 0; v < NV; ++v) Fv[v] = Fv[v] * a.sjac[DIR];
        T b = (Wr[0] - Wl[0]) * (Fb[0] - Fv[0]);
#pragma unroll
        for (int v = 1; v < NV; ++v) b = b + (Wr[v] - Wl[v]) * (Fb[v] - Fv[v]);
        const T dl = plain::hybrid_delta(b, a.blend, a.errflag);
#pragma unroll
        for (int v = 0; v < NV; ++v) Fx[v] = (T(1) - dl) * Fv[v] + dl * Fb[v];
    }
    __syncthreads();  // the table has been read
    if (item) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sTab[(v * N + s) * NL + l] = Fx[v];
    }
    __syncthreads();
    if (valid) {
        int f, ii;
        node_line<ND, N>(node, DIR, f, ii);
        const int ln = le * NPF + f;
        const Recip<T> iw(sw[ii]);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const T x = ii == 0 ? T(0) : sTab[(v * N + ii) * NL + ln];
            const T y = ii == N - 1 ? T(0) : sTab[(v * N + ii + 1) * NL + ln];
            acc[v] = acc[v] + iw.div(x - y);
        }
    }
    __syncthreads();  // the interface fluxes have been read
}

template <typename T, int ND, int N, int TP, bool DIAG>
__global__ void __launch_bounds__((HCfg<ND, N>::TPB)) k_hybrid(const RhsArgs<T> a) {
    using C = HCfg<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN;
    constexpr int NS = lds_slots<ND, TP>();
    constexpr int TAB = NV * (C::NPR > N * C::NL ? C::NPR : N * C::NL);
    __shared__ T sS[NS * C::SN];         // two-point flux inputs
    __shared__ T sQ[NV * C::SN];         // conservative states
    __shared__ T sW[NV * C::SN];         // entropy variables
    __shared__ T sTab[TAB];              // pair table of one direction, then its interface fluxes
    __shared__ T sFn[EPB * NF * NV * NPF];
    __shared__ T sC[N * N], sw[N], sM[ND * ND];

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const bool valid = tid < nel * NPE;
    const int le = tid / NPE, node = tid - le * NPE;
    const int64_t g0 = (int64_t)e0 * NPE;

    T q[NV], xv[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    const T* aux = stage_aux(a);
    if (aux && valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
    }
    for (int i = tid; i < N * N; i += TPB) sC[i] = (T(2) * a.ops[ops_w(N) + i / N]) * a.ops[ops_D(N) + i];
    for (int i = tid; i < N; i += TPB) sw[i] = a.ops[ops_w(N) + i];
    for (int i = tid; i < ND * ND; i += TPB) sM[i] = a.egeom[i];
    if (valid) {
        T P[NV], W[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, a.gamma, P, ir);
        const int j = Nodes<ND, N>::node(tid);
        plain::put_slots<T, ND, TP, C::SN, false>(sS + j, q, P, ir);
        plain::cons2entropy<T, ND>(q, a.gamma, a.errflag, W);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            sQ[v * C::SN + j] = q[v];
            sW[v * C::SN + j] = W[v];
        }
    }
    __syncthreads();

    // numerical fluxes on the element's faces (interface_fluxes!, applyBCs!); faces of a
    // Cartesian mesh have orientation 0 or are paired through face_nb_node
    for (int it = tid; it < EPB * NF * NPF; it += TPB) {
        const int le2 = it / (NF * NPF), r = it - le2 * (NF * NPF);
        const int k = r / NPF, f = r - k * NPF;
        if (le2 >= nel) continue;
        const int slot = (e0 + le2) * NF + k;
        const int info = a.finfo[slot], nbe = a.nb[slot];
        const T* g = a.fgeom + (int64_t)a.fgi[slot] * (3 * ND + 1);
        const int on = Nodes<ND, N>::node(le2 * NPE + line_node<ND, N>(k >> 1, f, (k & 1) ? N - 1 : 0));
        T own[NV], ext[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) own[v] = sQ[v * C::SN + on];
        if (nbe >= 0) {
            const int kp = finfo_nbpos(info);
            const T* Qn = a.Q + (int64_t)nbe * NPE +
                          line_node<ND, N>(kp >> 1, face_nb_node<ND, N>(f, info), (kp & 1) ? N - 1 : 0);
#pragma unroll
            for (int v = 0; v < NV; ++v) ext[v] = Qn[v * Nd];
        } else {
            const int bd = finfo_bd(info);
            const int type = a.bctype[bd];
            const T* src = type == BC_DIRICHLET ? a.bcstate + ((int64_t)a.fid[slot] * NPF + f) * NV
                                                : a.bcconst + bd * NV;
#pragma unroll
            for (int v = 0; v < NV; ++v) ext[v] = type == BC_DIRICHLET || type == BC_INFLOW ? src[v] : own[v];
            if (type == BC_SLIP) {
                T R[NV];
                plain::rotate2face<T, ND>(own, g, R);
                R[1] = -R[1];
                plain::rotate2phys<T, ND>(R, g, ext);
            }
        }
        const bool slave = finfo_side(info);
        T Ql[NV], Qr[NV], Rl[NV], Rr[NV], Fr[NV], F[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            Ql[v] = slave ? ext[v] : own[v];
            Qr[v] = slave ? own[v] : ext[v];
        }
        plain::rotate2face<T, ND>(Ql, g, Rl);
        plain::rotate2face<T, ND>(Qr, g, Rr);
        plain::euler_numericalflux<T, ND>(Rl, Rr, a.savg, a.sdiss, a.typo, a.intensity, a.gamma, a.errflag, Fr);
        plain::rotate2phys<T, ND>(Fr, g, F);
        const T jac = g[3 * ND];
        T* o = sFn + ((le2 * NF + k) * NV) * NPF + f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const T x = F[v] * jac;
            o[v * NPF] = slave ? -x : x;
        }
    }

    T acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    direction<T, ND, N, TP, DIAG, 0>(a, sS, sQ, sW, sTab, sC, sw, sM, nel, tid, le, node, valid, acc);
    if constexpr (ND >= 2)
        direction<T, ND, N, TP, DIAG, 1>(a, sS, sQ, sW, sTab, sC, sw, sM, nel, tid, le, node, valid, acc);
    if constexpr (ND >= 3)
        direction<T, ND, N, TP, DIAG, 2>(a, sS, sQ, sW, sTab, sC, sw, sM, nel, tid, le, node, valid, acc);
    if (!valid) return;

    // FR lift: dQ[line[ii]] -= ∂gl[ii]*Fn_left + ∂gr[ii]*Fn_right, direction by direction
#pragma unroll
    for (int dir = 0; dir < ND; ++dir) {
        int f, ii;
        node_line<ND, N>(node, dir, f, ii);
        const T gm = a.ops[ops_gm(N) + ii], gp = a.ops[ops_gp(N) + ii];
        const T* s = sFn + ((le * NF + 2 * dir) * NV) * NPF + f;
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = acc[v] - (gm * s[v * NPF] + gp * s[(NV + v) * NPF]);
    }
    const Recip<T> iJ(a.egeom[ND * ND]);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

// ---- axis-aligned elements in 1-D and 2-D --------------------------------------------------------
//
// A thread group of two waves per direction: the pair tables of all directions are filled at
// once, then one flux per thread: the N-1 interfaces of a line and its two faces (positions 0
// and N) are items of the same kind, whose numerical fluxes (the longest chain of dependent
// operations here) run side by side.  Small meshes, a block or two per CU, are bound by that
// chain (2175 elements: 3 waves per CU, VALU 26 % busy): six rounds of pairs and three of
// fluxes in k_hybrid, three and one here.  Faces read the order of their frame by index
// (faces.hpp), neighbours' traces are loaded before the pairs.
// Measured, N=5, Chandrasekhar and MatrixDissipation, 2175 elements: 25.6 -> 21 us per stage.
template <int ND, int N>
struct LCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND, NV = ND + 2;
    static constexpr int G = 128, TPB = ND * G;          // threads per direction and block
    static constexpr int EPB = G / (NPF * (N + 1));      // an item per thread
    static constexpr int NN = EPB * NPE;
    static constexpr int NL = EPB * NPF;                 // lines per direction
    static constexpr int NPAIR = N * (N - 1) / 2;
    static constexpr int NPR = NL * NPAIR;
    static constexpr int SN = EPB * Nodes<ND, N>::ES;
    static constexpr int TAB = NV * (NPAIR > N + 1 ? NPR : (N + 1) * NL);
};

template <typename T, int ND, int N, int TP, int DIR>
__device__ __forceinline__ void line_pairs(const T* sS, const T* sQ, T* sTab, T ja, T gm1, int* err, int nel, int i) {
    using C = LCfg<ND, N>;
    using M = Nodes<ND, N>;
    constexpr int NV = C::NV, SN = C::SN, NS = plain::tp_slots<ND, TP>(), NSL = lds_slots<ND, TP>();
    constexpr int ST = M::template step<DIR>();
#pragma unroll 1
    for (int k = i; k < C::NPR; k += C::G) {
        const int pr = k / C::NL, l = k - pr * C::NL;
        const int le = l / C::NPF, f = l - le * C::NPF;
        if (le >= nel) continue;
        const int ab = pair_ab<N>(pr);
        const int base = le * M::ES + M::template line<DIR>(f);
        const int ia = base + (ab >> 3) * ST, ib = base + (ab & 7) * ST;
        T A[NS], B[NS], F[NV];
#pragma unroll
        for (int c = 0; c < NS; ++c) {  // StdAverage's conservative slots lie in sQ
            A[c] = c < NSL ? sS[c * SN + ia] : T(0.5) * sQ[(1 + c - NSL) * SN + ia];
            B[c] = c < NSL ? sS[c * SN + ib] : T(0.5) * sQ[(1 + c - NSL) * SN + ib];
        }
        plain::pair_flux<T, ND, TP, DIR>(A, B, ja, gm1, err, F);
#pragma unroll
        for (int v = 0; v < NV; ++v) sTab[v * C::NPR + k] = F[v];
    }
}

template <typename T, int ND, int N, int TP>
__global__ void __launch_bounds__((LCfg<ND, N>::TPB)) k_hybrid_lines(const RhsArgs<T> a) {
    using C = LCfg<ND, N>;
    using M = Nodes<ND, N>;
    constexpr int NV = C::NV, NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NL = C::NL, SN = C::SN;
    __shared__ T sS[lds_slots<ND, TP>() * SN];  // two-point flux inputs
    __shared__ T sQ[NV * SN];                   // conservative states
    __shared__ T sW[NV * SN];                   // entropy variables
    __shared__ T sTab[ND][C::TAB];              // pair fluxes, then the fluxes at positions 0..N
    __shared__ T sC[N * N], sw[N];

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs, g0 = (int64_t)e0 * NPE;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const bool valid = tid < nel * NPE;
    const int le = tid / NPE, node = tid - le * NPE;

    // ---- the thread's item: position s of line l of its direction --------------------------
    const int dir = ND == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / C::G), it = tid - dir * C::G;
    const int s = it / NL, l = it - s * NL, fe = l / NPF, ff = l - fe * NPF;
    const bool item = s <= N && fe < nel, face = item && (s == 0 || s == N);
    int info = 0, nbe = -1, slot = 0, fgi = 0;
    if (face) {
        slot = (e0 + fe) * NF + 2 * dir + (s == N ? 1 : 0);
        info = a.finfo[slot];
        nbe = a.nb[slot];
        fgi = a.fgi[slot];
    }
    T q[NV], xv[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = valid ? a.Q[v * Nd + g0 + tid] : T(1);
    const T* aux = stage_aux(a);
    if (aux && valid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[v] = aux[v * Nd + g0 + tid];
    }
    for (int i = tid; i < N * N; i += TPB) sC[i] = (T(2) * a.ops[ops_w(N) + i / N]) * a.ops[ops_D(N) + i];
    for (int i = tid; i < N; i += TPB) sw[i] = a.ops[ops_w(N) + i];
    T ext[NV], sn = T(1), fj = T(1);
    if (face) {
        if (nbe >= 0) {
            const int kp = finfo_nbpos(info);
            load_trace<T, ND, NV>(a.Q + (int64_t)nbe * NPE +
                                      line_node<ND, N>(kp >> 1, face_nb_node<ND, N>(ff, info), (kp & 1) ? N - 1 : 0),
                                  Nd, dir, ext);
        }
        const T* g = a.fgeom + (int64_t)fgi * (3 * ND + 1);
        sn = g[dir];
        fj = g[3 * ND];
    }
    if (valid) {
        T P[NV], W[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, a.gamma, P, ir);
        const int j = M::node(tid);
        plain::put_slots<T, ND, TP, SN, false>(sS + j, q, P, ir);
        plain::cons2entropy<T, ND>(q, a.gamma, a.errflag, W);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            sQ[v * SN + j] = q[v];
            sW[v * SN + j] = W[v];
        }
    }
    __syncthreads();

    // ---- pair fluxes, each once ----------------------------------------------------------------
    T* const tab = sTab[dir];
    const T gm1 = a.gamma - T(1);
    if (dir == 0) line_pairs<T, ND, N, TP, 0>(sS, sQ, tab, a.egeom[0], gm1, a.errflag, nel, it);
    else line_pairs<T, ND, N, TP, ND - 1>(sS, sQ, tab, a.egeom[ND * ND - 1], gm1, a.errflag, nel, it);
    __syncthreads();

    // ---- the item's flux ---------------------------------------------------------------------
    T Fx[NV];
    if (item) {
        const int base = fe * M::ES + (dir == 0 ? M::template line<0>(ff) : M::template line<ND - 1>(ff));
        const int st = dir == 0 ? M::template step<0>() : M::template step<ND - 1>();
        // lower and upper node; for a face its own node, and the sides' order is the master's
        const int nr = base + (s < N ? s : N - 1) * st, nl = s == 0 || s == N ? nr : nr - st;
        T Rl[NV], Rr[NV], Vl[NV], Vr[NV], Fr[NV];
        load_trace<T, ND, NV>(sQ + nl, SN, dir, Rl);
        load_trace<T, ND, NV>(sW + nl, SN, dir, Vl);
        load_trace<T, ND, NV>(sQ + nr, SN, dir, Rr);
        load_trace<T, ND, NV>(sW + nr, SN, dir, Vr);
        const bool slave = face && finfo_side(info);
        if (face) {
            if (nbe < 0) boundary_trace<T, ND, NPF, NV>(a, info, slot, ff, dir, Rl, ext);
            T W[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) W[v] = T(0);
            if (a.sdiss == DISS_MATRIX) plain::cons2entropy<T, ND>(ext, a.gamma, a.errflag, W);
            Rl[1] = sn * Rl[1]; Rr[1] = sn * Rr[1]; ext[1] = sn * ext[1];
            Vl[1] = sn * Vl[1]; Vr[1] = sn * Vr[1]; W[1] = sn * W[1];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if (slave) { Rl[v] = ext[v]; Vl[v] = W[v]; }
                else { Rr[v] = ext[v]; Vr[v] = W[v]; }
            }
        }
        plain::euler_numericalflux<T, ND>(Rl, Rr, a.savg, a.sdiss, a.typo, a.intensity, a.gamma, a.errflag, Fr, Vl, Vr);
        if (face) {
            Fr[1] = sn * Fr[1];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const T x = Fr[v] * fj;
                Fr[v] = slave ? -x : x;
            }
        } else {
            T Fb[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) Fb[v] = T(0);
            for (int ik = s; ik < N; ++ik)
                for (int il = 0; il < s; ++il) {
                    const int pr = il * (2 * N - il - 1) / 2 + (ik - il - 1);
                    const T* t = tab + pr * NL + l;
                    const T c = sC[il * N + ik];
#pragma unroll
                    for (int v = 0; v < NV; ++v) Fb[v] = Fb[v] + c * t[v * C::NPR];
                }
            T Fv[NV], b = T(0);
#pragma unroll
            for (int v = 0; v < NV; ++v) Fv[v] = Fr[v] * a.sjac[dir];
            // the entropy production, summed over the physical variables in their order
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int w = v == 0 || v == NV - 1 ? v : face_frame<ND>(dir, v);
                const T x = (Vr[w] - Vl[w]) * (Fb[v] - Fv[w]);
                b = v == 0 ? x : b + x;
            }
            const T dl = plain::hybrid_delta(b, a.blend, a.errflag);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int w = v == 0 || v == NV - 1 ? v : face_frame<ND>(dir, v);
                Fx[v] = (T(1) - dl) * Fv[w] + dl * Fb[v];
            }
        }
        if (face) {
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int w = v == 0 || v == NV - 1 ? v : face_frame<ND>(dir, v);
                Fx[v] = Fr[w];
            }
        }
    }
    __syncthreads();  // the tables have been read
    if (item) {
#pragma unroll
        for (int v = 0; v < NV; ++v) tab[(v * (N + 1) + s) * NL + l] = Fx[v];
    }
    __syncthreads();
    if (!valid) return;

    // ---- interface differences, FR lift, mass matrix and stage epilogue --------------------------
    T acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        int f, ii;
        node_line<ND, N>(node, d, f, ii);
        const Recip<T> iw(sw[ii]);
        const T* t = sTab[d] + ii * NL + le * NPF + f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const T x = ii == 0 ? T(0) : t[v * (N + 1) * NL];
            const T y = ii == N - 1 ? T(0) : t[(v * (N + 1) + 1) * NL];
            acc[v] = acc[v] + iw.div(x - y);
        }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        int f, ii;
        node_line<ND, N>(node, d, f, ii);
        const T gm = a.ops[ops_gm(N) + ii], gp = a.ops[ops_gp(N) + ii];
        const T* t = sTab[d] + le * NPF + f;
#pragma unroll
        for (int v = 0; v < NV; ++v)
            acc[v] = acc[v] - (gm * t[v * (N + 1) * NL] + gp * t[(v * (N + 1) + N) * NL]);
    }
    const Recip<T> iJ(a.egeom[ND * ND]);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

template <typename T, int ND, int N, int TP, bool DIAG>
static hipError_t launch(const RhsArgs<T>& a, hipStream_t s) {
    using C = HCfg<ND, N>;
    hipLaunchKernelGGL((k_hybrid<T, ND, N, TP, DIAG>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

template <typename T, int ND, int N, int TP>
static hipError_t launch_lines(const RhsArgs<T>& a, hipStream_t s) {
    using C = LCfg<ND, N>;
    hipLaunchKernelGGL((k_hybrid_lines<T, ND, N, TP>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

template <typename T, int ND, int N, bool DIAG>
static hipError_t (*pick_tp(int tp))(const RhsArgs<T>&, hipStream_t) {
    switch (tp) {
        case TP_STDAVG: return &launch<T, ND, N, TP_STDAVG, DIAG>;
        case TP_CHANDRASEKHAR: return &launch<T, ND, N, TP_CHANDRASEKHAR, DIAG>;
        case TP_KENNEDY_GRUBER: return &launch<T, ND, N, TP_KENNEDY_GRUBER, DIAG>;
        default: return nullptr;
    }
}

// k_hybrid_lines on small meshes, else null: blocks that all run at once, three per CU in FP64, four
// in FP32.  k_hybrid over it, all node counts, matrix dissipation and LxF, at 256, 512 and 768 blocks: 2-D FP64 1.2 to
// 1.7, 1.0 to 1.5 and 1.04 to 1.5 (1024: 0.78 to 1.23); 2-D FP32 1.2 to 1.6, 1.2 to 1.5, 1.1 to 1.5, and at 1024
// 1.01 to 1.36 (1536: 0.95 to 1.2); 1-D FP32 1.04 to 1.2 at 256, 1.0 to 1.1 at 1024.  1-D FP64: 1.02 to 1.3 up to one
// block per CU; above that 0.88 to 1.02 while k_hybrid, whose blocks hold twice the elements and more, still has one
// per CU, then 0.99 to 1.3.
template <typename T, int ND, int N>
static hipError_t (*pick_lines(int tp, int64_t ne))(const RhsArgs<T>&, hipStream_t) {
    constexpr int CUS = 256;
    const int64_t nb = (ne + LCfg<ND, N>::EPB - 1) / LCfg<ND, N>::EPB;
    if (nb > (sizeof(T) == 8 ? 3 : 4) * CUS) return nullptr;
    if (ND == 1 && sizeof(T) == 8 && nb > CUS && (ne + HCfg<ND, N>::EPB - 1) / HCfg<ND, N>::EPB <= CUS) return nullptr;
    switch (tp) {
        case TP_STDAVG: return &launch_lines<T, ND, N, TP_STDAVG>;
        case TP_CHANDRASEKHAR: return &launch_lines<T, ND, N, TP_CHANDRASEKHAR>;
        case TP_KENNEDY_GRUBER: return &launch_lines<T, ND, N, TP_KENNEDY_GRUBER>;
        default: return nullptr;
    }
}

template <typename T, int ND, bool DIAG>
static hipError_t (*pick_n(int n, int tp))(const RhsArgs<T>&, hipStream_t) {
    switch (n) {
        case 2: return pick_tp<T, ND, 2, DIAG>(tp);
        case 3: return pick_tp<T, ND, 3, DIAG>(tp);
        case 4: return pick_tp<T, ND, 4, DIAG>(tp);
        case 5: return pick_tp<T, ND, 5, DIAG>(tp);
        case 6: return pick_tp<T, ND, 6, DIAG>(tp);
        case 7: return pick_tp<T, ND, 7, DIAG>(tp);
        case 8: return pick_tp<T, ND, 8, DIAG>(tp);
        default: return nullptr;
    }
}

}  // namespace hybrid

#if defined(FLOUHIP_PREC_F64)
#define FLOUHIP_SCALAR double
#define FLOUHIP_PTAG f64
#elif defined(FLOUHIP_PREC_F32)
#define FLOUHIP_SCALAR float
#define FLOUHIP_PTAG f32
#else
#error "define FLOUHIP_PREC_F64 or FLOUHIP_PREC_F32"
#endif
#define FLOUHIP_CAT_(k, p, d) k##p##_##d
#define FLOUHIP_CAT(k, p, d) FLOUHIP_CAT_(k, p, d)

hipError_t (*FLOUHIP_CAT(hybrid_, FLOUHIP_PTAG, FLOUHIP_ND)(int n, int tp, bool diag))(const RhsArgs<FLOUHIP_SCALAR>&,
                                                                                       hipStream_t) {
#if FLOUHIP_ND > 1
    if (!diag) return hybrid::pick_n<FLOUHIP_SCALAR, FLOUHIP_ND, false>(n, tp);
#endif
    return hybrid::pick_n<FLOUHIP_SCALAR, FLOUHIP_ND, true>(n, tp);
}

#if FLOUHIP_ND < 3
hipError_t (*FLOUHIP_CAT(hybrid_lines_, FLOUHIP_PTAG, FLOUHIP_ND)(int n, int tp, int64_t ne))(
    const RhsArgs<FLOUHIP_SCALAR>&, hipStream_t) {
    switch (n) {
        case 2: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 2>(tp, ne);
        case 3: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 3>(tp, ne);
        case 4: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 4>(tp, ne);
        case 5: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 5>(tp, ne);
        case 6: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 6>(tp, ne);
        case 7: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 7>(tp, ne);
        case 8: return hybrid::pick_lines<FLOUHIP_SCALAR, FLOUHIP_ND, 8>(tp, ne);
        default: return nullptr;
    }
}
#endif

}  // namespace flouhip
