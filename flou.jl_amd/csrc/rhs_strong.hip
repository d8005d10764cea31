// Strong-form rhs on axis-aligned affine elements (Flou's CartesianMesh), GLL nodes: Euler with
// the StdAverage or LxF(StdAverage) surface flux, and linear advection; with the RK stage
// epilogue.  The plain kernel's arithmetic (rhs_plain.hip, every FP64 value rounded where the
// reference rounds it) without the work that this geometry makes void.
//
// What bounds it: HBM at large sizes and, below, the chain of dependent loads and barriers.
//   * a node's primitives are formed once, for the contravariant fluxes of all directions, each
//     of one term (the metric is diagonal), and stay in registers;
//   * the fluxes lie in LDS in vectors of 16 bytes, so that a line's entry is one or two reads;
//   * all loads come first, the face tables, then the node's state and the neighbours' traces:
//     two dependent global loads from start to end;
//   * faces as in faces.hpp; the lift touches the end nodes only (∂g is exactly zero elsewhere).
// Measured against k_plain, rhs, 0.9 M nodes, Euler, N nodes per line: 3-D N=5 FP32 37.8 -> 22 us,
// FP64 72 -> 35; 3-D N=8 FP32 46 -> 18.6, FP64 130 -> 33; 2-D N=6 FP32 20.5 -> 13.4, FP64 37 -> 20.  An
// SSPRK33 step of 7182 elements, 3-D N=5, FP32: 116 -> 64 us; ten of advection on 256 elements, 2-D
// N=5, FP64: 163 -> 148 us.  Blocks of 128 threads: 2-D N=6 FP32 15.8 us, FP64 26.  (FP32 with fused
// operations: 57 us, but the 2N schemes' register, a small difference of large sums, then differs
// from the plain kernel's in its third digit.)
// Compile with -DFLOUHIP_PREC_F64 or -DFLOUHIP_PREC_F32 and -DFLOUHIP_ND=1|2|3.
#include "common.hpp"
#include "faces.hpp"
#include "physics_plain.hpp"
#include "stage.hpp"

namespace flouhip {
namespace strong {

template <int ND, int N>
struct TCfg {
    static constexpr int NPE = Cfg<ND, N>::NPE, NPF = Cfg<ND, N>::NPF, NF = 2 * ND;
    static constexpr int EPB = NPE >= 256 ? 1 : 256 / NPE;
    static constexpr int NN = EPB * NPE;               // nodes per block
    static constexpr int TPB = block_threads(NN);      // threads per block
    static constexpr int NFN = EPB * NF * NPF;         // face nodes per block
    static constexpr int NR = (NFN + TPB - 1) / TPB;   // face nodes per thread
};

// NV values per node of NN nodes in LDS, in vectors of 16 bytes as far as they go.
template <typename T, int NV, int NN>
struct Table {
    static constexpr int W = 16 / sizeof(T), NVV = NV / W;
    static constexpr int SIZE = (NV * NN + W - 1) / W * W;
    typedef T Vec __attribute__((ext_vector_type(16 / sizeof(T))));
    __device__ __forceinline__ static void put(T* s, int j, const T* x) {
#pragma unroll
        for (int k = 0; k < NVV; ++k) {
            Vec y;
#pragma unroll
            for (int c = 0; c < W; ++c) y[c] = x[k * W + c];
            *reinterpret_cast<Vec*>(s + (k * NN + j) * W) = y;
        }
#pragma unroll
        for (int v = NVV * W; v < NV; ++v) s[v * NN + j] = x[v];
    }
    __device__ __forceinline__ static void get(const T* s, int j, T* x) {
#pragma unroll
        for (int k = 0; k < NVV; ++k) {
            const Vec y = *reinterpret_cast<const Vec*>(s + (k * NN + j) * W);
#pragma unroll
            for (int c = 0; c < W; ++c) x[k * W + c] = y[c];
        }
#pragma unroll
        for (int v = NVV * W; v < NV; ++v) x[v] = s[v * NN + j];
    }
};

template <typename T, int ND, int N, int EQ>
__global__ void __launch_bounds__((TCfg<ND, N>::TPB)) k_strong(const RhsArgs<T> a) {
    using C = TCfg<ND, N>;
    constexpr int NV = EQ == EQ_ADVECTION ? 1 : ND + 2;
    constexpr int NPE = C::NPE, NPF = C::NPF, NF = C::NF, EPB = C::EPB, TPB = C::TPB, NN = C::NN, NR = C::NR;
    using Tab = Table<T, NV, NN>;
    // Own traces from LDS, or from memory beside the neighbours' where a block per CU more fits
    // without the states (rhs, 0.9 M nodes, N nodes per line, LDS and memory: FP64 3-D N=4 45 and
    // 38 us, N=7 60 and 47, N=8 44 and 33; FP32 3-D N=7 25.2 and 22.4, N=5 22.1 and 22.9, 2-D FP64
    // N=6 20.9 and 22.4).
    constexpr bool GLB = ND == 3 && (sizeof(T) == 8 ? N > 2 : N == 7);
    __shared__ __align__(16) T sF[ND][Tab::SIZE];  // contravariant fluxes per direction
    __shared__ T sQ[GLB ? 1 : NV * NN];            // states, for the own traces
    __shared__ T sFn[NV * C::NFN];                 // face fluxes [face][v][face node]
    __shared__ T sD[N * N];

    const int tid = threadIdx.x;
    const int e0 = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int64_t Nd = a.ndofs, g0 = (int64_t)e0 * NPE;
    const int nel = a.ne - e0 < EPB ? a.ne - e0 : EPB;
    const bool valid = tid < nel * NPE;
    const int le = tid / NPE, node = tid - le * NPE;
    const T avel[3] = {a.a0, a.a1, a.a2};

    // ---- loads: face tables, own node, geometry; then what depends on the tables -------------
    // (spare lanes and boundary faces load something valid instead of branching)
    int fs[NR], info[NR], nbe[NR], fgi[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int it = tid + r * TPB;
        fs[r] = e0 * NF + (it < nel * NF * NPF ? it / NPF : 0);  // face slot of face node `it`
        info[r] = a.finfo[fs[r]];
        nbe[r] = a.nb[fs[r]];
        fgi[r] = a.fgi[fs[r]];
    }
    const int tn = valid ? tid : 0;
    T q[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = (a.Q + (v * Nd + g0))[tn];
    const T* eg = a.egeom + (int64_t)(valid ? e0 + le : e0) * a.egeom_stride;
    T ja[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) ja[d] = eg[d * (ND + 1)];
    const T jac = eg[ND * ND];
    const T Dv = a.ops[ops_Ds(N) + (tid < N * N ? tid : 0)];
    T own[NR][NV], ext[NR][NV], sn[NR], fj[NR], xv[NV];
    const T* aux = stage_aux(a);
    if (aux) {
#pragma unroll
        for (int v = 0; v < NV; ++v) xv[v] = (aux + (v * Nd + g0))[tn];
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int it = tid + r * TPB;
        const int k = (it / NPF) % NF, f = it % NPF, dir = k >> 1;
        const int kp = nbe[r] >= 0 ? finfo_nbpos(info[r]) : 0;
        load_trace<T, ND, NV>(a.Q + (int64_t)(nbe[r] >= 0 ? nbe[r] : e0) * NPE +
                                  line_node<ND, N>(kp >> 1, f, (kp & 1) ? N - 1 : 0),
                              Nd, dir, ext[r]);
        if constexpr (GLB) {
            const int le2 = it < nel * NF * NPF ? it / (NF * NPF) : 0;
            load_trace<T, ND, NV>(a.Q + g0 + le2 * NPE + line_node<ND, N>(dir, f, (k & 1) ? N - 1 : 0), Nd, dir, own[r]);
        }
        const T* g = a.fgeom + (int64_t)fgi[r] * (3 * ND + 1);
        sn[r] = g[dir];
        fj[r] = g[3 * ND];
    }

    // ---- contravariant fluxes ------------------------------------------------------------
    T F[ND][NV];
    if constexpr (EQ == EQ_ADVECTION) {
#pragma unroll
        for (int d = 0; d < ND; ++d) F[d][0] = (avel[d] * q[0]) * ja[d];
    } else {
        T P[NV];
        const Recip<T> ir(q[0]);
        plain::cons2prim<T, ND>(q, a.gamma, P, ir);
        const T p = P[ND + 1];
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const T u = P[1 + d];
            F[d][0] = q[1 + d] * ja[d];
#pragma unroll
            for (int c = 0; c < ND; ++c)
                F[d][1 + c] = (c == d ? q[1 + d] * P[1 + c] + p : q[1 + d] * P[1 + c]) * ja[d];
            F[d][NV - 1] = ((q[NV - 1] + p) * u) * ja[d];
        }
    }
    if (valid) {
#pragma unroll
        for (int d = 0; d < ND; ++d) Tab::put(sF[d], tid, F[d]);
        if constexpr (!GLB) {
#pragma unroll
            for (int v = 0; v < NV; ++v) sQ[v * NN + tid] = q[v];
        }
    }

    if (tid < N * N) sD[tid] = Dv;
    __syncthreads();

    // ---- volume terms, in the reference's order ------------------------------------------------
    T acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = T(0);
    if (valid) {
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            int f, ii;
            node_line<ND, N>(node, d, f, ii);
            constexpr int S[3] = {1, N, N * N};
            const int base = tid - ii * S[d];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const T Dik = sD[ii * N + k];
                T x[NV];
                Tab::get(sF[d], base + k * S[d], x);
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[v] = acc[v] - Dik * x[v];
            }
        }
    }

    // ---- numerical fluxes on the element's faces --------------------------------------------------
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int it = tid + r * TPB;
        if (it >= nel * NF * NPF) continue;
        const int k = (it / NPF) % NF, f = it % NPF, dir = k >> 1;
        if constexpr (!GLB)
            load_trace<T, ND, NV>(sQ + it / (NF * NPF) * NPE + line_node<ND, N>(dir, f, (k & 1) ? N - 1 : 0), NN, dir,
                                  own[r]);
        if (nbe[r] < 0) boundary_trace<T, ND, NPF, NV>(a, info[r], fs[r], f, dir, own[r], ext[r]);
        const bool slave = finfo_side(info[r]);
        T* o = sFn + (it / NPF) * (NV * NPF) + f;
        if constexpr (EQ == EQ_ADVECTION) {
            const T an = (dir == 0 ? avel[0] : dir == 1 ? avel[1] : avel[2]) * sn[r];
            const T sg = slave ? T(-1) : T(1);
            T Fn = (an * (own[r][0] + ext[r][0])) / T(2);
            if (a.sdiss == DISS_LXF) Fn = Fn + sg * (((fabs(an) * (own[r][0] - ext[r][0])) / T(2)) * a.intensity);
            o[0] = Fn * (sg * fj[r]);
        } else {
            T Fn[NV];
            axis_flux<T, ND>(own[r], ext[r], sn[r], fj[r], slave, a.sdiss, a.gamma, a.intensity, a.errflag, Fn);
            o[0] = Fn[0];
#pragma unroll
            for (int c = 0; c < ND; ++c) o[face_mom<ND>(dir, c) * NPF] = Fn[1 + c];
            o[(NV - 1) * NPF] = Fn[NV - 1];
        }
    }
    __syncthreads();
    if (!valid) return;

    // ---- FR lift on the end nodes, mass matrix and stage epilogue -----------------------------
    const T gm0 = a.ops[ops_gm(N)], gpn = a.ops[ops_gp(N) + N - 1];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        int f, ii;
        node_line<ND, N>(node, d, f, ii);
        if (ii == 0 || ii == N - 1) {
            const T* s = sFn + (le * NF + 2 * d + (ii ? 1 : 0)) * (NV * NPF) + f;
            const T c = ii ? gpn : gm0;
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = acc[v] - c * s[v * NPF];
        }
    }
    const Recip<T> iJ(jac);
    const StageOut<T> so(a);
#pragma unroll
    for (int v = 0; v < NV; ++v) so.put(v * Nd + g0 + tid, iJ.div(acc[v]), q[v], xv[v]);
}

template <typename T, int ND, int N, int EQ>
static hipError_t launch(const RhsArgs<T>& a, hipStream_t s) {
    using C = TCfg<ND, N>;
    hipLaunchKernelGGL((k_strong<T, ND, N, EQ>), dim3((a.ne + C::EPB - 1) / C::EPB), dim3(C::TPB), 0, s, a);
    return hipGetLastError();
}

template <typename T, int ND, int N>
static hipError_t (*pick(int eq))(const RhsArgs<T>&, hipStream_t) {
    return eq == EQ_ADVECTION ? &launch<T, ND, N, EQ_ADVECTION> : &launch<T, ND, N, EQ_EULER>;
}

}  // namespace strong

#if defined(FLOUHIP_PREC_F64)
#define FLOUHIP_SCALAR double
#define FLOUHIP_PTAG strong_f64_
#elif defined(FLOUHIP_PREC_F32)
#define FLOUHIP_SCALAR float
#define FLOUHIP_PTAG strong_f32_
#else
#error "define FLOUHIP_PREC_F64 or FLOUHIP_PREC_F32"
#endif

#define FLOUHIP_CAT_(a, b) a##b
#define FLOUHIP_CAT(a, b) FLOUHIP_CAT_(a, b)

hipError_t (*FLOUHIP_CAT(FLOUHIP_PTAG, FLOUHIP_ND)(int n, int eq))(const RhsArgs<FLOUHIP_SCALAR>&, hipStream_t) {
    switch (n) {
        case 2: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 2>(eq);
        case 3: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 3>(eq);
        case 4: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 4>(eq);
        case 5: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 5>(eq);
        case 6: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 6>(eq);
        case 7: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 7>(eq);
        case 8: return strong::pick<FLOUHIP_SCALAR, FLOUHIP_ND, 8>(eq);
        default: return nullptr;
    }
}

}  // namespace flouhip
