// FP64 reductions over the state: CFL time step (get_max_dt), conservation integral
// (integrate) and monitors, plus the small element-wise helpers the host API needs.
//
// One kernel per reduction: wavefront and block reductions in registers, one partial per
// block, and the block that finishes last reduces the partials in index order (so results are
// deterministic run to run) and writes the result, the domain-error flag and the call's
// number to pinned host memory, where the host reads them.  A second kernel over the partials
// and a copy of the result cost a CFL-controlled 2-D run of 65,575 nodes about 35 us per step
// of round trips (five steps: 395 -> 316 us without them).
//
// What bounds them: HBM reads (NV·s or s bytes per node).  A thread's nodes lie a multiple of
// the nodes per element apart, so its node position within the element, and with it the
// quadrature weight, is constant and no 64-bit division is left in the loop; quotients share
// reciprocals (exact_div.hpp); on meshes with one Δx the CFL quotient is formed once from the
// largest signal speed, which gives the same rounded minimum (division by a growing speed
// is monotone).  48^3 hexahedra, N=5, FP64 (0.96 GB): get_max_dt 262 -> 186 us, entropy monitor
// 260 -> 203 us, kinetic energy 244 -> 140 us, integrate 57 -> 53 us (3.6 TB/s; a copy of 4 GiB
// moves 4.7).  At least four nodes per thread: 65,575 nodes 8.2 -> 7.1 us against one.
#include "common.hpp"
#include "exact_div.hpp"
#include "reduce.hpp"

namespace flouhip {

static constexpr int RB = 256;
static constexpr int MAX_BLOCKS = 2048;  // 8 blocks of 4 waves per CU

struct OpMin {
    static constexpr double id = INFINITY;
    __device__ static double op(double x, double y) { return (y < x) ? y : x; }
};
struct OpMax {
    static constexpr double id = -1.0;  // of non-negative speeds
    __device__ static double op(double x, double y) { return (y > x) ? y : x; }
};
struct OpSum {
    static constexpr double id = 0.0;
    __device__ static double op(double x, double y) { return x + y; }
};

template <typename OP>
__device__ inline double block_reduce(double x) {
    __shared__ double s[RB / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = OP::op(x, __shfl_xor(x, o, 64));
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) s[w] = x;
    __syncthreads();
    if (w == 0) {
        x = (l < RB / 64) ? s[l] : OP::id;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x = OP::op(x, __shfl_xor(x, o, 64));
    }
    return x;
}

// Result to the host: value, error flag, then the call's number (the host waits for it).
__device__ inline void publish(const ReduceOut& r, double x) {
    r.host->value = x;
    r.host->flag = __hip_atomic_load(r.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&r.host->seq, r.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sets an error bit and waits until it is set (the block's arrival follows a barrier).
__device__ inline void raise(int* err, int bit) {
    __hip_atomic_fetch_or(err, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Block partials, reduced by the block that arrives last; fin maps the reduced value to the
// result.  A partial is an agent-scope atomic store, written through to where every XCD reads
// it, and the wait before the arrival lets it complete there; a release at agent scope would
// write back the whole L2 as well, once per block (2048 blocks: integrate 53 -> 134 us).  The
// error flag is raised by atomics at the same scope.
template <typename OP, typename FIN>
__device__ inline void finish(double x, const ReduceOut& r, FIN fin) {
    __shared__ bool last;
    x = block_reduce<OP>(x);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&r.partial[blockIdx.x], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        last = __hip_atomic_fetch_add(r.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    double y = OP::id;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += RB)
        y = OP::op(y, __hip_atomic_load(&r.partial[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    __syncthreads();  // block_reduce's shared values are free again
    y = block_reduce<OP>(y);
    if (threadIdx.x == 0) {
        __hip_atomic_store(r.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        publish(r, fin(y));
    }
}

// The nodes of a thread: i = first, first + step, .. with step a multiple of npe; e and k,
// element and node in the element, of the first (k is the same for all).
struct Walk {
    int64_t i, step, e, estep;
    int k;
    __device__ Walk(int64_t ndofs, int npe) {
        const unsigned total = gridDim.x * RB, t = blockIdx.x * RB + threadIdx.x;
        const unsigned used = total / npe;  // elements the grid covers at once
        step = (int64_t)used * npe;
        estep = used;
        e = t / (unsigned)npe;
        k = (int)(t - (unsigned)e * npe);
        i = t < step ? t : ndofs;
    }
};

// Signal speed |u| + c of node i.
template <typename T, int ND>
__device__ inline double signal_speed(const T* __restrict__ Q, int64_t ndofs, int64_t i, double gamma, bool& bad) {
    double q[ND + 2];
#pragma unroll
    for (int v = 0; v < ND + 2; ++v) q[v] = (double)Q[v * ndofs + i];
    const Recip<double> ir(q[0]);
    double s = q[1] * q[1];
#pragma unroll
    for (int k = 1; k < ND; ++k) s = s + q[1 + k] * q[1 + k];
    const double p = (gamma - 1.0) * (q[ND + 1] - ir.div2(s));
    const double c2 = ir.div(gamma * p);
    bad |= c2 < 0.0;
    const double c = sqrt(c2);
    double u = ir.div(q[1]);
    if (ND == 1) return fabs(u) + c;
    double ss = u * u;
#pragma unroll
    for (int k = 1; k < ND; ++k) {
        u = ir.div(q[1 + k]);
        ss = ss + u * u;
    }
    return sqrt(ss) + c;
}

// Local Δt = cfl Δx / (|u| + c) per node in FP64 (FlouCommon/Euler.jl:116-135;
// LinearAdvection.jl:46-48), Δx = (vol / n^d)^(1/d) per element, min over nodes.
// UNI: one Δx (dxe[0]) and cfl > 0.
template <typename T, int ND, bool UNI>
__global__ void __launch_bounds__(RB) k_max_dt(const T* __restrict__ Q, int64_t ndofs, int npe, double gamma,
                                               double cfl, const double* __restrict__ dxe, ReduceOut r) {
    const Walk w(ndofs, npe);
    double m = UNI ? OpMax::id : OpMin::id;
    bool bad = false;
    int64_t e = w.e;
#pragma unroll 2
    for (int64_t i = w.i; i < ndofs; i += w.step, e += w.estep) {
        const double s = signal_speed<T, ND>(Q, ndofs, i, gamma, bad);
        m = UNI ? OpMax::op(m, s) : OpMin::op(m, cfl * dxe[e] / s);
    }
    if (bad) raise(r.err, ERR_SQRT_NEG);
    if constexpr (UNI)
        finish<OpMax>(m, r, [&](double s) { return s < 0.0 ? (double)INFINITY : cfl * dxe[0] / s; });
    else
        finish<OpMin>(m, r, [](double x) { return x; });
}

// Linear advection: the smallest Δx over the constant speed.
__global__ void __launch_bounds__(RB) k_max_dt_adv(int64_t ne, double cfl, double anorm,
                                                   const double* __restrict__ dxe, ReduceOut r) {
    double m = OpMin::id;
    for (int64_t e = (int64_t)blockIdx.x * RB + threadIdx.x; e < ne; e += (int64_t)gridDim.x * RB)
        m = OpMin::op(m, cfl * dxe[e] / anorm);
    finish<OpMin>(m, r, [](double x) { return x; });
}

// Σ_e Σ_i J_e ω_i s(Q)_i with s the nodal value Q_i (KIND -1: MultielementDiscontinuous.jl:
// 148-160), the kinetic energy (0) or the mathematical entropy (1) (Euler.jl:541-590).  Curved
// elements: npe = 1, jac per node.
template <typename T, int ND, int KIND>
__device__ inline double density(const T* __restrict__ Q, int64_t ndofs, int64_t i, double gamma, bool& bad) {
    if constexpr (KIND < 0) return (double)Q[i];
    constexpr int NQ = KIND == 0 ? ND + 1 : ND + 2;
    double q[ND + 2];
#pragma unroll
    for (int v = 0; v < NQ; ++v) q[v] = (double)Q[v * ndofs + i];
    double m2 = q[1] * q[1];
#pragma unroll
    for (int k = 1; k < ND; ++k) m2 = m2 + q[1 + k] * q[1 + k];
    const double ke = Recip<double>(q[0]).div2(m2);
    if constexpr (KIND == 0) return ke;
    const double p = (gamma - 1.0) * (q[ND + 1] - ke);
    bad |= p < 0.0 || q[0] < 0.0;
    const double ent = log(p) - gamma * log(q[0]);
    return -(q[0] * ent);
}

template <typename T, int ND, int KIND>
__global__ void __launch_bounds__(RB) k_sum(const T* __restrict__ Q, int64_t ndofs, int npe, double gamma,
                                            const double* __restrict__ jac, const double* __restrict__ w,
                                            ReduceOut r) {
    const Walk k(ndofs, npe);
    const double wk = w[k.k];
    const Recip<double> ig(gamma - 1.0);
    double s = 0.0;
    bool bad = false;
    int64_t e = k.e;
#pragma unroll 4
    for (int64_t i = k.i; i < ndofs; i += k.step, e += k.estep) {
        const double d = density<T, ND, KIND>(Q, ndofs, i, gamma, bad);
        s += (jac[e] * wk) * (KIND == 1 ? ig.div(d) : d);
    }
    if (bad) raise(r.err, ERR_LOG_NEG);
    finish<OpSum>(s, r, [](double x) { return x; });
}

// The domain-error flag to the host.
__global__ void k_flag(ReduceOut r) {
    if (threadIdx.x == 0) publish(r, 0.0);
}

// Blocks of a reduction over n items, each covering at least one element of npe nodes.
static int grid_for(int64_t n, int npe) {
    int64_t g = (n + 4 * RB - 1) / (4 * RB);
    if (g > MAX_BLOCKS) g = MAX_BLOCKS;
    const int least = (npe + RB - 1) / RB;
    return (int)(g < least ? least : g);
}

template <typename T, int ND>
static void max_dt_nd(const T* Q, int64_t ndofs, int npe, double gamma, double cfl, bool uniform, const double* dxe,
                      const ReduceOut& r, hipStream_t s) {
    const dim3 g(grid_for(ndofs, npe)), b(RB);
    if (uniform && cfl > 0.0)
        hipLaunchKernelGGL((k_max_dt<T, ND, true>), g, b, 0, s, Q, ndofs, npe, gamma, cfl, dxe, r);
    else
        hipLaunchKernelGGL((k_max_dt<T, ND, false>), g, b, 0, s, Q, ndofs, npe, gamma, cfl, dxe, r);
}

template <typename T>
hipError_t launch_max_dt(const T* Q, int64_t ndofs, int npe, int nd, int eq, double gamma,
                         double anorm, double cfl, const double* dxe, bool uniform, const ReduceOut& r, hipStream_t s) {
    if (eq == EQ_ADVECTION)
        hipLaunchKernelGGL(k_max_dt_adv, dim3(grid_for(ndofs / npe, 1)), dim3(RB), 0, s, ndofs / npe, cfl, anorm, dxe, r);
    else if (nd == 1)
        max_dt_nd<T, 1>(Q, ndofs, npe, gamma, cfl, uniform, dxe, r, s);
    else if (nd == 2)
        max_dt_nd<T, 2>(Q, ndofs, npe, gamma, cfl, uniform, dxe, r, s);
    else
        max_dt_nd<T, 3>(Q, ndofs, npe, gamma, cfl, uniform, dxe, r, s);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_integrate(const T* Q, int64_t ndofs, int npe, const double* jac, const double* w, const ReduceOut& r,
                            hipStream_t s) {
    hipLaunchKernelGGL((k_sum<T, 1, -1>), dim3(grid_for(ndofs, npe)), dim3(RB), 0, s, Q, ndofs, npe, 1.4, jac, w, r);
    return hipGetLastError();
}

template <typename T, int ND>
static void monitor_nd(const T* Q, int64_t ndofs, int npe, double gamma, int kind, const double* jac, const double* w,
                       const ReduceOut& r, hipStream_t s) {
    const dim3 g(grid_for(ndofs, npe)), b(RB);
    if (kind == 0)
        hipLaunchKernelGGL((k_sum<T, ND, 0>), g, b, 0, s, Q, ndofs, npe, gamma, jac, w, r);
    else
        hipLaunchKernelGGL((k_sum<T, ND, 1>), g, b, 0, s, Q, ndofs, npe, gamma, jac, w, r);
}

template <typename T>
hipError_t launch_monitor(const T* Q, int64_t ndofs, int npe, int nd, double gamma, int kind, const double* jac,
                          const double* w, const ReduceOut& r, hipStream_t s) {
    if (nd == 1) monitor_nd<T, 1>(Q, ndofs, npe, gamma, kind, jac, w, r, s);
    else if (nd == 2) monitor_nd<T, 2>(Q, ndofs, npe, gamma, kind, jac, w, r, s);
    else monitor_nd<T, 3>(Q, ndofs, npe, gamma, kind, jac, w, r, s);
    return hipGetLastError();
}

hipError_t launch_flag(const ReduceOut& r, hipStream_t s) {
    hipLaunchKernelGGL(k_flag, dim3(1), dim3(64), 0, s, r);
    return hipGetLastError();
}

template hipError_t launch_max_dt<double>(const double*, int64_t, int, int, int, double, double, double,
                                          const double*, bool, const ReduceOut&, hipStream_t);
template hipError_t launch_max_dt<float>(const float*, int64_t, int, int, int, double, double, double,
                                         const double*, bool, const ReduceOut&, hipStream_t);
template hipError_t launch_integrate<double>(const double*, int64_t, int, const double*, const double*,
                                             const ReduceOut&, hipStream_t);
template hipError_t launch_integrate<float>(const float*, int64_t, int, const double*, const double*,
                                            const ReduceOut&, hipStream_t);
template hipError_t launch_monitor<double>(const double*, int64_t, int, int, double, int, const double*,
                                           const double*, const ReduceOut&, hipStream_t);
template hipError_t launch_monitor<float>(const float*, int64_t, int, int, double, int, const double*, const double*,
                                          const ReduceOut&, hipStream_t);

int reduce_max_blocks() { return MAX_BLOCKS; }

}  // namespace flouhip
