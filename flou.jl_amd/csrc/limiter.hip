// Stage limiter and monitors of the Euler path (Equations/Euler.jl:541-654).
//
// k_zhang_shu: Flou's Zhang & Shu positivity limiter.  Element means and minima are
// sequential folds over the element's nodes (the reference's order), so the FP64 result is
// reproducible bit for bit.
// k_monitor: Σ Jω · s(Q) with s the kinetic energy or the mathematical entropy, FP64
// accumulation, block partials + one finishing block (fixed tree, deterministic).
#include "common.hpp"
#include "reduce.hpp"

namespace flouhip {

static constexpr int LB = 256;  // limiter block
static constexpr int MB = 256;  // monitor block

// Elements per limiter block, the LDS stride of an element's nodes (odd: the folds' lanes,
// one element apart, then read distinct banks) and the block's LDS values.
__host__ __device__ constexpr int lim_epb(int npe) { return npe >= LB ? 1 : LB / npe; }
__host__ __device__ constexpr int lim_stride(int npe) { return npe | 1; }
__host__ __device__ constexpr int lim_lds(int npe, int nv) {
    return lim_epb(npe) * ((nv + 2) * lim_stride(npe) + nv + 3);
}

// Nodes are loaded and written coalesced, one thread per node; the means and minima are the
// reference's sequential folds, one lane per (element, variable) over the staged nodes.  An
// element per thread, which read a cache line per lane and node, took 22 us on 2175 2-D
// elements at N=5 in FP64; this 6.5 us.
template <typename T, int NV>
__global__ void __launch_bounds__(LB) k_zhang_shu(T* __restrict__ Q, int64_t ndofs, int64_t ne, int npe,
                                                 int wnpe, const double* __restrict__ jac,
                                                 const double* __restrict__ w,
                                                 const double* __restrict__ vol, T minval, T gamma) {
    constexpr int ND = NV - 2, NM = NV + 3;
    extern __shared__ double lim_smem[];
    const int epb = lim_epb(npe), ps = lim_stride(npe), S = epb * ps;
    T* const sq = reinterpret_cast<T*>(lim_smem);  // [v][element][node]
    T* const sj = sq + NV * S;                     // quadrature weights Jω
    T* const sp = sj + S;                          // pressures
    T* const sm = sp + S;                          // per element: means, density minimum, mean and least pressure
    const int64_t e0 = (int64_t)blockIdx.x * epb, g0 = e0 * npe;
    const int nel = ne - e0 < epb ? (int)(ne - e0) : epb;
    const int nn = nel * npe, tid = threadIdx.x;
    for (int j = tid; j < nn; j += LB) {
        const int le = j / npe, i = j - le * npe, o = le * ps + i;
#pragma unroll
        for (int v = 0; v < NV; ++v) sq[v * S + o] = Q[v * ndofs + g0 + j];
        // wnpe is npe (J per element) or 1 (Jω per node)
        sj[o] = (T)(wnpe == 1 ? jac[g0 + j] * w[0] : jac[e0 + le] * w[i]);
    }
    __syncthreads();
    // element means and density minimum
    for (int t = tid; t < nel * (NV + 1); t += LB) {
        const int le = t / (NV + 1), v = t - le * (NV + 1);
        const T* c = sj + le * ps;
        if (v < NV) {
            const T* x = sq + v * S + le * ps;
            T s = T(0);
            for (int i = 0; i < npe; ++i) s = s + c[i] * x[i];
            sm[le * NM + v] = s / (T)vol[e0 + le];
        } else {
            const T* x = sq + le * ps;
            T r = x[0];
            for (int i = 0; i < npe; ++i) r = x[i] < r ? x[i] : r;
            sm[le * NM + NV] = r;
        }
    }
    __syncthreads();
    // density limiting and the pressures of the updated nodes
    for (int j = tid; j < nn; j += LB) {
        const int le = j / npe, o = le * ps + (j - le * npe);
        const T qm = sm[le * NM], rmin = sm[le * NM + NV];
        const T m = minval < qm ? minval : qm;
        const T th = fabs((qm - m) / (qm - rmin));
        T r = sq[o];
        if (th <= T(1)) {
            r = th * (r - qm) + qm;
            sq[o] = r;
            Q[g0 + j] = r;
        }
        T s = sq[S + o] * sq[S + o];
#pragma unroll
        for (int k = 1; k < ND; ++k) s = s + sq[(1 + k) * S + o] * sq[(1 + k) * S + o];
        sp[o] = (gamma - T(1)) * (sq[(ND + 1) * S + o] - s / (T(2) * r));
    }
    __syncthreads();
    for (int t = tid; t < 2 * nel; t += LB) {
        const int le = t >> 1;
        const T* x = sp + le * ps;
        if (t & 1) {
            T r = x[0];
            for (int i = 1; i < npe; ++i) r = x[i] < r ? x[i] : r;
            sm[le * NM + NV + 2] = r;
        } else {
            const T* c = sj + le * ps;
            T s = T(0);
            for (int i = 0; i < npe; ++i) s = s + c[i] * x[i];
            sm[le * NM + NV + 1] = s / (T)vol[e0 + le];
        }
    }
    __syncthreads();
    // pressure limiting: every variable towards its mean
    for (int j = tid; j < nn; j += LB) {
        const int le = j / npe, o = le * ps + (j - le * npe);
        const T pm = sm[le * NM + NV + 1], pmin = sm[le * NM + NV + 2];
        const T m = minval < pm ? minval : pm;
        const T th = fabs((pm - m) / (pm - pmin));
        if (th <= T(1)) {
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const T qm = sm[le * NM + v];
                Q[v * ndofs + g0 + j] = th * (sq[v * S + o] - qm) + qm;
            }
        }
    }
}

__device__ inline double mwarp_sum(double x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

template <typename T>
__global__ void __launch_bounds__(MB) k_monitor(const T* __restrict__ Q, int64_t ndofs, int wnpe, int nd,
                                               double gamma, int kind, const double* __restrict__ jac,
                                               const double* __restrict__ w, double* __restrict__ partial,
                                               int* err) {
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * MB + threadIdx.x; i < ndofs; i += (int64_t)gridDim.x * MB) {
        double q[5];
        for (int v = 0; v < nd + 2; ++v) q[v] = (double)Q[v * ndofs + i];
        double m2 = q[1] * q[1];
        for (int k = 1; k < nd; ++k) m2 = m2 + q[1 + k] * q[1 + k];
        double val;
        if (kind == 0) {
            val = m2 / (2.0 * q[0]);
        } else {
            const double p = (gamma - 1.0) * (q[nd + 1] - m2 / (2.0 * q[0]));
            if (p < 0.0 || q[0] < 0.0) atomicOr(err, ERR_LOG_NEG);
            const double ent = log(p) - gamma * log(q[0]);
            val = -(q[0] * ent) / (gamma - 1.0);
        }
        const int64_t k = i / wnpe;
        s += (jac[k] * w[i - k * wnpe]) * val;
    }
    __shared__ double sh[MB / 64];
    s = mwarp_sum(s);
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) sh[wv] = s;
    __syncthreads();
    if (wv == 0) {
        s = l < MB / 64 ? sh[l] : 0.0;
        s = mwarp_sum(s);
        if (l == 0) partial[blockIdx.x] = s;
    }
}

__global__ void __launch_bounds__(MB) k_monitor_finish(const double* __restrict__ partial, int n,
                                                      double* __restrict__ out) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += MB) s += partial[i];
    __shared__ double sh[MB / 64];
    s = mwarp_sum(s);
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) sh[wv] = s;
    __syncthreads();
    if (wv == 0) {
        s = l < MB / 64 ? sh[l] : 0.0;
        s = mwarp_sum(s);
        if (l == 0) *out = s;
    }
}

template <typename T>
hipError_t launch_zhang_shu(T* Q, int64_t ndofs, int64_t ne, int npe, int nd, int wnpe,
                            const double* jac, const double* w, const double* vol, double minval,
                            double gamma, hipStream_t s) {
    const int epb = lim_epb(npe);
    const int g = (int)((ne + epb - 1) / epb);
    const size_t lds = lim_lds(npe, nd + 2) * sizeof(T);
    if (nd == 1)
        hipLaunchKernelGGL((k_zhang_shu<T, 3>), dim3(g), dim3(LB), lds, s, Q, ndofs, ne, npe, wnpe, jac, w, vol, (T)minval, (T)gamma);
    else if (nd == 2)
        hipLaunchKernelGGL((k_zhang_shu<T, 4>), dim3(g), dim3(LB), lds, s, Q, ndofs, ne, npe, wnpe, jac, w, vol, (T)minval, (T)gamma);
    else
        hipLaunchKernelGGL((k_zhang_shu<T, 5>), dim3(g), dim3(LB), lds, s, Q, ndofs, ne, npe, wnpe, jac, w, vol, (T)minval, (T)gamma);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_monitor(const T* Q, int64_t ndofs, int wnpe, int nd, double gamma, int kind,
                          const double* jac, const double* w, double* partial, int max_blocks,
                          double* out, int* err, hipStream_t s) {
    int64_t g = (ndofs + MB - 1) / MB;
    if (g > max_blocks) g = max_blocks;
    if (g < 1) g = 1;
    hipLaunchKernelGGL(k_monitor<T>, dim3((int)g), dim3(MB), 0, s, Q, ndofs, wnpe, nd, gamma, kind, jac, w,
                       partial, err);
    hipLaunchKernelGGL(k_monitor_finish, dim3(1), dim3(MB), 0, s, partial, (int)g, out);
    return hipGetLastError();
}

template hipError_t launch_zhang_shu<double>(double*, int64_t, int64_t, int, int, int, const double*,
                                             const double*, const double*, double, double, hipStream_t);
template hipError_t launch_zhang_shu<float>(float*, int64_t, int64_t, int, int, int, const double*,
                                            const double*, const double*, double, double, hipStream_t);
template hipError_t launch_monitor<double>(const double*, int64_t, int, int, double, int, const double*,
                                           const double*, double*, int, double*, int*, hipStream_t);
template hipError_t launch_monitor<float>(const float*, int64_t, int, int, double, int, const double*,
                                          const double*, double*, int, double*, int*, hipStream_t);

}  // namespace flouhip
