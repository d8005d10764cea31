// Stage limiter of the Euler path (Equations/Euler.jl:596-654).
//
// k_zhang_shu: Flou's Zhang & Shu positivity limiter.  Element means and minima are
// sequential folds over the element's nodes (the reference's order), so the FP64 result is
// reproducible bit for bit.
#include "common.hpp"
#include "reduce.hpp"

namespace flouhip {

static constexpr int LB = 256;  // limiter block

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

template hipError_t launch_zhang_shu<double>(double*, int64_t, int64_t, int, int, int, const double*,
                                             const double*, const double*, double, double, hipStream_t);
template hipError_t launch_zhang_shu<float>(float*, int64_t, int64_t, int, int, int, const double*,
                                            const double*, const double*, double, double, hipStream_t);

}  // namespace flouhip
