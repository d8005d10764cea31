// Launchers of the FP64 reductions (reduce.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace flouhip {

// Where the last block of a reduction leaves its result for the host: pinned, coherent memory.
struct HostResult {
    double value;
    int flag;                 // the domain-error flag after every earlier kernel of the stream
    unsigned long long seq;   // number of the call that wrote it
};

// Output of a reduction: the host's result, the call's number, the block partials
// (reduce_max_blocks()), the arrival counter (0 between calls) and the error flag.
struct ReduceOut {
    HostResult* host;
    unsigned long long seq;
    double* partial;
    unsigned* counter;
    int* err;
};

// get_max_dt; uniform: every dxe entry is alike.
template <typename T>
hipError_t launch_max_dt(const T* Q, int64_t ndofs, int npe, int nd, int eq, double gamma,
                         double anorm, double cfl, const double* dxe, bool uniform, const ReduceOut& r, hipStream_t s);

// integrate: node i's weight is jac[i / npe] * w[i % npe].
template <typename T>
hipError_t launch_integrate(const T* Q, int64_t ndofs, int npe, const double* jac, const double* w, const ReduceOut& r,
                            hipStream_t s);

// Writes the error flag to r.host.
hipError_t launch_flag(const ReduceOut& r, hipStream_t s);

// Zhang & Shu limiter in place (limiter.hip); the quadrature weight of node i of element e
// is jac[k]*w[g - k*wnpe] with g = e*npe + i, k = g / wnpe.
template <typename T>
hipError_t launch_zhang_shu(T* Q, int64_t ndofs, int64_t ne, int npe, int nd, int wnpe,
                            const double* jac, const double* w, const double* vol, double minval,
                            double gamma, hipStream_t s);

// Monitor Σ Jω s(Q), kind 0 kinetic energy, 1 mathematical entropy (reduce.hip).
template <typename T>
hipError_t launch_monitor(const T* Q, int64_t ndofs, int npe, int nd, double gamma, int kind, const double* jac,
                          const double* w, const ReduceOut& r, hipStream_t s);

// Element-wise projection onto m^nd equispaced points (output.hip): for each of the ncols
// columns c and elements e, Qe[(c*ne + e)*m^nd + i] = ((A ⊗ .. ⊗ A) Q_e)_i with
// Q_e = Q[(c*ne + e)*n^nd + :] and A the m x n row-major interpolation matrix (device
// memory).  hipErrorInvalidValue when the generic kernel's LDS footprint exceeds 64 KB.
template <typename T>
hipError_t launch_equispaced(const T* Q, T* Qe, const double* A, int nd, int n, int m, int64_t ne, int ncols,
                             hipStream_t s);
// LDS bytes of the generic kernel and its units per block
int equispaced_lds_bytes(int nd, int n, int m, int elem_bytes, int* upb_out);

// Number of partials the reductions may write (size of the partial buffer).
int reduce_max_blocks();

}  // namespace flouhip
