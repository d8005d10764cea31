// Numerical fluxes on the faces of axis-aligned affine elements (Flou's CartesianMesh), GLL
// nodes, StdAverage or LxF(StdAverage) surface flux.
//
// The face frame is n = ±e_d, t = ±e_{d+1}, b = ±e_{d+2}, so a trace is read in the order
// (ρ, normal and transverse momenta, E) by index, and only the normal's sign is applied:
// signs of the transverse axes commute with every rounding of these fluxes.
#pragma once

#include "common.hpp"
#include "physics_plain.hpp"

namespace flouhip {

// Physical variable of the c-th face-frame momentum of a face of direction dir.
template <int ND>
__device__ __forceinline__ int face_mom(int dir, int c) {
    return 1 + (dir + c) % ND;
}

// Place in that order of the physical momentum v (1..ND).
template <int ND>
__device__ __forceinline__ int face_frame(int dir, int v) {
    return 1 + (v - 1 + ND - dir) % ND;
}

// A neighbour's trace, in the order above: node n of its element nbe.
template <typename T, int ND, int NV>
__device__ __forceinline__ void load_trace(const T* Qn, int64_t Nd, int dir, T* ext) {
    ext[0] = Qn[0];
    if constexpr (NV > 1) {
#pragma unroll
        for (int c = 0; c < ND; ++c) ext[1 + c] = Qn[face_mom<ND>(dir, c) * Nd];
        ext[NV - 1] = Qn[(NV - 1) * Nd];
    }
}

// The exterior state of face node f of boundary face `slot` (applyBCs!); own: the trace there.
template <typename T, int ND, int NPF, int NV>
__device__ __forceinline__ void boundary_trace(const RhsArgs<T>& a, int info, int slot, int f, int dir, const T* own,
                                               T* ext) {
    const int bd = finfo_bd(info);
    const int type = a.bctype[bd];
    if (type == BC_DIRICHLET || type == BC_INFLOW) {
        const T* src = type == BC_DIRICHLET ? a.bcstate + ((int64_t)a.fid[slot] * NPF + f) * NV : a.bcconst + bd * NV;
        load_trace<T, ND, NV>(src, 1, dir, ext);
    } else {
#pragma unroll
        for (int v = 0; v < NV; ++v) ext[v] = own[v];
        if (NV > 1 && type == BC_SLIP) ext[1] = -ext[1];
    }
}

// The flux through the face times its surface Jacobian, outward from the master for the
// master and with the opposite sign for the slave, in the order above; own and ext are changed.
// sn: the sign of the master's normal along e_dir.
template <typename T, int ND>
__device__ __forceinline__ void axis_flux(T* own, T* ext, T sn, T jac, bool slave, int sdiss, T gamma, T intensity,
                                          int* err, T* Fn) {
    constexpr int NV = ND + 2;
    // The master's and the slave's terms commute in every sum but the momentum's, and the jump
    // only changes sign.
    own[1] = sn * own[1];
    ext[1] = sn * ext[1];
    const T sg = slave ? T(-1) : T(1);
    const Recip<T> iro(own[0]), irx(ext[0]);
    const T po = plain::pressure<T, ND>(own, gamma, iro), px = plain::pressure<T, ND>(ext, gamma, irx);
    const T uo = iro.div(own[1]), ux = irx.div(ext[1]);
    const T mo = own[1] * uo, mx = ext[1] * ux;
    Fn[0] = (own[1] + ext[1]) / T(2);
    Fn[1] = ((((slave ? mx : mo) + (slave ? px : po)) + (slave ? mo : mx)) + (slave ? po : px)) / T(2);
#pragma unroll
    for (int c = 1; c < ND; ++c) Fn[1 + c] = (own[1 + c] * uo + ext[1 + c] * ux) / T(2);
    Fn[NV - 1] = ((own[NV - 1] + po) * uo + (ext[NV - 1] + px) * ux) / T(2);
    if (sdiss == DISS_LXF) {
        const T lo = fabs(uo) + plain::dsqrt(iro.div(gamma * po), err);
        const T lx = fabs(ux) + plain::dsqrt(irx.div(gamma * px), err);
        // the larger speed, the master's where they do not compare
        const T lam = sg * (slave ? ((lx < lo) ? lo : lx) : ((lo < lx) ? lx : lo));
#pragma unroll
        for (int v = 0; v < NV; ++v) Fn[v] = Fn[v] + ((lam * (own[v] - ext[v])) / T(2)) * intensity;
    }
    Fn[1] = sn * Fn[1];
    const T js = sg * jac;
#pragma unroll
    for (int v = 0; v < NV; ++v) Fn[v] = Fn[v] * js;
}

}  // namespace flouhip
