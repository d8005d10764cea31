// Pieces shared by the plain-arithmetic element kernels: the pairs of a line and the RK
// stage epilogue.
#pragma once

#include "common.hpp"
#include "exact_div.hpp"

namespace flouhip {

// Line position a (bits 3..5) and b (bits 0..2) of pair `pr`, pairs (a < b) in row order,
// ten to a 64-bit word.
template <int N>
struct PairTab {
    unsigned long long w[3] = {0, 0, 0};
    constexpr PairTab() {
        int k = 0;
        for (int a = 0; a < N; ++a)
            for (int b = a + 1; b < N; ++b, ++k) w[k / 10] |= (unsigned long long)(a * 8 + b) << (6 * (k % 10));
    }
};
template <int N>
__device__ __forceinline__ int pair_ab(int pr) {
    constexpr PairTab<N> T;
    if (N * (N - 1) / 2 <= 10) return (int)(T.w[0] >> (6 * pr)) & 63;
    const unsigned long long w = pr < 10 ? T.w[0] : (pr < 20 ? T.w[1] : T.w[2]);
    return (int)(w >> (6 * (pr < 10 ? pr : (pr < 20 ? pr - 10 : pr - 20)))) & 63;
}

// The stage epilogue's second operand: the RK register or the SSP base state, null if the
// stage has none.
template <typename T>
__device__ __forceinline__ const T* stage_aux(const RhsArgs<T>& a) {
    return (a.mode == MODE_2N && !a.first) ? a.reg
         : ((a.mode == MODE_SSP2 || a.mode == MODE_SSP3) ? a.ubase : nullptr);
}

// Writes entry idx of the stage's result from L(u_in) (kv), the stage input and the second
// operand there.
template <typename T>
struct StageOut {
    const RhsArgs<T>& a;
    Recip<T> i3;
    __device__ explicit StageOut(const RhsArgs<T>& a_) : a(a_), i3(T(3)) {}
    __device__ __forceinline__ void put(int64_t idx, T kv, T uin, T aux) const {
        switch (a.mode) {
            case MODE_RHS:
                a.out[idx] = kv;
                break;
            case MODE_2N: {
                const T t = a.first ? a.dt * kv : a.A * aux + a.dt * kv;
                a.reg[idx] = t;
                a.out[idx] = uin + a.B * t;
                break;
            }
            case MODE_SSP1:
                a.out[idx] = uin + a.dt * kv;
                break;
            case MODE_SSP2:
                a.out[idx] = ((T(3) * aux + uin) + a.dt * kv) / T(4);
                break;
            default:
                a.out[idx] = i3.div((aux + T(2) * uin) + (T(2) * a.dt) * kv);
                break;
        }
    }
};

}  // namespace flouhip
