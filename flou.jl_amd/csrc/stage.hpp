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

// Threads of a block of n nodes: whole waves, and eight waves for five to seven.  Only one block
// of six waves ran on a CU where two of eight do (FP64 3-D N=6: 343 nodes, 69 to 80 KB of LDS, 100 to
// 131 registers; 5.9 waves per CU; CK2N54 step of 16.7 M nodes 14.5 -> 8.7 ms).
constexpr int block_threads(int n) {
    return n > 256 && n <= 512 ? 512 : (n + 63) / 64 * 64;
}

// Node arrays of a block in LDS: with PAD one value after every row of N nodes, so that lanes on
// consecutive x-lines, N values apart, read distinct banks for even N too.
template <int ND, int N, bool PAD>
struct NodeLds {
    static constexpr int RS = PAD ? N + 1 : N;               // row stride
    static constexpr int ES = Cfg<ND, N>::NPE / N * RS;      // element stride
    __device__ __forceinline__ static int node(int j) { return PAD ? j + j / N : j; }  // block node j
    // first node of line f of direction DIR in an element, and the step along the line
    template <int DIR>
    __device__ __forceinline__ static int line(int f) {
        if (ND == 1) return 0;
        if (DIR == 0) return RS * f;
        if (ND == 2) return f;
        return f % N + RS * (DIR == 1 ? N : 1) * (f / N);
    }
    template <int DIR>
    static constexpr int step() {
        return DIR == 0 ? 1 : (DIR == 1 ? RS : RS * N);
    }
};

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
