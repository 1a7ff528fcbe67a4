// Lane-level helpers of the flow-map kernels: data exchange between the lanes of
// a 2- or 4-lane particle group by DPP quad permutations, and divisions that
// share a reciprocal.
#pragma once

#include <hip/hip_runtime.h>

namespace nbx {

// Permutations: the value of a pair's even lane, of its odd lane, of the
// other lane of the pair, and of the lane two further in the quad.
constexpr int kPairEven = 0xA0, kPairOdd = 0xF5, kPairSwap = 0xB1, kQuadCross = 0x4E;

template <int Ctrl>
__device__ __forceinline__ int quad_move(int v) {
    return __builtin_amdgcn_mov_dpp(v, Ctrl, 0xF, 0xF, false);
}
template <int Ctrl>
__device__ __forceinline__ float quad_move(float v) {
    return __int_as_float(quad_move<Ctrl>(__float_as_int(v)));
}
template <int Ctrl>
__device__ __forceinline__ double quad_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = quad_move<Ctrl>(static_cast<int>(b & 0xffffffffll));
    const int hi = quad_move<Ctrl>(static_cast<int>(b >> 32));
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// Correctly rounded quotients by one divisor: its reciprocal by the steps of
// the hardware's division sequence, shared (and formed ahead of the
// numerators), then per quotient the product, one remainder and the fix-up of
// special operands.  Equal to num / den wherever den, its reciprocal and the
// quotient are normal numbers and |num| is at least 2^-969: the remainder is
// then exact (nearer the smallest numbers it underflows: 6% of quotients of
// numerators near 2^-1020 are off by a unit in the last place).
__device__ __forceinline__ double div_recip(double den) {
    double r = __builtin_amdgcn_rcp(den);
    r = fma(r, fma(-den, r, 1.0), r);
    return fma(r, fma(-den, r, 1.0), r);
}
__device__ __forceinline__ double div_with(double num, double den, double recip) {
    const double q = num * recip;
    return __builtin_amdgcn_div_fixup(fma(fma(-den, q, num), recip, q), den, num);
}

}  // namespace nbx
