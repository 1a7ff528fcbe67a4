// The surrogate's activations: bf16 conversions, GELU and its slope by the
// library's tanh, and short forms of GELU, sine and cosine that say where their
// rounding to bf16 is not decided.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace nbx {
namespace {

// bf16 as raw 16-bit patterns in memory; round to nearest even.
__device__ __forceinline__ uint16_t f2bf(float f) {
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
    const uint32_t lsb = (u >> 16) & 1u;
    return static_cast<uint16_t>((u + 0x7fffu + lsb) >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t h) {
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

constexpr float kGeluC = 0.7978845608028654f;  // sqrt(2/pi)
constexpr float kGeluA = 0.044715f;

__device__ __forceinline__ float gelu(float a) {
    const float t = tanhf(kGeluC * (a + kGeluA * a * a * a));
    return 0.5f * a * (1.0f + t);
}

__device__ __forceinline__ float gelu_grad(float a) {
    const float inner = kGeluC * (a + kGeluA * a * a * a);
    const float t = tanhf(inner);
    const float dinner = kGeluC * (1.0f + 3.0f * kGeluA * a * a);
    return 0.5f * (1.0f + t) + 0.5f * a * (1.0f - t * t) * dinner;
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// two floats to bf16 (round to nearest even), as f2bf rounds each
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const bf16x2 v = __builtin_convertvector((f32x2{a, b}), bf16x2);
    uint32_t r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}

// gelu(a) = a / (1 + exp(-2 inner)) by the hardware's exp2 and reciprocal.
// It differs from gelu(a) by less than (d + 6) units in its last float place,
// d = 1 + exp(-2 inner) (the library form's own rounding grows with d: 1 + tanh
// cancels), so undecided is set where a bf16 rounding boundary (low half
// 0x8000) is that near.  Checked for every float (tests/native): where undecided
// is not set, both round to the same bf16.
__device__ __forceinline__ float gelu_near(float a, bool& undecided) {
    constexpr float c0 = -2.0f * 1.4426950408889634f * kGeluC, c1 = c0 * kGeluA;
    const float d = 1.0f + __builtin_amdgcn_exp2f(a * fmaf(c1, a * a, c0));
    const float g = a * __builtin_amdgcn_rcpf(d);
    // the low half as a signed number lies at +-0x8000 on a boundary
    const float low = static_cast<float>(static_cast<int16_t>(__float_as_uint(g)));
    undecided = fabsf(low) + d >= 32768.0f - 6.0f;
    return g;
}

// sine (x) and cosine (y) of 2 pi s to bf16 by the hardware's functions of a
// revolution: both lie within delta of sinf / cosf of the rounded product, which
// k_features takes (7e-7 |s| is that product's rounding, 5e-7 the hardware's
// own error; largest seen over every float: 0.78 delta), so undecided is set
// where the two ends of that interval round differently.
__device__ __forceinline__ uint2 sincos_near(float s, bool& und_s, bool& und_c) {
    const float f = __builtin_amdgcn_fractf(s), delta = fmaf(fabsf(s), 7e-7f, 5e-7f);
    const float sn = __builtin_amdgcn_sinf(f), cs = __builtin_amdgcn_cosf(f);
    const uint2 b = make_uint2(pack_bf16(sn - delta, sn + delta), pack_bf16(cs - delta, cs + delta));
    const bool wide = !(fabsf(s) < 1e4f);
    und_s = (b.x >> 16) != (b.x & 0xffffu) || wide;
    und_c = (b.y >> 16) != (b.y & 0xffffu) || wide;
    return b;
}

}  // namespace
}  // namespace nbx
