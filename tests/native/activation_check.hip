// The surrogate's short activation forms against the library's functions, over
// every float (see test_gpu_activations.py).
#include "../../numbacs_amd/csrc/activations.h"

namespace nbx {
namespace {

__device__ __forceinline__ bool same_bf16(uint16_t a, uint16_t b) {
    const bool nan_a = (a & 0x7fffu) > 0x7f80u, nan_b = (b & 0x7fffu) > 0x7f80u;
    return a == b || (nan_a && nan_b);
}

// counts = (decided values that round otherwise than the library's, undecided
// values) of: 0 GELU, 1 sine, 2 cosine.  2^24 threads, 256 floats each.
__global__ __launch_bounds__(256) void k_check(int which, unsigned long long* counts) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    unsigned long long wrong = 0, open = 0;
    for (uint32_t k = 0; k < 256; ++k) {
        const float a = __uint_as_float(k << 24 | t);
        bool und[2];
        uint16_t got, want;
        if (which == 0) {
            const float g = gelu_near(a, und[0]);
            got = static_cast<uint16_t>(pack_bf16(g, 0.0f));
            want = f2bf(gelu(a));
        } else {
            const uint2 b = sincos_near(a, und[0], und[1]);
            float sn, cs;
            sincosf(a * 6.283185307179586f, &sn, &cs);
            got = static_cast<uint16_t>(which == 1 ? b.x : b.y);
            want = f2bf(which == 1 ? sn : cs);
            und[0] = which == 1 ? und[0] : und[1];
        }
        open += und[0];
        wrong += !und[0] && !same_bf16(got, want);
    }
    if (wrong) atomicAdd(&counts[0], wrong);
    if (open) atomicAdd(&counts[1], open);
}

__global__ __launch_bounds__(256) void k_gelu(const float* __restrict__ a, int64_t n,
                                              uint16_t* __restrict__ out) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(256) + threadIdx.x;
    if (i < n) out[i] = f2bf(gelu(a[i]));
}

}  // namespace
}  // namespace nbx

extern "C" {

// counts: two zeroed 64-bit words on the device
int activation_check(int which, unsigned long long* counts, void* stream) {
    nbx::k_check<<<1 << 16, 256, 0, static_cast<hipStream_t>(stream)>>>(which, counts);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// out[i] = bf16 of the library form's gelu(a[i])
int activation_gelu(const float* a, int64_t n, uint16_t* out, void* stream) {
    nbx::k_gelu<<<static_cast<unsigned>((n + 255) / 256), 256, 0,
                  static_cast<hipStream_t>(stream)>>>(a, n, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // extern "C"
