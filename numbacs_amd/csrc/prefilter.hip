// Spline prefilter: natural cubic B-spline coefficients of (nt, nx, ny) samples.
// Per axis n samples -> n+2 coefficients c[-1..n]: (c[i-1] + 4c[i] + c[i+1])/6
// = f[i], zero second derivative at both ends, i.e. c[0] = f[0],
// c[n-1] = f[n-1], interior by the Thomas algorithm, then
// c[-1] = 2c[0]-c[1], c[n] = 2c[n-1]-c[n-2].
//
// Reference: get_interp_arrays_2D (flows.py:9-46) over interpolation.prefilter.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.h"

namespace nbx {
namespace {

// ---------------------------------------------------------------------------
// Lines in LDS.  A block takes L neighbouring lines of one axis: all its
// threads load their samples (a few loads each, in flight together), L lanes
// run the two sweeps in LDS, all threads store the coefficients.  What
// bounds the sweeps is their serial chain -- per sample one subtraction, the
// quotient's product, remainder and correction -- so a line must not wait
// for memory at each step, and short groups of lines keep many blocks in
// flight: 32 lines are 256 contiguous bytes of an x- or t-axis row.  One
// component of 96 x 271 x 101 samples: 325 -> 69 us (1.8 TB/s over the three
// passes' reads and writes), of 480 frames 1040 -> 309 us (2.0 TB/s); before,
// one thread per line swept global memory, every step's load waiting behind
// the previous step's store.
//
// The quotient by the k-th pivot p[k] = 4 - cp[k-1] uses cp[k] = 1/p[k], the
// correctly rounded reciprocal the back substitution needs anyway: product,
// exact remainder, correction (Markstein), equal to the IEEE quotient on 4e7
// sampled dividends for each of the pivots (dividends below 2^-969, whose
// remainder underflows, aside); the fix-up keeps infinities and NaN as a
// division gives them.  cp reaches its fixed point by k = 13.
constexpr int kThreads = 256;
constexpr int kPivots = 16;
struct Pivots {
    double p[kPivots], cp[kPivots];
    constexpr Pivots() : p(), cp() {
        double c = 0.0;
        for (int k = 0; k < kPivots; ++k) {
            p[k] = 4.0 - c;
            c = 1.0 / p[k];
            cp[k] = c;
        }
    }
};
__device__ constexpr Pivots kPivot;

__device__ __forceinline__ double over_pivot(double t, double p, double cp) {
    const double q = t * cp;
    return __builtin_amdgcn_div_fixup(fma(fma(-p, q, t), cp, q), p, t);
}

// One line's coefficients in place: element i (-1..n) at c[(i + 1) * st].
// (products and differences stay apart: contract(off))
__device__ __forceinline__ void solve_line(double* c, int st, int n) {
#pragma clang fp contract(off)
    auto C = [&](int i) -> double& { return c[(i + 1) * st]; };
    if (n == 1) {
        C(-1) = C(0);
        C(1) = C(0);
        return;
    }
    const double first = C(0), last = C(n - 1);
    if (n > 2) {
        const int m = n - 2;
        // forward: d[k] at C(k + 1), k = 0..m-1 (p[0] = 4 exactly)
        double d = fma(6.0, C(1), -first);
        if (m == 1) d -= last;
        d *= 0.25;
        C(1) = d;
        auto forward = [&](int k, double f, double p, double cp) {
            double t = 6.0 * f;
            if (k == m - 1) t -= last;
            d = over_pivot(t - d, p, cp);
            C(k + 1) = d;
        };
#pragma unroll
        for (int k = 1; k < kPivots; ++k)
            if (k < m) forward(k, C(k + 1), kPivot.p[k], kPivot.cp[k]);
        constexpr double p = kPivot.p[kPivots - 1], cp = kPivot.cp[kPivots - 1];
        int k = kPivots;
        for (; k + 8 <= m; k += 8) {
            double f[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) f[q] = C(k + 1 + q);
#pragma unroll
            for (int q = 0; q < 8; ++q) forward(k + q, f[q], p, cp);
        }
        for (; k < m; ++k) forward(k, C(k + 1), p, cp);
        // back substitution
        double x = d;
        for (k = m - 2; k - 7 >= kPivots - 1; k -= 8) {
            double f[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) f[q] = C(k + 1 - q);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                x = fma(-cp, x, f[q]);
                C(k + 1 - q) = x;
            }
        }
        for (; k >= kPivots; --k) {
            x = fma(-cp, x, C(k + 1));
            C(k + 1) = x;
        }
#pragma unroll
        for (int j = kPivots - 1; j >= 0; --j)
            if (j <= k) {
                x = fma(-kPivot.cp[j], x, C(j + 1));
                C(j + 1) = x;
            }
    }
    C(-1) = fma(2.0, first, -C(1));
    C(n) = fma(2.0, last, -C(n - 2));
}

// y axis: lines (a, b) of samples, contiguous, into the coefficient array's
// rows.  In LDS a line is contiguous too, its pitch odd (the sweeping lanes
// then fall in different banks).
template <int L>
__global__ __launch_bounds__(kThreads) void k_prefilter_y(const double* __restrict__ U, int nt, int nx,
                                                    int ny, double* __restrict__ C) {
    extern __shared__ double buf[];
    const int pitch = (ny + 2) | 1;
    const int64_t lines = static_cast<int64_t>(nt) * nx;
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * L;
    const int cnt = static_cast<int>(lines - l0 < L ? lines - l0 : L);
    const double* src = U + l0 * ny;
    const int lane = static_cast<int>(threadIdx.x);
    // (line, element) of this lane's element among the block's cnt * ny
    const int dq = kThreads / ny, dr = kThreads % ny;
    int q = lane / ny, r = lane % ny;
    const int total = cnt * ny;
#pragma unroll 8
    for (int e = lane; e < total; e += kThreads) {
        buf[q * pitch + r + 1] = src[e];
        q += dq;
        r += dr;
        if (r >= ny) {
            r -= ny;
            ++q;
        }
    }
    __syncthreads();
    if (lane < cnt) solve_line(buf + lane * pitch, 1, ny);
    __syncthreads();
    const int n2 = ny + 2;
    for (int l = lane >> 6; l < cnt; l += kThreads / 64) {
        const int64_t a = (l0 + l) / nx, b = (l0 + l) % nx;
        double* dst = C + ((a + 1) * (nx + 2) + (b + 1)) * n2;
        for (int c = lane & 63; c < n2; c += 64) dst[c] = buf[l * pitch + c];
    }
}

// x and t axes, in place: group g's lines start at `base + l`, l < cnt, their
// elements `st` apart (element -1 first; samples at 1..n).  axis 1: lines c
// of slice a = blockIdx.y + 1; axis 0: lines of the flattened (b, c) plane.
template <int L>
__global__ __launch_bounds__(kThreads) void k_prefilter_strided(double* __restrict__ C, int nx, int ny,
                                                          int n, int axis) {
    extern __shared__ double buf[];
    const int64_t n2 = ny + 2, n1 = (nx + 2) * n2;
    const int64_t st = axis == 1 ? n2 : n1, lines = axis == 1 ? n2 : n1;
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * L;
    const int cnt = static_cast<int>(lines - l0 < L ? lines - l0 : L);
    double* base = C + l0 + (axis == 1 ? (blockIdx.y + 1) * n1 : 0);
    const int lane = static_cast<int>(threadIdx.x), l = lane & (L - 1);
    constexpr int kRows = kThreads / L;
    if (l < cnt) {
#pragma unroll 8
        for (int i = 1 + lane / L; i <= n; i += kRows) buf[i * L + l] = base[i * st + l];
    }
    __syncthreads();
    if (lane < cnt) solve_line(buf + lane, L, n);
    __syncthreads();
    if (l < cnt) {
#pragma unroll 4
        for (int i = lane / L; i < n + 2; i += kRows) base[i * st + l] = buf[i * L + l];
    }
}

// Lines per block: 32 while their elements fit 64 KiB of LDS (axes of up to
// 253 samples; 96 x 271 x 101 samples with 16 everywhere 77 us, with 32 where
// they fit 69 us, with 64 no faster), fewer for longer axes; 0 where not even
// one does.
int lines_per_block(int n) {
    for (int L : {32, 16, 8, 4, 2, 1})
        if (static_cast<int64_t>(L) * (n + 3) * 8 <= 65536) return L;
    return 0;
}

// ---------------------------------------------------------------------------
// Lines too long for LDS or too many for one launch of groups (2^29 of up to 253
// samples): one thread per line in global memory, the samples first scattered
// into the coefficient array.

__device__ void prefilter_line(double* p, long stride, int n) {
    auto C = [&](int k) -> double& { return p[(static_cast<long>(k) + 1) * stride]; };
    if (n == 1) {
        C(-1) = C(0);
        C(1) = C(0);
        return;
    }
    if (n > 2) {
        // forward sweep; the modified super-diagonal cp[k] = 1/(4 - cp[k-1])
        // is recomputed on the way back instead of stored
        const int m = n - 2;
        double cp = 0.0, prev_d = 0.0;
        for (int k = 0; k < m; ++k) {
            const int i = k + 1;
            double rhs = 6.0 * C(i);
            if (i == 1) rhs -= C(0);
            if (i == n - 2) rhs -= C(n - 1);
            const double denom = 4.0 - (k > 0 ? cp : 0.0);
            cp = 1.0 / denom;
            const double d = (rhs - (k > 0 ? prev_d : 0.0)) / denom;
            C(i) = d;
            prev_d = d;
        }
        // back substitution needs cp[k] for k = m-2 .. 0.  The recurrence
        // cp[k] = 1/(4 - cp[k-1]) reaches its double-precision fixed point
        // (2 - sqrt(3)) by k = 13 and stays there, so 32 stored terms give
        // every cp[k] exactly.
        constexpr int kLocal = 32;
        double cps[kLocal];
        double c = 0.0;
        for (int k = 0; k < kLocal; ++k) {
            c = 1.0 / (4.0 - (k > 0 ? c : 0.0));
            cps[k] = c;
        }
        for (int k = m - 2; k >= 0; --k)
            C(k + 1) = C(k + 1) - cps[k < kLocal ? k : kLocal - 1] * C(k + 2);
    }
    C(-1) = 2 * C(0) - C(1);
    C(n) = 2 * C(n - 1) - C(n - 2);
}

__global__ void k_prefilter_scatter(const double* __restrict__ U, int nt, int nx, int ny,
                                    double* __restrict__ C) {
    const long n2 = ny + 2, n1 = static_cast<long>(nx + 2) * n2;
    const long total = static_cast<long>(nt + 2) * n1;
    for (long k = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; k < total;
         k += static_cast<long>(gridDim.x) * blockDim.x) {
        const int a = static_cast<int>(k / n1);
        const int b = static_cast<int>((k / n2) % (nx + 2));
        const int c = static_cast<int>(k % n2);
        double v = 0.0;
        if (a >= 1 && a <= nt && b >= 1 && b <= nx && c >= 1 && c <= ny)
            v = U[(static_cast<long>(a - 1) * nx + (b - 1)) * ny + (c - 1)];
        C[k] = v;
    }
}

// axis: 2 = y lines (a in 1..nt, b in 1..nx), 1 = x lines (a in 1..nt,
// c in 0..ny+1), 0 = t lines (b in 0..nx+1, c in 0..ny+1)
__global__ void k_prefilter_axis(double* __restrict__ C, int nt, int nx, int ny, int axis) {
    const long n2 = ny + 2, n1 = static_cast<long>(nx + 2) * n2;
    long lines, stride;
    int n;
    if (axis == 2) { lines = static_cast<long>(nt) * nx; stride = 1; n = ny; }
    else if (axis == 1) { lines = static_cast<long>(nt) * (ny + 2); stride = n2; n = nx; }
    else { lines = static_cast<long>(nx + 2) * (ny + 2); stride = n1; n = nt; }
    const long L = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (L >= lines) return;
    double* p;
    if (axis == 2) {
        const long a = 1 + L / nx, b = 1 + L % nx;
        p = C + a * n1 + b * n2;
    } else if (axis == 1) {
        const long a = 1 + L / (ny + 2), c = L % (ny + 2);
        p = C + a * n1 + c;
    } else {
        const long b = L / (ny + 2), c = L % (ny + 2);
        p = C + b * n2 + c;
    }
    prefilter_line(p, stride, n);
}

template <int L>
int launch_axis(const double* U, int nt, int nx, int ny, double* C, int axis, hipStream_t s) {
    if (axis == 2) {
        const int64_t lines = static_cast<int64_t>(nt) * nx;
        k_prefilter_y<L><<<static_cast<unsigned>((lines + L - 1) / L), kThreads,
                           sizeof(double) * L * ((ny + 2) | 1), s>>>(U, nt, nx, ny, C);
        NBX_LAUNCHED("prefilter_y");
        return 0;
    }
    const int n = axis == 1 ? nx : nt;
    const int64_t lines = axis == 1 ? ny + 2 : static_cast<int64_t>(nx + 2) * (ny + 2);
    const dim3 grid(static_cast<unsigned>((lines + L - 1) / L), axis == 1 ? nt : 1);
    k_prefilter_strided<L><<<grid, kThreads, sizeof(double) * L * (n + 2), s>>>(C, nx, ny, n, axis);
    NBX_LAUNCHED("prefilter_strided");
    return 0;
}

int prefilter_axis(const double* U, int nt, int nx, int ny, double* C, int axis, hipStream_t s) {
    const int n = axis == 2 ? ny : axis == 1 ? nx : nt;
    const int64_t lines = axis == 2   ? static_cast<int64_t>(nt) * nx
                          : axis == 1 ? ny + 2
                                      : static_cast<int64_t>(nx + 2) * (ny + 2);
    int L = lines_per_block(n);
    // (a launch holds fewer than 2^32 threads -- past that its last blocks do not
    // run, and no error says so -- and its grid's y extent 65535 slices)
    if (L > 0 && (lines + L - 1) / L * kThreads >= int64_t(1) << 32) L = 0;
    if (axis == 1 && nt > 65535) L = 0;
    switch (L) {
        case 32: return launch_axis<32>(U, nt, nx, ny, C, axis, s);
        case 16: return launch_axis<16>(U, nt, nx, ny, C, axis, s);
        case 8: return launch_axis<8>(U, nt, nx, ny, C, axis, s);
        case 4: return launch_axis<4>(U, nt, nx, ny, C, axis, s);
        case 2: return launch_axis<2>(U, nt, nx, ny, C, axis, s);
        case 1: return launch_axis<1>(U, nt, nx, ny, C, axis, s);
        default: break;
    }
    if (axis == 2) {
        const long total = static_cast<long>(nt + 2) * (nx + 2) * (ny + 2);
        k_prefilter_scatter<<<std::min(blocks_for(total, 256), 8192u), 256, 0, s>>>(U, nt, nx, ny,
                                                                                    C);
        NBX_LAUNCHED("prefilter_scatter");
    }
    k_prefilter_axis<<<blocks_for(axis == 1 ? nt * lines : lines, 128), 128, 0, s>>>(C, nt, nx, ny,
                                                                                     axis);
    NBX_LAUNCHED("prefilter_axis");
    return 0;
}

}  // namespace
}  // namespace nbx

using namespace nbx;

extern "C" int nbx_prefilter3(const double* U, int nt, int nx, int ny, double* C,
                              nbx_stream stream) {
    NBX_REQUIRE(U != nullptr && C != nullptr, "NULL argument");
    NBX_REQUIRE(nt >= 1 && nx >= 1 && ny >= 1, "empty grid");
    hipStream_t s = as_stream(stream);
    // every coefficient is written: the y pass fills the sampled rows, the x
    // pass adds their border rows, the t pass the border slices
    for (int axis : {2, 1, 0})
        if (const int rc = prefilter_axis(U, nt, nx, ny, C, axis, s)) return rc;
    return 0;
}
