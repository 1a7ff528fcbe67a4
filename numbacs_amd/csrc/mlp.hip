// BF16 MFMA kernels of the flow-map surrogate (an MLP mapping
// (x0, y0, t0, T) to the 2-D displacement): Fourier features, hidden layers
// as BF16 GEMMs with FP32 accumulation on v_mfma_f32_16x16x32_bf16 with
// fused bias/GELU epilogues, their backward GEMMs, the small output layer,
// the loss and an Adam update.  No reference counterpart: the surrogate is
// an addition on top of the reference's integrator path.
//
// GEMM tiling: a 256-thread block computes a 64x64 tile of C = A * B; each of
// its four wavefronts owns a 32x32 quarter as 2x2 MFMA 16x16 tiles.  K runs
// in turns of 128: the block stages a 64x128 slice of A and a 128x64 slice of B
// in LDS with k contiguous (chunks of 8 k permuted by row against bank
// conflicts), transposing on the way in when the operand is stored with the
// other dimension contiguous, so forward (X W), backward-data (dY W^T) and
// backward-weight (X^T dY) products all use the same kernel, and multiplies
// them in steps of 32.
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16, wave64): lane l supplies
// A[l % 16][8*(l/16) .. +7] and B[8*(l/16) .. +7][l % 16]; it receives
// D[4*(l/16) + i][l % 16], i = 0..3.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "activations.h"
#include "common.h"

namespace nbx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr int BM = 64, BN = 64, BK = 32;

// EPI_F32_ADD: split-K partial sums added into C32 (zeroed beforehand)
enum Epilogue { EPI_F32 = 0, EPI_BIAS_GELU = 1, EPI_GELU_GRAD = 2, EPI_F32_ADD = 3 };

// C(m, n) = sum_k A(m, k) B(k, n), A(m, k) = A[m*sam + k*sak],
// B(k, n) = B[k*sbk + n*sbn].  AK: sak == 1 (else sam == 1); BKC: sbk == 1
// (else sbn == 1).  M, N multiples of 64, K a multiple of 32.  Block z
// covers k in [z*ksplit, min((z+1)*ksplit, K)) (ksplit a multiple of 32;
// ksplit = K without a split).
// 64 x 64 outputs a block, 16 x 16 MFMA tiles, 2 x 2 a wavefront.  A turn loads
// up to 128 k of both operands at once (8 loads of 16 bytes a thread in flight:
// a turn costs one latency, and the latencies bound these sizes) and multiplies
// them in k-steps of 32.  8192 x 256 x 256: forward 13.4 -> 10.8 us, backward data
// 13.6 -> 10.3, backward weight 18.8 -> 11.6 (turns of 32 k before).
constexpr int kTurn = 128;

// element of the LDS tile for (row, k): rows of 16 chunks of 8 k, permuted so
// that both 16 rows of one chunk (fragments) and every eighth row's (operands
// stored along the rows) lie in different banks
__device__ __forceinline__ int tile_at(int row, int k) {
    return row * kTurn + (((k >> 3) ^ ((row ^ (row >> 3)) & 15)) << 3) + (k & 7);
}

// a turn's 64 rows x kTurn k of an operand: KC, element (row, k) at
// src[row * step + k]; else at src[row + k * step].  Slabs of 32 k from ks on
// are not read.
template <bool KC>
struct TurnLoad {
    u16x8 v[4];
    __device__ __forceinline__ void load(const uint16_t* __restrict__ src, long step, int ks) {
        const int t = threadIdx.x;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (KC) {  // 32 k a step: thread -> row t / 4, 8 k
                if (32 * q < ks)
                    v[q] = *reinterpret_cast<const u16x8*>(src + (t >> 2) * step + 32 * q +
                                                           8 * (t & 3));
            } else {  // two neighbouring k: thread -> 8 rows, k pair t / 8 (+ 32)
                const int k = 64 * (q >> 1) + 2 * (t >> 3) + (q & 1);
                if (k < ks)
                    v[q] = *reinterpret_cast<const u16x8*>(src + 8 * (t & 7) + k * step);
            }
        }
    }
    // !KC: sums[i] += the thread's rows 8 (t & 7) + i over its k
    __device__ __forceinline__ void add_columns(float (&sums)[8], int ks) const {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (64 * (q >> 1) + 2 * static_cast<int>(threadIdx.x >> 3) + (q & 1) >= ks) continue;
#pragma unroll
            for (int i = 0; i < 8; ++i) sums[i] += bf2f(v[q][i]);
        }
    }
    __device__ __forceinline__ void store(uint16_t* __restrict__ tile) const {
        const int t = threadIdx.x;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (KC) {
                *reinterpret_cast<u16x8*>(tile + tile_at(t >> 2, 32 * q + 8 * (t & 3))) = v[q];
            } else if (q & 1) {
                const int k = 64 * (q >> 1) + 2 * (t >> 3);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    *reinterpret_cast<uint32_t*>(tile + tile_at(8 * (t & 7) + i, k)) =
                        v[q - 1][i] | static_cast<uint32_t>(v[q][i]) << 16;
            }
        }
    }
};

template <bool AK, bool BKC, int EPI>
__global__ __launch_bounds__(256) void k_gemm(const uint16_t* __restrict__ A, long sam, long sak,
                                              const uint16_t* __restrict__ B, long sbk, long sbn,
                                              int M, int N, int K, float* __restrict__ C32,
                                              long ldc, uint16_t* __restrict__ C16, long ldc16,
                                              const float* __restrict__ bias,
                                              const float* __restrict__ pre, long ldp,
                                              int ksplit, float* __restrict__ colsum) {
    static_assert(BM == 64 && BN == 64 && BK == 32, "a turn's loads are laid out for these");
    __shared__ __attribute__((aligned(16))) uint16_t As[BM * kTurn];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * kTurn];
    const int t = threadIdx.x;
    const int lane = t & 63, w = t >> 6;
    const int wm = w >> 1, wn = w & 1;
    const long m0 = static_cast<long>(blockIdx.y) * BM, n0 = static_cast<long>(blockIdx.x) * BN;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the bf16 epilogues take the products transposed: a lane then holds four
    // neighbouring columns of one row
    constexpr bool kColumns = EPI == EPI_BIAS_GELU || EPI == EPI_GELU_GRAD;
    const int kb = static_cast<int>(blockIdx.z) * ksplit;
    const int ke = kb + ksplit < K ? kb + ksplit : K;
    const int r16 = lane & 15, kk = 8 * (lane >> 4);
    TurnLoad<AK> la;
    TurnLoad<BKC> lb;
    auto load = [&](int k0) {
        la.load(A + m0 * sam + k0 * sak, AK ? sam : sak, ke - k0);
        lb.load(B + n0 * sbn + k0 * sbk, BKC ? sbn : sbk, ke - k0);
    };
    load(kb);
    float slope[2][2][4];  // the epilogue's inputs, on their way meanwhile
    if constexpr (EPI == EPI_GELU_GRAD) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    slope[i][j][q] = pre[(m0 + 32 * wm + 16 * i + r16) * ldp + n0 + 32 * wn +
                                         16 * j + 4 * (lane >> 4) + q];
    }
    // column sums of B by the blocks of the first row of tiles, from the
    // registers that B passes through
    constexpr bool kSums = !AK && !BKC;
    float sums[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k0 = kb; k0 < ke; k0 += kTurn) {
        if (kSums && colsum && blockIdx.y == 0) lb.add_columns(sums, ke - k0);
        la.store(As);
        lb.store(Bs);
        __syncthreads();
        if (k0 + kTurn < ke) load(k0 + kTurn);
#pragma unroll
        for (int ks = 0; ks < kTurn; ks += BK) {
            if (k0 + ks >= ke) break;
            bf16x8 af[2], bfr[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                af[i] = *reinterpret_cast<const bf16x8*>(
                    As + tile_at(32 * wm + 16 * i + r16, ks + kk));
                bfr[i] = *reinterpret_cast<const bf16x8*>(
                    Bs + tile_at(32 * wn + 16 * i + r16, ks + kk));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = kColumns ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                               bfr[j], af[i], acc[i][j], 0, 0, 0)
                                         : __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                               af[i], bfr[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    if (kSums && colsum && blockIdx.y == 0) {
        // one addition a column and block, 64 neighbours in one instruction
        // (additions to memory from each wavefront, eight apart, took 15 us more)
        float* const part = reinterpret_cast<float*>(As);  // (read no more)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float s = sums[i];
            s += __shfl_xor(s, 8);
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (lane < 8) part[64 * w + 8 * lane + i] = s;
        }
        __syncthreads();
        if (t < 64)
            atomicAdd(&colsum[n0 + t], part[t] + part[64 + t] + part[128 + t] + part[192 + t]);
    }
    const int rq = 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (kColumns) {
                const long m = m0 + 32 * wm + 16 * i + r16, n = n0 + 32 * wn + 16 * j + rq;
                float a[4], g[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float v = acc[i][j][q];
                    if constexpr (EPI == EPI_BIAS_GELU) {
                        a[q] = v + bias[n + q];
                        bool undecided;
                        g[q] = gelu_near(a[q], undecided);
                        if (undecided) g[q] = gelu(a[q]);
                    } else {
                        g[q] = bf2f(f2bf(v)) * gelu_grad(slope[i][j][q]);
                    }
                }
                if (EPI == EPI_BIAS_GELU && C32) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) C32[m * ldc + n + q] = a[q];
                }
                const uint32_t c[2] = {pack_bf16(g[0], g[1]), pack_bf16(g[2], g[3])};
                __builtin_memcpy(C16 + m * ldc16 + n, c, 8);
            } else {
                const long n = n0 + 32 * wn + 16 * j + r16;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const long m = m0 + 32 * wm + 16 * i + rq + q;
                    if (EPI == EPI_F32_ADD) atomicAdd(&C32[m * ldc + n], acc[i][j][q]);
                    else C32[m * ldc + n] = acc[i][j][q];
                }
            }
        }
    }
}

// Fourier features: u = (inp - shift)/scale, z = 2 pi u B, h0 = [sin z, cos z].
__global__ void k_features(const float* __restrict__ inp, int64_t n, const float* __restrict__ shift,
                           const float* __restrict__ scale, const float* __restrict__ Bf, int half,
                           uint16_t* __restrict__ h0) {
    const int64_t idx = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (idx >= n * half) return;
    // (a 64-bit division takes longer than the rest)
    const int64_t r = idx >> 32 ? idx / half : static_cast<uint32_t>(idx) / static_cast<uint32_t>(half);
    const int c = static_cast<int>(idx - r * half);
    float z = 0.f;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const float u = (inp[4 * r + d] - shift[d]) / scale[d];
        z += u * Bf[d * half + c];
    }
    z *= 6.283185307179586f;
    float sn, cs;
    sincosf(z, &sn, &cs);
    h0[r * 2 * half + c] = f2bf(sn);
    h0[r * 2 * half + half + c] = f2bf(cs);
}

// y = h W_out + b_out for a 2-column output layer: one row per thread, sums in
// k order.  The rows come through LDS (64 x 256 bf16, chunks permuted by row), so
// that the loads are whole lines, and the weights are floats there: read row by
// row, 64 lines a load, 8192 x 256 took 9.8 us, now 7.7.
constexpr int kOutThreads = 64, kOutChunk = 256;

__global__ __launch_bounds__(kOutThreads) void k_out_fwd(const uint16_t* __restrict__ h, int64_t n,
                                                         int width, const uint16_t* __restrict__ W,
                                                         const float* __restrict__ b,
                                                         float* __restrict__ y) {
    __shared__ __attribute__((aligned(16))) uint16_t hs[kOutThreads * kOutChunk];
    __shared__ float wf[2 * kOutChunk];
    const int t = threadIdx.x;
    const int64_t r0 = blockIdx.x * static_cast<int64_t>(kOutThreads);
    float s0 = 0.f, s1 = 0.f;
    for (int base = 0; base < width; base += kOutChunk) {
        const int m = width - base < kOutChunk ? width - base : kOutChunk;
        __syncthreads();
        for (int i = t; i < 2 * m; i += kOutThreads) wf[i] = bf2f(W[2 * base + i]);
        const int c8 = t & 31;
        if (8 * c8 < m) {
#pragma unroll 8
            for (int row = t >> 5; row < kOutThreads; row += 2) {
                const int64_t r = r0 + row < n ? r0 + row : n - 1;
                *reinterpret_cast<u16x8*>(hs + row * kOutChunk + 8 * (c8 ^ (row & 31))) =
                    *reinterpret_cast<const u16x8*>(h + r * width + base + 8 * c8);
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int k8 = 0; k8 < m; k8 += 8) {
            const u16x8 hv = *reinterpret_cast<const u16x8*>(hs + t * kOutChunk +
                                                             8 * ((k8 >> 3) ^ (t & 31)));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float a = bf2f(hv[q]);
                s0 += a * wf[2 * (k8 + q)];
                s1 += a * wf[2 * (k8 + q) + 1];
            }
        }
    }
    const int64_t r = r0 + t;
    if (r >= n) return;
    y[2 * r] = s0 + b[0];
    y[2 * r + 1] = s1 + b[1];
}

// d = y - target; dy = d / n; loss += 0.5 * |d|^2 / n (block-reduced).
__global__ void k_loss(const float* __restrict__ y, const float* __restrict__ target, int64_t n,
                       float* __restrict__ dy, float* __restrict__ loss) {
    __shared__ float part[256];
    const int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    float l = 0.f;
    if (r < n) {
        const float d0 = y[2 * r] - target[2 * r], d1 = y[2 * r + 1] - target[2 * r + 1];
        dy[2 * r] = d0 / static_cast<float>(n);
        dy[2 * r + 1] = d1 / static_cast<float>(n);
        l = 0.5f * (d0 * d0 + d1 * d1) / static_cast<float>(n);
    }
    part[threadIdx.x] = l;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, part[0]);
}

// da = bf16(bf16(dy W_out^T) * gelu'(pre)) for the last hidden layer, kOutStep
// rows' element of one column a thread: no division by the width, the column's
// weights read once (8192 x 256: 7.6 -> 5 us).  Groups of rows beyond kOutBlocks lie
// along the grid's y: a grid extent holds fewer than 2^32 threads.
constexpr int kOutStep = 4;
constexpr int64_t kOutBlocks = 1 << 23;

__global__ __launch_bounds__(256) void k_out_bwd_data(const float* __restrict__ dy, int64_t n,
                                                      int width, const uint16_t* __restrict__ W,
                                                      const float* __restrict__ pre,
                                                      uint16_t* __restrict__ da) {
    const int64_t r0 = (static_cast<int64_t>(blockIdx.y) * kOutBlocks + blockIdx.x) * kOutStep;
    for (int k = threadIdx.x; k < width; k += blockDim.x) {
        const float w0 = bf2f(W[2 * k]), w1 = bf2f(W[2 * k + 1]);
        float p[kOutStep];
#pragma unroll
        for (int q = 0; q < kOutStep; ++q)
            p[q] = pre[(r0 + q < n ? r0 + q : n - 1) * width + k];
#pragma unroll
        for (int q = 0; q < kOutStep; ++q) {
            const int64_t r = r0 + q;
            if (r >= n) break;
            const float dh = bf2f(f2bf(dy[2 * r] * w0 + dy[2 * r + 1] * w1));
            da[r * width + k] = f2bf(dh * gelu_grad(p[q]));
        }
    }
}

// The column-sum kernels: a block takes kSumRows rows, kSumGroups groups of 256
// threads a quarter of them each (their loads in flight together), and adds one
// sum per column and block to memory -- the additions to one address queue, so
// fewer, larger blocks: 8192 x 256, 32 rows and 256 threads a block 13.5 us
// (column sums) and 21.5 us (output layer), now 4.5 and 9.7.
constexpr int kSumGroups = 4, kSumRows = 32 * kSumGroups, kSumThreads = 256 * kSumGroups;

// the groups' sums of column threadIdx.x & 255, complete in group 0's threads
__device__ __forceinline__ float group_total(float s, float (*part)[256]) {
    const int g = threadIdx.x >> 8, c = threadIdx.x & 255;
    __syncthreads();
    if (g > 0) part[g - 1][c] = s;
    __syncthreads();
    if (g == 0) {
#pragma unroll
        for (int q = 0; q < kSumGroups - 1; ++q) s += part[q][c];
    }
    return s;
}

// gW_out[k][c] += sum_r h[r][k] dy[r][c], gb_out[c] += sum_r dy[r][c]
__global__ __launch_bounds__(kSumThreads) void k_out_bwd_weight(
    const uint16_t* __restrict__ h, const float* __restrict__ dy, int64_t n, int width,
    float* __restrict__ gW, float* __restrict__ gb) {
    __shared__ float part[kSumGroups - 1][256];
    const int g = threadIdx.x >> 8, c = threadIdx.x & 255;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSumRows + 32 * g;
    const int64_t r1 = r0 + 32 < n ? r0 + 32 : n;
    for (int base = 0; base < width; base += 256) {
        const int k = base + c;
        float s0 = 0.f, s1 = 0.f;
        if (k < width) {
#pragma unroll 8
            for (int64_t r = r0; r < r1; ++r) {
                const float a = bf2f(h[r * width + k]);
                s0 += a * dy[2 * r];
                s1 += a * dy[2 * r + 1];
            }
        }
        s0 = group_total(s0, part);
        s1 = group_total(s1, part);
        if (g == 0 && k < width) {
            atomicAdd(&gW[2 * k], s0);
            atomicAdd(&gW[2 * k + 1], s1);
        }
    }
    float s = 0.f;
    if (c < 2) {
#pragma unroll 8
        for (int64_t r = r0; r < r1; ++r) s += dy[2 * r + c];
    }
    s = group_total(s, part);
    if (threadIdx.x < 2) atomicAdd(&gb[c], s);
}

// gb[c] = sum_r da[r][c] (bf16 rows)
__global__ __launch_bounds__(kSumThreads) void k_colsum(const uint16_t* __restrict__ da, int64_t n,
                                                        int width, float* __restrict__ gb) {
    __shared__ float part[kSumGroups - 1][256];
    const int g = threadIdx.x >> 8;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSumRows + 32 * g;
    const int64_t r1 = r0 + 32 < n ? r0 + 32 : n;
    for (int base = 0; base < width; base += 256) {
        const int c = base + (threadIdx.x & 255);
        float s = 0.f;
        if (c < width) {
#pragma unroll 8
            for (int64_t r = r0; r < r1; ++r) s += bf2f(da[r * width + c]);
        }
        s = group_total(s, part);
        if (g == 0 && c < width) atomicAdd(&gb[c], s);
    }
}

__global__ void k_fill_f32(float* __restrict__ p, int64_t n, float v) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill2_f32(float* __restrict__ a, int64_t na, float* __restrict__ b, int64_t nb) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < na) a[i] = 0.f;
    else if (i < na + nb) b[i - na] = 0.f;
}

// Adam with bias correction on FP32 master weights; writes the BF16 copy.
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, uint16_t* __restrict__ w16, int64_t n, float lr,
                       float b1, float b2, float eps, float c1, float c2, float wd) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float upd = (mi / c1) / (sqrtf(vi / c2) + eps) + wd * w[i];
    const float wi = w[i] - lr * upd;
    w[i] = wi;
    if (w16) w16[i] = f2bf(wi);
}

// Adam with the learning rate and both bias corrections read from device
// memory (sched = [lr, 1 - b1^t, 1 - b2^t]), so one captured training step
// can be replayed for every step of a schedule.
__global__ void k_adam_sched(float* __restrict__ w, const float* __restrict__ g,
                             float* __restrict__ m, float* __restrict__ v,
                             uint16_t* __restrict__ w16, int64_t n,
                             const float* __restrict__ sched, float b1, float b2, float eps,
                             float wd) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const float lr = sched[0], c1 = sched[1], c2 = sched[2];
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float upd = (mi / c1) / (sqrtf(vi / c2) + eps) + wd * w[i];
    const float wi = w[i] - lr * upd;
    w[i] = wi;
    if (w16) w16[i] = f2bf(wi);
}

__global__ void k_to_bf16(const float* __restrict__ x, int64_t n, uint16_t* __restrict__ y) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// ---------------------------------------------------------------------------
// Fused inference: Fourier features, the four hidden layers and the head in
// one launch.  A 256-thread block takes 64 particles; their activations stay
// in LDS (64 x 256 bf16, each layer writing over its inputs once every
// wavefront has read them), each wavefront computes a 64 x 64 quarter of a
// layer's output as 4 x 4 MFMA 16x16x32 tiles.  Four blocks share a CU: 40 KiB
// of LDS and 128 registers each.  Weights are stored transposed (k contiguous);
// a wavefront reads 16 rows' 64 bytes with neighbouring lanes on one row and
// turns them into fragments through its own 2 KiB of LDS, the next k-step's
// loads in flight meanwhile (read as fragments straight from global memory,
// neighbouring lanes on different rows, the same bytes cost four times the L1
// accesses and bound the kernel: 2.97 ms).  The products run with the weights
// as the first operand, so a lane receives four consecutive columns of one
// particle: one 8-byte store each.  Every step is the unfused path's arithmetic
// in its order: the features of k_features, per layer the same k-steps of 32
// accumulated in order then bias + GELU + bf16 (k_gemm's epilogue), the head's
// sequential fp32 sums of k_out_fwd and the output scaling -- so the result
// equals the unfused forward pass bit for bit.
//
// What bounds it is the VALU (some 70% of the issue slots, MFMA another 25%):
// 1,024 GELUs and 128 sines a particle.  Both are kept to 8 bits only, so they
// are first formed from the hardware's exp2, reciprocal, sine and cosine with a
// bound on how far these can lie from the library's float value; only where a
// rounding boundary to bf16 lies within that bound does the library function
// itself decide (gelu_near: about one activation in a thousand near zero, all
// below -4; sincos_near).  Those are listed per wavefront and evaluated 64 at a
// time.  2701 x 1001 particles: 5.38 -> 2.15 ms (231 -> 577 TFLOP/s of products;
// two 67 KB blocks a CU and the library's tanh, sin and cos throughout before).
constexpr int kInferRows = 64, kInferWidth = 256, kInferHalf = 64;
// bytes of a wavefront's own LDS: two weight fragments in the k-loop, else a
// list of undecided activations, at the end the head's weights
constexpr int kWaveBytes = 2048, kUndecided = kWaveBytes / 8;

// element of act that holds column c of a row: the 16-byte chunks of a row are
// permuted by the row's low bits, so 16 rows' chunks of one column lie in
// different banks without padding
__device__ __forceinline__ int act_at(int row, int c) {
    return row * kInferWidth + (((c >> 3) ^ (row & 15)) << 3) + (c & 7);
}

struct MlpNetDev {
    const float* shift;
    const float* scale;
    const float* Bf;
    const uint16_t* WT[4];
    const float* b[4];
    const uint16_t* Wout;
    const float* bout;
    const float* out_scale;
};

// position of the lane among those set in m
__device__ __forceinline__ int rank_in(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0));
}

__global__ __launch_bounds__(256, 4) void k_mlp_infer(MlpNetDev net, const float* __restrict__ inp,
                                                      int64_t n, float* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) uint16_t act[kInferRows * kInferWidth];
    __shared__ __attribute__((aligned(16))) uint8_t own[4][kWaveBytes];
    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kInferRows;
    uint2* const undecided = reinterpret_cast<uint2*>(own[w]);  // (argument, element of act)
    int held = 0;
    // ---- Fourier features (k_features): a particle a lane, 16 frequencies a
    // wavefront
    {
        const int64_t gr = r0 + lane < n ? r0 + lane : n - 1;
        float u[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) u[d] = (inp[4 * gr + d] - net.shift[d]) / net.scale[d];
#pragma unroll 1
        for (int i = 0; i < 16; ++i) {
            const int c = 16 * w + i;
            float z = 0.f;
#pragma unroll
            for (int d = 0; d < 4; ++d) z += u[d] * net.Bf[d * kInferHalf + c];
            bool und[2];
            const uint2 g = sincos_near(z, und[0], und[1]);
            const int at[2] = {act_at(lane, c), act_at(lane, kInferHalf + c)};
            act[at[0]] = static_cast<uint16_t>(g.x);
            act[at[1]] = static_cast<uint16_t>(g.y);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint64_t m = __ballot(und[q]);
                if (und[q])
                    undecided[held + rank_in(m)] =
                        make_uint2(__float_as_uint(z), static_cast<uint32_t>(at[q]) | q << 31);
                held += __popcll(m);
            }
            if (held <= kUndecided - 128 && i < 15) continue;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
            for (int first = lane; first < held; first += 64) {
                const uint2 e = undecided[first];
                float sn, cs;
                sincosf(__uint_as_float(e.x) * 6.283185307179586f, &sn, &cs);
                act[e.y & 0x7fffffffu] = f2bf(e.y >> 31 ? cs : sn);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            held = 0;
        }
    }
    __syncthreads();
    // ---- hidden layers
    const int r16 = lane & 15, g4 = lane >> 4;
    bf16x8* const stage = reinterpret_cast<bf16x8*>(own[w]);
    const bf16x8* const fragment =
        reinterpret_cast<const bf16x8*>(own[w]) + 4 * r16 + (g4 ^ (r16 >> 2));
#pragma unroll 1
    for (int l = 0; l < 4; ++l) {
        const int K = l == 0 ? 2 * kInferHalf : kInferWidth;
        f32x4 acc[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const uint16_t* const wt =
            net.WT[l] + (64 * w + (lane >> 2)) * K + 8 * ((lane & 3) ^ g4);
        bf16x8 raw[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) raw[j] = *reinterpret_cast<const bf16x8*>(wt + 16 * j * K);
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += 32) {
            const int next = k0 + 32 < K ? k0 + 32 : k0;
            bf16x8 bf[4];
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                stage[lane] = raw[h];
                stage[64 + lane] = raw[h + 1];
#pragma unroll
                for (int j = h; j < h + 2; ++j)
                    raw[j] = *reinterpret_cast<const bf16x8*>(wt + 16 * j * K + next);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                bf[h] = fragment[0];
                bf[h + 1] = fragment[64];
            }
            const int col = ((k0 >> 3) + g4) ^ r16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bf16x8 af = *reinterpret_cast<const bf16x8*>(
                    act + (16 * i + r16) * kInferWidth + 8 * col);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af, acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();  // every wavefront has read the layer's inputs
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            const int nc = 64 * w + 16 * j + 4 * g4;
            const int at0 = act_at(r16, nc);
            float bias[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) bias[q] = net.b[l][nc + q];
            uint64_t open[4][4];
            uint64_t any = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float g[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    bool und;
                    g[q] = gelu_near(acc[i][0][q] + bias[q], und);
                    open[i][q] = __ballot(und);
                    any |= open[i][q];
                }
                *reinterpret_cast<uint2*>(act + at0 + 16 * i * kInferWidth) =
                    make_uint2(pack_bf16(g[0], g[1]), pack_bf16(g[2], g[3]));
            }
            // list the undecided; evaluate where the list is full or complete
            while (any != 0ull || (j == 3 && held > 0)) {
                any = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint64_t m = open[i][q];
                        const int count = __popcll(m);
                        if (count == 0) continue;
                        if (held + count > kUndecided) {
                            any |= m;
                            continue;
                        }
                        if (m >> lane & 1)
                            undecided[held + rank_in(m)] =
                                make_uint2(__float_as_uint(acc[i][0][q] + bias[q]),
                                           at0 + 16 * i * kInferWidth + q);
                        held += count;
                        open[i][q] = 0;
                    }
                if (any == 0ull && j < 3) break;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
                for (int first = lane; first < held; first += 64) {
                    const uint2 e = undecided[first];
                    act[e.y] = f2bf(gelu(__uint_as_float(e.x)));
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                held = 0;
            }
            // the next column of tiles (static registers: the loop stays rolled)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[i][c] = acc[i][c + 1];
        }
        __syncthreads();
    }
    // ---- head (k_out_fwd's sequential sums) and output scaling: one wavefront,
    // a particle a lane, the 512 weights as floats over the list's memory
    static_assert(kWaveBytes >= 2 * kInferWidth * sizeof(float), "");
    if (w != (blockIdx.x & 3)) return;
    float* const wf = reinterpret_cast<float*>(own[w]);
    {
        const u16x8 h = *reinterpret_cast<const u16x8*>(net.Wout + 8 * lane);
#pragma unroll
        for (int q = 0; q < 8; ++q) wf[8 * lane + q] = bf2f(h[q]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (r0 + lane >= n) return;
    float s0 = 0.f, s1 = 0.f;
#pragma unroll 4
    for (int k8 = 0; k8 < kInferWidth; k8 += 8) {
        const u16x8 h = *reinterpret_cast<const u16x8*>(act + act_at(lane, k8));
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            s0 += bf2f(h[q]) * wf[2 * (k8 + q)];
            s1 += bf2f(h[q]) * wf[2 * (k8 + q) + 1];
        }
    }
    out[2 * (r0 + lane)] = (s0 + net.bout[0]) * net.out_scale[0];
    out[2 * (r0 + lane) + 1] = (s1 + net.bout[1]) * net.out_scale[1];
}

int check_gemm_shape(int M, int N, int K) {
    NBX_REQUIRE(M > 0 && N > 0 && K > 0, "empty GEMM");
    NBX_REQUIRE(M % BM == 0 && N % BN == 0 && K % BK == 0,
                "GEMM sizes must be multiples of 64 (M, N) and 32 (K)");
    return 0;
}

// gW = A^T @ B with A stored (K x M), B stored (K x N); with gb also B's column
// sums, which the product's blocks take on the way (8192 x 256: four launches of
// 1.8 + 11.6 + 1.3 + 4.5 us apart from it, two of 1.9 + 10.4 us with it).
void weight_grad(const uint16_t* A, const uint16_t* B, int M, int N, int K, float* gW, float* gb,
                 hipStream_t s) {
    // K is the batch: split it over blocks when the output has few tiles (a
    // 256 x 256 weight is 16 tiles on 256 CUs), each block adding its partial
    // tile into gW
    const int tiles = (M / BM) * (N / BN);
    const int64_t size = static_cast<int64_t>(M) * N;
    int splits = 256 / tiles;
    if (splits > K / 256) splits = K / 256;
    if (splits <= 1) {
        if (gb) k_fill_f32<<<blocks_for(N, 256), 256, 0, s>>>(gb, N, 0.f);
        k_gemm<false, false, EPI_F32><<<dim3(N / BN, M / BM), 256, 0, s>>>(
            A, 1, M, B, N, 1, M, N, K, gW, N, nullptr, 0, nullptr, nullptr, 0, K, gb);
        return;
    }
    const int ksplit = (K / splits + BK - 1) / BK * BK;
    const dim3 grid(N / BN, M / BM, (K + ksplit - 1) / ksplit);
    k_fill2_f32<<<blocks_for(size + N, 256), 256, 0, s>>>(gW, size, gb, gb ? N : 0);
    k_gemm<false, false, EPI_F32_ADD><<<grid, 256, 0, s>>>(A, 1, M, B, N, 1, M, N, K, gW, N,
                                                           nullptr, 0, nullptr, nullptr, 0, ksplit,
                                                           gb);
}

}  // namespace
}  // namespace nbx

using namespace nbx;

extern "C" {

int nbx_mlp_gemm(int mode, const uint16_t* A, const uint16_t* B, int M, int N, int K,
                 float* C32, uint16_t* C16, const float* bias, const float* pre,
                 nbx_stream stream) {
    if (int rc = check_gemm_shape(M, N, K)) return rc;
    NBX_REQUIRE(A != nullptr && B != nullptr, "NULL operand");
    hipStream_t s = as_stream(stream);
    const dim3 grid(N / BN, M / BM);
    switch (mode) {
        case 0:  // forward: C16 = gelu(A (MxK) @ B (KxN) + bias), C32 = pre-activation
            NBX_REQUIRE(C16 != nullptr && bias != nullptr, "forward needs C16 and bias");
            k_gemm<true, false, EPI_BIAS_GELU><<<grid, 256, 0, s>>>(A, K, 1, B, N, 1, M, N, K, C32,
                                                                    N, C16, N, bias, nullptr, 0,
                                                                    K, nullptr);
            break;
        case 1:  // backward data: C16 = bf16(bf16(A (MxK) @ B^T) * gelu'(pre)), B stored (N x K)
            NBX_REQUIRE(C16 != nullptr && pre != nullptr, "backward-data needs C16 and pre");
            k_gemm<true, true, EPI_GELU_GRAD><<<grid, 256, 0, s>>>(A, K, 1, B, 1, K, M, N, K,
                                                                   nullptr, 0, C16, N, nullptr,
                                                                   pre, N, K, nullptr);
            break;
        case 2:  // backward weight: C32 = A^T @ B with A stored (K x M), B stored (K x N)
            NBX_REQUIRE(C32 != nullptr, "backward-weight needs C32");
            weight_grad(A, B, M, N, K, C32, nullptr, s);
            break;
        case 3:  // plain: C32 = A (MxK) @ B (KxN)
            NBX_REQUIRE(C32 != nullptr, "plain GEMM needs C32");
            k_gemm<true, false, EPI_F32><<<grid, 256, 0, s>>>(A, K, 1, B, N, 1, M, N, K, C32, N,
                                                              nullptr, 0, nullptr, nullptr, 0, K,
                                                              nullptr);
            break;
        default:
            set_error("unknown GEMM mode");
            return -2;
    }
    NBX_LAUNCHED("mlp_gemm");
    return 0;
}

int nbx_mlp_weight_grad(const uint16_t* h, const uint16_t* da, int M, int N, int K, float* gW,
                        float* gb, nbx_stream stream) {
    if (int rc = check_gemm_shape(M, N, K)) return rc;
    NBX_REQUIRE(h && da && gW && gb, "NULL array");
    weight_grad(h, da, M, N, K, gW, gb, as_stream(stream));
    NBX_LAUNCHED("mlp_weight_grad");
    return 0;
}

int nbx_mlp_features(const float* inp, int64_t n, const float* shift, const float* scale,
                     const float* Bf, int half, uint16_t* h0, nbx_stream stream) {
    NBX_REQUIRE(n >= 0 && half > 0, "bad feature shape");
    if (n == 0) return 0;
    k_features<<<blocks_for(n * half, 256), 256, 0, as_stream(stream)>>>(inp, n, shift, scale, Bf,
                                                                        half, h0);
    NBX_LAUNCHED("mlp_features");
    return 0;
}

int nbx_mlp_out_forward(const uint16_t* h, int64_t n, int width, const uint16_t* W,
                        const float* b, float* y, nbx_stream stream) {
    if (n == 0) return 0;
    k_out_fwd<<<blocks_for(n, kOutThreads), kOutThreads, 0, as_stream(stream)>>>(h, n, width, W, b,
                                                                               y);
    NBX_LAUNCHED("mlp_out_fwd");
    return 0;
}

int nbx_mlp_loss(const float* y, const float* target, int64_t n, float* dy, float* loss,
                 nbx_stream stream) {
    NBX_REQUIRE(n > 0, "empty batch");
    hipStream_t s = as_stream(stream);
    k_fill_f32<<<1, 1, 0, s>>>(loss, 1, 0.f);
    k_loss<<<blocks_for(n, 256), 256, 0, s>>>(y, target, n, dy, loss);
    NBX_LAUNCHED("mlp_loss");
    return 0;
}

int nbx_mlp_out_backward(const float* dy, const uint16_t* h, const float* pre, int64_t n,
                         int width, const uint16_t* W, float* gW, float* gb, uint16_t* da,
                         nbx_stream stream) {
    NBX_REQUIRE(n > 0, "empty batch");
    hipStream_t s = as_stream(stream);
    k_fill2_f32<<<blocks_for(2 * width + 2, 256), 256, 0, s>>>(gW, 2 * width, gb, 2);
    k_out_bwd_weight<<<static_cast<unsigned>((n + kSumRows - 1) / kSumRows), kSumThreads, 0, s>>>(
        h, dy, n, width, gW, gb);
    const int64_t groups = (n + kOutStep - 1) / kOutStep;
    const dim3 grid(static_cast<unsigned>(groups < kOutBlocks ? groups : kOutBlocks),
                    static_cast<unsigned>((groups + kOutBlocks - 1) / kOutBlocks));
    k_out_bwd_data<<<grid, 256, 0, s>>>(dy, n, width, W, pre, da);
    NBX_LAUNCHED("mlp_out_bwd");
    return 0;
}

int nbx_mlp_colsum(const uint16_t* da, int64_t n, int width, float* gb, nbx_stream stream) {
    NBX_REQUIRE(n > 0, "empty batch");
    hipStream_t s = as_stream(stream);
    k_fill_f32<<<blocks_for(width, 256), 256, 0, s>>>(gb, width, 0.f);
    k_colsum<<<static_cast<unsigned>((n + kSumRows - 1) / kSumRows), kSumThreads, 0, s>>>(
        da, n, width, gb);
    NBX_LAUNCHED("mlp_colsum");
    return 0;
}

int nbx_mlp_adam(float* w, const float* g, float* m, float* v, uint16_t* w16, int64_t n, float lr,
                 float b1, float b2, float eps, int step, float weight_decay, nbx_stream stream) {
    NBX_REQUIRE(step >= 1, "Adam steps count from 1");
    if (n == 0) return 0;
    const float c1 = 1.f - powf(b1, static_cast<float>(step));
    const float c2 = 1.f - powf(b2, static_cast<float>(step));
    k_adam<<<blocks_for(n, 256), 256, 0, as_stream(stream)>>>(w, g, m, v, w16, n, lr, b1, b2, eps,
                                                              c1, c2, weight_decay);
    NBX_LAUNCHED("mlp_adam");
    return 0;
}

int nbx_mlp_adam_sched(float* w, const float* g, float* m, float* v, uint16_t* w16, int64_t n,
                       const float* sched, float b1, float b2, float eps, float weight_decay,
                       nbx_stream stream) {
    NBX_REQUIRE(sched != nullptr, "NULL schedule");
    if (n == 0) return 0;
    k_adam_sched<<<blocks_for(n, 256), 256, 0, as_stream(stream)>>>(w, g, m, v, w16, n, sched,
                                                                    b1, b2, eps, weight_decay);
    NBX_LAUNCHED("mlp_adam_sched");
    return 0;
}

int nbx_mlp_infer(const nbx_mlp_net* net, const float* inp, int64_t n, float* out,
                  nbx_stream stream) {
    NBX_REQUIRE(net != nullptr, "NULL network");
    NBX_REQUIRE(n >= 0, "negative particle count");
    NBX_REQUIRE(net->half == kInferHalf && net->width == kInferWidth && net->layers == 4,
                "the fused inference kernel runs the 128-feature, 4 x 256 network");
    if (n == 0) return 0;
    NBX_REQUIRE(inp != nullptr && out != nullptr, "NULL array");
    MlpNetDev d{net->shift, net->scale, net->Bf, {}, {}, net->Wout, net->bout, net->out_scale};
    for (int l = 0; l < 4; ++l) {
        NBX_REQUIRE(net->WT[l] != nullptr && net->b[l] != nullptr, "NULL layer");
        d.WT[l] = net->WT[l];
        d.b[l] = net->b[l];
    }
    NBX_REQUIRE(d.shift && d.scale && d.Bf && d.Wout && d.bout && d.out_scale, "NULL parameter");
    const int64_t blocks = (n + kInferRows - 1) / kInferRows;
    NBX_REQUIRE(blocks < (static_cast<int64_t>(1) << 31), "too many particles for one launch");
    k_mlp_infer<<<static_cast<unsigned>(blocks), 256, 0, as_stream(stream)>>>(d, inp, n, out);
    NBX_LAUNCHED("mlp_infer");
    return 0;
}

int nbx_mlp_to_bf16(const float* x, int64_t n, uint16_t* y, nbx_stream stream) {
    if (n == 0) return 0;
    k_to_bf16<<<blocks_for(n, 256), 256, 0, as_stream(stream)>>>(x, n, y);
    NBX_LAUNCHED("mlp_to_bf16");
    return 0;
}

}  // extern "C"
