// FTLE ridge extraction: percentile threshold, ridge predicate, stream
// compaction, 8-connected labelling and grouping into ridges.
//
// Reference: ftle_ridge_pts (extraction/ridges.py:9-76), _ftle_ridges
// (ridges.py:79-154) and ftle_ridges (ridges.py:186-229), which use
// np.percentile (linear method) and scipy.ndimage.label with a full 3x3
// structure.
//
// Device pipeline (with a percentile threshold no host round trip before the
// end, the grouping stage being sized by a bound on the ridge-point count;
// without one the count is read back to size it):
//   percentile  : two radix selects (6 passes of 11 or 10 bits over
//                 order-preserving 64-bit keys, each pass's blocks first
//                 picking the previous pass's digit) for the order statistics
//                 around the virtual index, then numpy's two-sided lerp --
//                 f_min stays in HBM;
//   predicate   : one thread per grid point, the reference's central
//                 differences and Steger sub-pixel test;
//   labelling   : union-find (the larger root linked under the smaller), in LDS
//                 within 16 x 64 tiles by the predicate's blocks, then
//                 lock-free (atomicMin) across the tiles' borders, then path
//                 flattening; every root is its component's smallest raveled
//                 index, so ordering components by root is
//                 scipy.ndimage.label's raster order of first pixels;
//   compaction  : counts of ridge points and roots a 1024-point tile, their
//                 scan, then the points in raveled (i*ny+j) order and the
//                 roots' ranks;
//   grouping    : stable radix sort of the points by component, segment
//                 starts, min_ridge_pts filter and a scatter.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "common.h"
#include "ordered_ridges.h"

// Scratch of nbx_ridges_noalloc: a fixed 64 MiB device array in place of the
// allocated workspace, for callers that cannot allocate.  The host never
// uses the array's name as an address: each device's copy lives at its own
// address, which hipGetSymbolAddress returns (once per device, with that
// device current, in scratch_address below) and which is then passed to the
// kernels.
static __device__ __align__(256) char scratch[static_cast<size_t>(64) << 20];

namespace nbx {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;  // 1024 flags per block

// Radix-select state.  The digit picked from pass p's histograms is
// computed by every block of pass p+1 (and by the finishing kernel after the
// last pass) instead of by a launch of its own, so the histograms rotate
// over three buffers (pass p adds into hist[p % 3], reads hist[(p-1) % 3]
// and clears hist[(p+1) % 3], which no block of p reads or writes) and the
// digit state over two (pass p's blocks read the state of pass p-1's
// search, block 0 stores the updated one for pass p+1).  While both searches
// share a prefix only search 0's histogram is filled, for both.
constexpr int kSelThreads = 1024, kSelPasses = 6, kSelBins = 2048;
constexpr int kSelOwn = kSelBins / kSelThreads;  // bins a thread
// keys kept once their first 22 bits are known (all later passes read these)
constexpr int64_t kSelHeld = 65536;
constexpr unsigned kSelStage = 1024;  // of them a block collects before one append

struct SelState {
    unsigned long long prefix[2][2];  // [pass & 1][search]
    unsigned long long mask[2][2];
    long long k[2][2];
    unsigned int hist[3][2][kSelBins];  // [pass % 3][search][bin]
    unsigned int nan_count;
    unsigned int held;  // keys offered to the list; past its room it is not used
    double result;
};

// digits of 11, 11, 11, 11, 10 and 10 bits from the top
__host__ __device__ constexpr int sel_shift(int pass) {
    return pass < 4 ? 53 - 11 * pass : 10 * (kSelPasses - 1 - pass);
}
__host__ __device__ constexpr unsigned sel_digit(int pass) { return pass < 4 ? 2047u : 1023u; }

__device__ __forceinline__ unsigned long long order_key(double v) {
    const unsigned long long b = __double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double key_value(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double(static_cast<long long>(b));
}

__global__ void k_sel_init(SelState* st, long long k_lo, long long k_hi) {
    const int t = threadIdx.x;
    for (int b = t; b < kSelBins; b += blockDim.x) st->hist[0][0][b] = st->hist[0][1][b] = 0;
    if (t == 0) {
        st->prefix[0][0] = st->prefix[0][1] = 0;
        st->mask[0][0] = st->mask[0][1] = 0;
        st->k[0][0] = k_lo;
        st->k[0][1] = k_hi;
        st->nan_count = 0;
        st->held = 0;
        st->result = 0.0;
    }
}

// Digit state of both searches after pass `prev`, into LDS: the bin whose
// cumulative count first exceeds k.  Called by all kSelThreads threads,
// kSelOwn neighbouring bins each; ends with a barrier.  Sum holds the number of
// keys: 32 bits below 2^32 of them, as every grid has (64 bits throughout: FTLE
// and ridges of 8 M values 333 -> 337 us).
template <class Sum>
__device__ void sel_advance(const SelState* st, int prev, unsigned long long* sp,
                            unsigned long long* sm, long long* sk) {
    __shared__ Sum waves[2][kSelThreads / 64];
    const int t = threadIdx.x, lane = t & 63;
    const int sb = prev & 1, hb = prev % 3;
    const int same = st->prefix[sb][0] == st->prefix[sb][1];
    unsigned int c[2][kSelOwn];
    Sum before[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        Sum x = 0;
#pragma unroll
        for (int q = 0; q < kSelOwn; ++q) {
            c[s][q] = st->hist[hb][same ? 0 : s][kSelOwn * t + q];
            x += c[s][q];
        }
        before[s] = x;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const Sum y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        before[s] = x - before[s];
        if (lane == 63) waves[s][t >> 6] = x;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        for (int w = 0; w < (t >> 6); ++w) before[s] += waves[s][w];
        const long long k = st->k[sb][s];
        long long at = static_cast<long long>(before[s]);
#pragma unroll
        for (int q = 0; q < kSelOwn; ++q) {
            // exactly one bin has at <= k < at + count (k < total always holds)
            if (at <= k && k < at + c[s][q]) {
                sk[s] = k - at;
                sp[s] = st->prefix[sb][s] |
                        static_cast<unsigned long long>(kSelOwn * t + q) << sel_shift(prev);
                sm[s] = st->mask[sb][s] |
                        static_cast<unsigned long long>(sel_digit(prev)) << sel_shift(prev);
            }
            at += c[s][q];
        }
    }
    __syncthreads();
}

// h[bin] += 1 for the lanes with `on`, the first lane's bin in one step: the
// leading digits of a smooth field agree over most of a wavefront, and 64
// atomics on one LDS word take 64 turns.
__device__ __forceinline__ void sel_count(unsigned int* h, unsigned int bin, bool on) {
    const uint64_t m = __ballot(on);
    if (m == 0) return;
    const int first = __builtin_ctzll(m);
    const unsigned int b0 = __builtin_amdgcn_readlane(bin, first);
    const uint64_t same = __ballot(on && bin == b0);
    if (static_cast<int>(threadIdx.x & 63) == first)
        atomicAdd(&h[b0], static_cast<unsigned int>(__popcll(same)));
    else if (on && bin != b0)
        atomicAdd(&h[bin], 1u);
}

// Pass `pass` of both searches.  Passes 0 to 2 read the array; pass 2 also
// lists the keys that match either prefix (22 bits: some thousands of 8 M
// values of an FTLE field), and the later passes read that list.  Where it
// overflows (many values equal in 22 bits) they read the array again.
// Bound by the reads (13 us of the 17 to 21 a pass over 8 M values takes; then
// 5.5 us a pass over the list): the whole percentile 156 -> 84 us, with digits of
// 8 bits and every pass over the array before.
template <class Sum>
__global__ __launch_bounds__(kSelThreads) void k_sel_hist(const double* __restrict__ f, int64_t n,
                                                          SelState* st, int pass,
                                                          unsigned long long* held,
                                                          int64_t room) {
    __shared__ unsigned int h[2][kSelBins];
    __shared__ unsigned long long sp[2], sm[2];
    __shared__ long long sk[2];
    __shared__ unsigned long long own[kSelStage];
    __shared__ unsigned int staged, fits, out;
    const int t = threadIdx.x;
    const int shift = sel_shift(pass);
    if (t == 0) {
        staged = 0;
        fits = kSelStage;
    }
    for (int b = t; b < 2 * kSelBins; b += kSelThreads) h[0][b] = 0;
    if (pass == 0) {
        if (t < 2) {
            sp[t] = st->prefix[0][t];
            sm[t] = st->mask[0][t];
            sk[t] = st->k[0][t];
        }
        __syncthreads();
    } else {
        sel_advance<Sum>(st, pass - 1, sp, sm, sk);
    }
    if (blockIdx.x == 0) {
        if (pass > 0 && t < 2) {
            st->prefix[pass & 1][t] = sp[t];
            st->mask[pass & 1][t] = sm[t];
            st->k[pass & 1][t] = sk[t];
        }
        unsigned int* next = st->hist[(pass + 1) % 3][0];
        for (int b = t; b < 2 * kSelBins; b += kSelThreads) next[b] = 0;
    }
    const unsigned long long p0 = sp[0], p1 = sp[1], mask = sm[0];  // one mask: equal digits
    const bool one = p0 == p1;
    const bool listed = pass > 2 && st->held <= room;
    const int64_t count = listed ? st->held : n;
    const unsigned long long* from =
        listed ? held : reinterpret_cast<const unsigned long long*>(f);
    bool room_left = pass == 2;
    unsigned int nans = 0;
    for (int64_t base = blockIdx.x * static_cast<int64_t>(4 * kSelThreads); base < count;
         base += static_cast<int64_t>(gridDim.x) * (4 * kSelThreads)) {
        unsigned long long key[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t k = base + q * kSelThreads + t;
            key[q] = from[k < count ? k : count - 1];
        }
        if (!listed) {
#pragma unroll
            for (int q = 0; q < 4; ++q) key[q] = order_key(__longlong_as_double(key[q]));
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool in = base + q * kSelThreads + t < count;
            const double v = key_value(key[q]);
            if (pass == 0 && in && v != v) ++nans;
            const unsigned int bin =
                static_cast<unsigned int>(key[q] >> shift) & sel_digit(pass);
            const bool on0 = in && (key[q] & mask) == p0;
            const bool on1 = in && !one && (key[q] & mask) == p1;
            sel_count(h[0], bin, on0);
            if (!one) sel_count(h[1], bin, on1);
            if (!room_left) continue;
            const uint64_t m = __ballot(on0 || on1);
            if (m == 0) continue;
            const int lane = t & 63, first = __builtin_ctzll(m);
            const unsigned int c = __popcll(m), rank = __popcll(m & ((1ull << lane) - 1));
            unsigned int at = 0;
            if (lane == first) at = atomicAdd(&staged, c);
            at = __builtin_amdgcn_readlane(at, first);
            if (at + c <= kSelStage) {
                if (on0 || on1) own[at + rank] = key[q];
                continue;
            }
            // the block's own list is full (and stays so: staged only grows, and
            // what fitted ends where the first that did not began): straight to
            // memory
            if (lane == first) {
                atomicMin(&fits, at);
                at = atomicAdd(&st->held, c);
            }
            at = __builtin_amdgcn_readlane(at, first);
            room_left = at + c <= room;
            if (room_left && (on0 || on1)) held[at + rank] = key[q];
        }
    }
    __syncthreads();
    const unsigned int list = staged < fits ? staged : fits;
    if (list) {  // pass 2 only
        if (t == 0) out = atomicAdd(&st->held, list);
        __syncthreads();
        for (unsigned int b = t; b < list; b += kSelThreads)
            if (out + b < room) held[out + b] = own[b];
    }
    unsigned int* gh = st->hist[pass % 3][0];
    for (int b = t; b < 2 * kSelBins; b += kSelThreads)
        if (h[0][b]) atomicAdd(&gh[b], h[0][b]);
    if (nans) atomicAdd(&st->nan_count, nans);
}

// The last digit, then numpy's _lerp: a + (b-a)*g, or b - (b-a)*(1-g) when
// g >= 0.5.
template <class Sum>
__global__ __launch_bounds__(kSelThreads) void k_sel_finish(SelState* st, double gamma,
                                                            double* out) {
    __shared__ unsigned long long sp[2], sm[2];
    __shared__ long long sk[2];
    sel_advance<Sum>(st, kSelPasses - 1, sp, sm, sk);
    if (threadIdx.x != 0) return;
    const double a = key_value(sp[0]);
    const double b = key_value(sp[1]);
    const double diff = b - a;
    double r = gamma >= 0.5 ? b - diff * (1 - gamma) : a + diff * gamma;
    if (st->nan_count) r = __longlong_as_double(0x7ff8000000000000ll);
    st->result = r;
    if (out) *out = r;
}

// held: room for min(n, kSelHeld) keys
int percentile_device(const double* f, int64_t n, double q, SelState* st,
                      unsigned long long* held, double* out, hipStream_t s) {
    NBX_REQUIRE(n >= 1, "percentile of an empty array");
    NBX_REQUIRE(q >= 0 && q <= 100, "percentile must be in [0, 100]");
    // numpy 'linear': virtual index (n-1) * (q/100); neighbours clamped to the
    // last element at or above n-1
    const double vi = static_cast<double>(n - 1) * (q / 100.0);
    const double lo = floor(vi);
    long long klo = static_cast<long long>(lo);
    long long khi = klo + 1;
    if (vi >= static_cast<double>(n - 1)) klo = khi = n - 1;
    if (khi > n - 1) khi = n - 1;
    const double gamma = vi - lo;
    k_sel_init<<<1, 256, 0, s>>>(st, klo, khi);
    NBX_LAUNCHED("sel_init");
    // one turn of 4 keys a thread, at most a block a CU: every block adds its
    // nonzero bins to the same global counters (8 M values: 75 us for the passes;
    // 512 blocks 77, of half the threads 83)
    const bool narrow = n < int64_t(1) << 32;
    auto* hist = narrow ? &k_sel_hist<unsigned int> : &k_sel_hist<unsigned long long>;
    auto* finish = narrow ? &k_sel_finish<unsigned int> : &k_sel_finish<unsigned long long>;
    unsigned nb = blocks_for(n, kSelThreads * 4);
    if (nb > 256) nb = 256;
    for (int pass = 0; pass < kSelPasses; ++pass) {
        hist<<<nb, kSelThreads, 0, s>>>(f, n, st, pass, held, n < kSelHeld ? n : kSelHeld);
        NBX_LAUNCHED("sel_hist");
    }
    finish<<<1, kSelThreads, 0, s>>>(st, gamma, out);
    NBX_LAUNCHED("sel_finish");
    return 0;
}

// ---------------------------------------------------------------------------
// Ridge predicate (ridges.py:52-74) at grid point (i, j): whether the test
// passes, then pts[k] = the sub-pixel ridge point and sdd = the second
// derivative.
__device__ __forceinline__ bool ridge_test(const double* __restrict__ f,
                                           const double2* __restrict__ evec,
                                           const double* __restrict__ xs,
                                           const double* __restrict__ ys, int nx, int ny, int i,
                                           int j, double f0, double dx, double dy,
                                           double sdd_thresh, double f_min,
                                           double2* __restrict__ pts, double& sdd) {
    // the reference's expressions in its source order, uncontracted: ridge
    // points and second derivatives equal the oracle's bit for bit, so the
    // ordered-ridge linking (which compares them) takes the same decisions
#pragma clang fp contract(off)
    if (i < 2 || i >= nx - 2 || j < 2 || j >= ny - 2) return false;
    if (!(f0 > f_min)) return false;
    const long k = static_cast<long>(i) * ny + j;
    const double fe = f[k + ny], fw = f[k - ny], fn = f[k + 1], fs = f[k - 1];
    const double fx = (fe - fw) / (2 * dx);
    const double fy = (fn - fs) / (2 * dy);
    const double fxx = (fe - 2 * f0 + fw) / (dx * dx);
    const double fyy = (fn - 2 * f0 + fs) / (dy * dy);
    const double fxy =
        (f[k + ny + 1] - f[k + ny - 1] - f[k - ny + 1] + f[k - ny - 1]) / (4 * dx * dy);
    const double2 e = evec[k];
    const double ex = e.x, ey = e.y;
    const double c2 = ex * (fxx * ex + fxy * ey) + ey * (fxy * ex + fyy * ey);
    if (!(c2 < -sdd_thresh)) return false;
    const double t = -(fx * ex + fy * ey) / c2;
    if (!(fabs(t * ex) <= dx / 2 && fabs(t * ey) <= dy / 2)) return false;
    pts[k] = make_double2(xs[i] + t * ex, ys[j] + t * ey);
    sdd = c2;
    return true;
}

// flag[k] = 1 where the test passes, 0 elsewhere
__global__ __launch_bounds__(256) void k_ridge_predicate(
    const double* __restrict__ f, const double2* __restrict__ evec, const double* __restrict__ xs,
    const double* __restrict__ ys, int nx, int ny, double dx, double dy, double sdd_thresh,
    const double* __restrict__ fmin_dev, int32_t* __restrict__ flag, double2* __restrict__ pts,
    double* __restrict__ sdd_out) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    const int i = blockIdx.y * 4 + threadIdx.y;
    if (i >= nx || j >= ny) return;
    const long k = static_cast<long>(i) * ny + j;
    double sdd = 0.0;
    flag[k] = ridge_test(f, evec, xs, ys, nx, ny, i, j, f[k], dx, dy, sdd_thresh,
                         fmin_dev ? *fmin_dev : 0.0, pts, sdd);
    if (sdd_out != nullptr) sdd_out[k] = sdd;
}

// ---------------------------------------------------------------------------
// Exclusive scan of int32 values, or of int32 pairs scanned together (sums
// must fit in int32).

struct I2 {
    int32_t a, b;
};
__device__ __forceinline__ I2 operator+(I2 x, I2 y) { return I2{x.a + y.a, x.b + y.b}; }
__device__ __forceinline__ I2& operator+=(I2& x, I2 y) {
    x.a += y.a;
    x.b += y.b;
    return x;
}

__device__ __forceinline__ int32_t lane_up(int32_t x, int off) { return __shfl_up(x, off); }
__device__ __forceinline__ I2 lane_up(I2 x, int off) {
    return I2{__shfl_up(x.a, off), __shfl_up(x.b, off)};
}

// over the block's kScanThreads values; sh holds one value per wavefront
template <class T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* sh, T* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const T y = lane_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) sh[w] = x;
    const T prev = lane_up(x, 1);
    T ex = lane > 0 ? prev : T{};
    __syncthreads();
    T sum{};
#pragma unroll
    for (int q = 0; q < kScanThreads / 64; ++q) {
        if (q == w) ex += sum;
        sum += sh[q];
    }
    *total = sum;
    __syncthreads();
    return ex;
}

template <class T>
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(const T* in, int64_t n, T* out,
                                                             T* __restrict__ tile_sums) {
    __shared__ T sh[kScanThreads / 64];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
    T v[kScanItems];
    T sum{};
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
        v[q] = base + q < n ? in[base + q] : T{};
        sum += v[q];
    }
    T total;
    T run = block_exclusive_scan(sum, sh, &total);
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
        if (base + q < n) out[base + q] = run;
        run += v[q];
    }
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// single block: exclusive scan of the tile sums in place; grand total to *total
template <class T>
__global__ __launch_bounds__(kScanThreads) void k_scan_sums(T* __restrict__ sums, int64_t m,
                                                            T* __restrict__ total) {
    __shared__ T sh[kScanThreads / 64];
    constexpr int kItems = 8;
    T carry{};
    for (int64_t base = 0; base < m; base += kScanThreads * kItems) {
        const int64_t k = base + threadIdx.x * kItems;
        T v[kItems], sum{}, chunk;
#pragma unroll
        for (int q = 0; q < kItems; ++q) {
            v[q] = k + q < m ? sums[k + q] : T{};
            sum += v[q];
        }
        T run = carry + block_exclusive_scan(sum, sh, &chunk);
#pragma unroll
        for (int q = 0; q < kItems; ++q) {
            if (k + q < m) sums[k + q] = run;
            run += v[q];
        }
        carry += chunk;
    }
    if (threadIdx.x == 0) *total = carry;
}

template <class T>
__global__ __launch_bounds__(256) void k_scan_add(T* __restrict__ out, int64_t n,
                                                  const T* __restrict__ tile_sums) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n) out[k] += tile_sums[k / kScanTile];
}

template <class T>
__global__ void k_set_zero(T* p) {
    *p = T{};
}

// out = exclusive scan of in; *total (device) = sum.  tmp holds
// ceil(n / 1024) values of T.
template <class T>
int exclusive_scan(const T* in, int64_t n, T* out, T* tmp, T* total, hipStream_t s) {
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (n == 0) {
        k_set_zero<<<1, 1, 0, s>>>(total);
        NBX_LAUNCHED("set_zero");
        return 0;
    }
    k_scan_tiles<<<static_cast<unsigned>(tiles), kScanThreads, 0, s>>>(in, n, out, tmp);
    NBX_LAUNCHED("scan_tiles");
    k_scan_sums<<<1, kScanThreads, 0, s>>>(tmp, tiles, total);
    NBX_LAUNCHED("scan_sums");
    k_scan_add<<<blocks_for(n, 256), 256, 0, s>>>(out, n, tmp);
    NBX_LAUNCHED("scan_add");
    return 0;
}

// The first two phases only: out holds each value's exclusive scan within
// its 1024-value tile and tile_off the tiles' offsets, so a consumer reads
// out[k] + tile_off[k / kScanTile] and no third pass is launched.
template <class T>
int exclusive_scan_tiled(const T* in, int64_t n, T* out, T* tile_off, T* total, hipStream_t s) {
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (n == 0) {
        k_set_zero<<<1, 1, 0, s>>>(total);
        NBX_LAUNCHED("set_zero");
        return 0;
    }
    k_scan_tiles<<<static_cast<unsigned>(tiles), kScanThreads, 0, s>>>(in, n, out, tile_off);
    NBX_LAUNCHED("scan_tiles");
    k_scan_sums<<<1, kScanThreads, 0, s>>>(tile_off, tiles, total);
    NBX_LAUNCHED("scan_sums");
    return 0;
}

// ---------------------------------------------------------------------------
// Compaction of flagged points in raveled order (pos: the flags' scan).
__global__ void k_compact(const int32_t* __restrict__ flag, const int32_t* __restrict__ pos,
                          const double2* __restrict__ pts_dense, int64_t n,
                          double2* __restrict__ pts_out) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n && flag[k]) pts_out[pos[k]] = pts_dense[k];
}

// ---------------------------------------------------------------------------
// Union-find labelling.
__device__ __forceinline__ int32_t uf_load(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int32_t uf_root(const int32_t* par, int32_t a) {
    int32_t p = uf_load(par + a);
    while (p != a) {
        a = p;
        p = uf_load(par + a);
    }
    return a;
}

__device__ void uf_unite(int32_t* par, int32_t a, int32_t b) {
    for (;;) {
        a = uf_root(par, a);
        b = uf_root(par, b);
        if (a == b) return;
        if (a < b) {
            const int32_t t = a;
            a = b;
            b = t;
        }
        // a > b: hang root a under b; if a stopped being a root meanwhile,
        // continue with what it now points to
        const int32_t old = atomicMin(par + a, b);
        if (old == a) return;
        a = old;
    }
}

__global__ void k_uf_init(const int32_t* __restrict__ flag, int64_t n, int32_t* __restrict__ par) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n) par[k] = flag[k] ? static_cast<int32_t>(k) : -1;
}

__global__ __launch_bounds__(256) void k_uf_union(const int32_t* __restrict__ flag, int nx, int ny,
                                                  int32_t* par) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    const int i = blockIdx.y * 4 + threadIdx.y;
    if (i >= nx || j >= ny) return;
    const int32_t k = i * ny + j;
    if (!flag[k]) return;
    if (j > 0 && flag[k - 1]) uf_unite(par, k, k - 1);
    if (i > 0) {
        const int32_t up = k - ny;
        if (j > 0 && flag[up - 1]) uf_unite(par, k, up - 1);
        if (flag[up]) uf_unite(par, k, up);
        if (j + 1 < ny && flag[up + 1]) uf_unite(par, k, up + 1);
    }
}

__global__ void k_uf_flatten(const int32_t* __restrict__ flag, int64_t n, int32_t* par) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n && flag[k]) par[k] = uf_root(par, static_cast<int32_t>(k));
}

__global__ void k_bytes_to_flags(const uint8_t* __restrict__ b, int64_t n,
                                 int32_t* __restrict__ flag) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n) flag[k] = b[k] ? 1 : 0;
}

__global__ void k_is_root(const int32_t* __restrict__ par, int64_t n, int32_t* __restrict__ out) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n) out[k] = par[k] == static_cast<int32_t>(k) ? 1 : 0;
}

__global__ void k_label_out(const int32_t* __restrict__ par, const int32_t* __restrict__ root_rank,
                            int64_t n, int32_t* __restrict__ labels) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k < n) labels[k] = par[k] >= 0 ? root_rank[par[k]] + 1 : 0;
}

// ---------------------------------------------------------------------------
// The grouped pipeline's labelling: par[k] = -1 off the ridges.

constexpr int kTileRows = 16, kTileCols = 64;

__device__ __forceinline__ int tile_root(const int* par, int a) {
    int p = __hip_atomic_load(par + a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (p != a) {
        a = p;
        p = __hip_atomic_load(par + a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return a;
}

__device__ __forceinline__ void tile_unite(int* par, int a, int b) {
    for (;;) {
        a = tile_root(par, a);
        b = tile_root(par, b);
        if (a == b) return;
        const int hi = a > b ? a : b, lo = a > b ? b : a;
        const int old = atomicMin(par + hi, lo);
        if (old == hi) return;
        a = old;
        b = lo;
    }
}

// Ridge predicate and the components within one 16 x 64 tile, linked in LDS:
// a global link is a chain of loads past the caches, so those are left to the
// tiles' borders (k_border_union), 8% of the points.  Position order within a
// tile is raveled order, so a tile's root is its component's smallest raveled
// index there.  The points above the threshold are listed first, so the test and
// the links run on full wavefronts.  Bound by memory (f, and the scattered lines
// of evec and pts at a tenth of the points): 2001 x 4001 points 62 us (predicate)
// + 80 us (every link global) -> 59 + 15 us.  Tiles of 8 and 32 rows are no
// faster.
__global__ __launch_bounds__(256) void k_ridge_label(
    const double* __restrict__ f, const double2* __restrict__ evec, const double* __restrict__ xs,
    const double* __restrict__ ys, int nx, int ny, double dx, double dy, double sdd_thresh,
    const double* __restrict__ fmin_dev, double2* __restrict__ pts, int32_t* __restrict__ par) {
    constexpr int kPoints = kTileRows * kTileCols, kRows = kTileRows / 4;
    __shared__ int own[kPoints];
    __shared__ uint16_t list[kPoints];  // points above the threshold
    __shared__ int listed;
    const int lj = threadIdx.x, t = threadIdx.y * kTileCols + lj;
    const int j0 = blockIdx.x * kTileCols, i0 = blockIdx.y * kTileRows, j = j0 + lj;
    const double f_min = fmin_dev ? *fmin_dev : 0.0;
    if (t == 0) listed = 0;
    double f0[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
        const int i = i0 + threadIdx.y + 4 * q;
        f0[q] = i < nx && j < ny ? f[static_cast<int64_t>(i) * ny + j] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
        const int i = i0 + threadIdx.y + 4 * q, at = (i - i0) * kTileCols + lj;
        const bool on = i < nx && j < ny && f0[q] > f_min;
        const uint64_t m = __ballot(on);
        own[at] = -1;
        if (m == 0) continue;
        int first = 0;
        if (lj == 0) first = atomicAdd(&listed, __popcll(m));
        first = __builtin_amdgcn_readfirstlane(first);
        if (on) list[first + __popcll(m & ((1ull << lj) - 1))] = static_cast<uint16_t>(at);
    }
    __syncthreads();
    const int count = listed;
    for (int c = t; c < count; c += 256) {
        const int at = list[c], i = i0 + at / kTileCols, jj = j0 + at % kTileCols;
        double sdd;
        if (ridge_test(f, evec, xs, ys, nx, ny, i, jj, f[static_cast<int64_t>(i) * ny + jj], dx, dy,
                       sdd_thresh, f_min, pts, sdd))
            own[at] = at;
    }
    __syncthreads();
    for (int c = t; c < count; c += 256) {
        const int at = list[c], li = at / kTileCols, l = at % kTileCols, up = at - kTileCols;
        if (own[at] < 0) continue;
        // with the point above set, the other neighbours are linked to it by
        // their own links; likewise the upper left one to the left one
        if (li > 0 && own[up] >= 0) {
            tile_unite(own, at, up);
            continue;
        }
        if (l > 0 && own[at - 1] >= 0) tile_unite(own, at, at - 1);
        else if (li > 0 && l > 0 && own[up - 1] >= 0) tile_unite(own, at, up - 1);
        if (li > 0 && l < kTileCols - 1 && own[up + 1] >= 0) tile_unite(own, at, up + 1);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
        const int li = threadIdx.y + 4 * q, at = li * kTileCols + lj;
        if (i0 + li >= nx || j >= ny) continue;
        int32_t r = -1;
        if (own[at] >= 0) {
            const int a = tile_root(own, at);
            r = (i0 + a / kTileCols) * ny + j0 + a % kTileCols;
        }
        par[static_cast<int64_t>(i0 + li) * ny + j] = r;
    }
}

// Links across the tiles' borders: thread t < rows * ny is a point of a tile's
// first row against the row above, the others are a row's pair across a border
// between tile columns.
__global__ __launch_bounds__(256) void k_border_union(int nx, int ny, int rows, int cols,
                                                      int32_t* par) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    const int64_t across = static_cast<int64_t>(rows) * ny;
    if (t < across) {
        const int i = (static_cast<int>(t / ny) + 1) * kTileRows, j = static_cast<int>(t % ny);
        const int32_t k = i * ny + j, up = k - ny;
        if (uf_load(par + k) < 0) return;
        if (uf_load(par + up) >= 0) {
            uf_unite(par, k, up);
            return;
        }
        if (j > 0 && uf_load(par + up - 1) >= 0) uf_unite(par, k, up - 1);
        if (j + 1 < ny && uf_load(par + up + 1) >= 0) uf_unite(par, k, up + 1);
        return;
    }
    const int64_t u = t - across;
    if (u >= static_cast<int64_t>(cols) * nx) return;
    const int i = static_cast<int>(u / cols), j = (static_cast<int>(u % cols) + 1) * kTileCols;
    const int32_t k = i * ny + j;
    const bool right = uf_load(par + k) >= 0, left = uf_load(par + k - 1) >= 0;
    if (right && left) {
        uf_unite(par, k, k - 1);
    } else if (i > 0) {
        if (right && uf_load(par + k - ny - 1) >= 0) uf_unite(par, k, k - ny - 1);
        if (left && uf_load(par + k - ny) >= 0) uf_unite(par, k - 1, k - ny);
    }
}

// Path flattening, and per kScanTile points the numbers of (ridge points,
// roots).
__global__ __launch_bounds__(kScanThreads) void k_flatten_count(int64_t n, int32_t* par,
                                                                I2* __restrict__ sums) {
    __shared__ I2 sh[kScanThreads / 64];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x;
    I2 c{0, 0};
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
        const int64_t k = base + q * kScanThreads;
        const int32_t p = k < n ? uf_load(par + k) : -1;
        if (p < 0) continue;
        const int32_t r = uf_root(par, p);
        if (r != p) __hip_atomic_store(par + k, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        c += I2{1, r == k ? 1 : 0};
    }
    I2 total;
    block_exclusive_scan(c, sh, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Ridge points in raveled order, and each root's number: components are
// numbered by root, i.e. by first pixel.
__global__ __launch_bounds__(kScanThreads) void k_compact_roots(
    const int32_t* __restrict__ par, int64_t n, const I2* __restrict__ tile_off,
    int32_t* __restrict__ idx, int32_t* __restrict__ number) {
    __shared__ I2 sh[kScanThreads / 64];
    const int64_t base =
        static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
    int32_t p[kScanItems];
    I2 c{0, 0}, total;
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
        p[q] = base + q < n ? par[base + q] : -1;
        c += I2{p[q] >= 0 ? 1 : 0, p[q] == base + q ? 1 : 0};
    }
    I2 at = block_exclusive_scan(c, sh, &total);
    if (total.a == 0) return;
    at += tile_off[blockIdx.x];
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
        if (p[q] < 0) continue;
        idx[at.a++] = static_cast<int32_t>(base + q);
        if (p[q] == base + q) number[base + q] = at.b++;
    }
}

// ---------------------------------------------------------------------------
// Stable radix sort of the ridge points by component number.  They come in
// raveled order, so after it each component's points are together and in that
// order.  A block takes kRadixTile points; a pass counts its digits (counts
// [digit][block]), scans the counts, and moves the points: each wavefront its
// own quarter, 64 at a time, a point's rank among the equal digits of its row
// from ballots.  Two passes cover 4 M components: 37 us at a capacity of 800,000
// points, and 19 us for the counts' scans (a bitonic sort of 2^20 64-bit keys
// took 280 us).  A tile of 4096 points leaves CUs idle (63 us), one of 512
// doubles the counts to scan.
constexpr int kRadixTile = 1024, kRadixBits = 11, kRadixWaves = kScanThreads / 64;

// FIRST: the numbers come from the labelling and are stored to comp
template <bool FIRST>
__global__ __launch_bounds__(kScanThreads) void k_radix_count(
    const int32_t* __restrict__ idx, const int32_t* __restrict__ par,
    const int32_t* __restrict__ number, const I2* __restrict__ total, int64_t m, int shift,
    int bits, int32_t* __restrict__ comp, int32_t* __restrict__ counts) {
    __shared__ int32_t h[1 << kRadixBits];
    const int bins = 1 << bits;
    for (int b = threadIdx.x; b < bins; b += kScanThreads) h[b] = 0;
    __syncthreads();
    const int64_t count = total->a < m ? total->a : m;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kRadixTile;
    for (int64_t t = base + threadIdx.x; t < base + kRadixTile && t < count; t += kScanThreads) {
        const int32_t c = FIRST ? number[par[idx[t]]] : comp[t];
        if (FIRST) comp[t] = c;
        atomicAdd(&h[(c >> shift) & (bins - 1)], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < bins; b += kScanThreads)
        counts[static_cast<int64_t>(b) * gridDim.x + blockIdx.x] = h[b];
}

__global__ __launch_bounds__(kScanThreads) void k_radix_move(
    const int32_t* __restrict__ idx, const int32_t* __restrict__ comp,
    const I2* __restrict__ total, int64_t m, int shift, int bits,
    const int32_t* __restrict__ starts, const int32_t* __restrict__ start_tile,
    int32_t* __restrict__ idx_out, int32_t* __restrict__ comp_out) {
    __shared__ int32_t next[kRadixWaves][1 << kRadixBits];
    const int64_t count = total->a < m ? total->a : m;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kRadixTile;
    if (first >= count) return;
    const int bins = 1 << bits, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int b = threadIdx.x; b < bins; b += kScanThreads)
#pragma unroll
        for (int q = 0; q < kRadixWaves; ++q) next[q][b] = 0;
    __syncthreads();
    constexpr int kQuarter = kRadixTile / kRadixWaves;
    const int64_t base = first + w * kQuarter;
    for (int r = 0; r < kQuarter; r += 64) {
        const int64_t t = base + r + lane;
        if (t < count) atomicAdd(&next[w][(comp[t] >> shift) & (bins - 1)], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < bins; b += kScanThreads) {
        const int64_t at = static_cast<int64_t>(b) * gridDim.x + blockIdx.x;
        int32_t run = starts[at] + start_tile[at / kScanTile];
#pragma unroll
        for (int q = 0; q < kRadixWaves; ++q) {
            const int32_t c = next[q][b];
            next[q][b] = run;
            run += c;
        }
    }
    __syncthreads();
    for (int r = 0; r < kQuarter && base + r < count; r += 64) {
        const int64_t t = base + r + lane;
        const bool in = t < count;
        const int32_t c = in ? comp[t] : 0, k = in ? idx[t] : 0;
        const int d = (c >> shift) & (bins - 1);
        uint64_t same = __ballot(in);
        for (int q = 0; q < bits; ++q) {
            const uint64_t set = __ballot(d >> q & 1);
            same &= d >> q & 1 ? set : ~set;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1));
        if (in) {
            const int32_t to = next[w][d] + rank;
            idx_out[to] = k;
            comp_out[to] = c;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (in && rank == 0) next[w][d] += static_cast<int32_t>(__popcll(same));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

__global__ void k_offsets_zero(int64_t* __restrict__ offsets) { offsets[0] = 0; }

// seg_first[c] = position of component c's first point in the sorted list;
// seg_first[nseg] = its length
__global__ void k_seg_first(const int32_t* __restrict__ comp, const I2* __restrict__ total,
                            int64_t cap, int32_t* __restrict__ seg_first) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t < cap && t < total->a && (t == 0 || comp[t] != comp[t - 1]))
        seg_first[comp[t]] = static_cast<int32_t>(t);
    if (t == 0) seg_first[total->b] = total->a;
}

// kept ridge sizes: len or 0
__global__ void k_seg_keep(const int32_t* __restrict__ seg_first, const I2* __restrict__ total,
                           int64_t cap, int min_pts, I2* __restrict__ kept) {
    const int64_t s = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (s >= cap) return;
    int32_t len = 0;
    if (s < total->b) len = seg_first[s + 1] - seg_first[s];
    const bool keep = len >= min_pts && len > 0;
    kept[s] = I2{keep ? len : 0, keep ? 1 : 0};
}

__global__ void k_group_scatter(const int32_t* __restrict__ idx, const int32_t* __restrict__ comp,
                                const int32_t* __restrict__ seg_first,
                                const I2* __restrict__ kept,
                                const I2* __restrict__ out_off_idx,
                                const I2* __restrict__ out_tile,
                                const I2* __restrict__ totals,
                                const double2* __restrict__ pts_dense,
                                const I2* __restrict__ all, int64_t cap,
                                double2* __restrict__ pts_out, int64_t* __restrict__ offsets) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t == 0) {
        const I2 tot = *totals;  // (points kept, ridges kept)
        offsets[tot.b] = tot.a;
    }
    if (t >= cap || t >= all->a) return;
    const int32_t s = comp[t];
    if (!kept[s].b) return;
    const I2 o = out_off_idx[s] + out_tile[s / kScanTile];  // output offset, ridge number
    const int32_t r = o.a + (static_cast<int32_t>(t) - seg_first[s]);
    pts_out[r] = pts_dense[idx[t]];
    if (t == seg_first[s]) offsets[o.b] = o.a;
}

// Bump allocator over one workspace block.
struct Arena {
    char* base;
    size_t used;
    template <class T>
    T* take(int64_t count) {
        const size_t bytes = (sizeof(T) * static_cast<size_t>(count) + 255) & ~static_cast<size_t>(255);
        T* p = reinterpret_cast<T*>(base + used);
        used += bytes;
        return p;
    }
};

size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }

// Read `count` (<= 16) int32 results back to the host: one DMA into a pinned
// staging buffer per host thread (allocated on the thread's first call and
// kept, 64 bytes), then a wait on the stream.  A pageable destination would
// make the runtime stage each copy itself, tens of microseconds apiece.
int read_counts(const int32_t* dev, int count, int32_t* host, hipStream_t s) {
    thread_local int32_t* pinned = nullptr;
    if (pinned == nullptr) NBX_HIP(hipHostMalloc(reinterpret_cast<void**>(&pinned), 64));
    NBX_HIP(hipMemcpyAsync(pinned, dev, sizeof(int32_t) * count, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    memcpy(host, pinned, sizeof(int32_t) * count);
    return 0;
}

// The percentile threshold, left at st->result (fmin_dev set to it); without
// one fmin_dev is NULL.
int ridge_threshold(const double* f, int64_t n, double percentile, SelState* st,
                    unsigned long long* held, const double** fmin_dev, hipStream_t s) {
    *fmin_dev = nullptr;
    if (percentile == 0) return 0;
    *fmin_dev = &st->result;
    return percentile_device(f, n, percentile, st, held, nullptr, s);
}

// Optional percentile + ridge predicate into flag and pts_dense (which holds
// the percentile's key list until then).
int run_predicate(const double* f, const double* evec, const double* x, const double* y, int nx,
                  int ny, double dx, double dy, double sdd_thresh, double percentile,
                  SelState* st, int32_t* flag, double2* pts_dense, hipStream_t s,
                  double* sdd = nullptr) {
    const double* fmin_dev;
    if (int rc = ridge_threshold(f, static_cast<int64_t>(nx) * ny, percentile, st,
                                 reinterpret_cast<unsigned long long*>(pts_dense), &fmin_dev, s))
        return rc;
    const dim3 block(64, 4), grid((ny + 63) / 64, (nx + 3) / 4);
    k_ridge_predicate<<<grid, block, 0, s>>>(f, reinterpret_cast<const double2*>(evec), x, y, nx,
                                             ny, dx, dy, sdd_thresh, fmin_dev, flag, pts_dense,
                                             sdd);
    NBX_LAUNCHED("ridge_predicate");
    return 0;
}

// Host linking and joining shared by both ordered-ridge entry points.
int link_and_join(const ordered::RidgeField& F, double dist_tol, double ep_tan_ang,
                  int min_ridge_pts, double sdd_thresh, double c, double* pts_host,
                  int64_t pts_cap, int64_t* offsets_host, int64_t offsets_cap,
                  int64_t* nridges_host, int64_t* npts_host) {
    const ordered::Linked L = ordered::link(F, sdd_thresh, c);
    std::vector<double> out;
    std::vector<int64_t> offsets;
    ordered::join(L, dist_tol, ep_tan_ang, min_ridge_pts, out, offsets);
    const int64_t nr = static_cast<int64_t>(offsets.size()) - 1;
    const int64_t np_ = static_cast<int64_t>(out.size() / 2);
    *nridges_host = nr;
    *npts_host = np_;
    NBX_REQUIRE(np_ <= pts_cap && nr + 1 <= offsets_cap,
                "output buffers too small (the counts hold the sizes needed)");
    std::copy(out.begin(), out.end(), pts_host);
    std::copy(offsets.begin(), offsets.end(), offsets_host);
    return 0;
}

int check_grid(int nx, int ny) {
    NBX_REQUIRE(nx >= 0 && ny >= 0, "negative grid size");
    NBX_REQUIRE(static_cast<int64_t>(nx) * ny < (static_cast<int64_t>(1) << 31) - 1,
                "grid too large for 32-bit point indices");
    return 0;
}

constexpr size_t kNoAllocScratchBytes = sizeof(scratch);  // 64 MiB
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
char* g_scratch_addr[kMaxDevices] = {};  // per-device address of `scratch`

int scratch_address(char** out) {
    int dev = 0;
    NBX_HIP(hipGetDevice(&dev));
    NBX_REQUIRE(dev >= 0 && dev < kMaxDevices, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_addr[dev] == nullptr) {
        void* p = nullptr;
        NBX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        NBX_REQUIRE(p != nullptr, "hipGetSymbolAddress returned NULL for the scratch array");
        g_scratch_addr[dev] = static_cast<char*>(p);
    }
    *out = g_scratch_addr[dev];
    return 0;
}

// Scratch layout of the grouped-ridge pipeline for n grid points.
struct RidgeLayout {
    SelState* st;
    int32_t *par, *number, *idx[2], *comp[2], *seg_first, *tmp, *counts;
    // total[0..1] = the pair scan's (points, ridges) total, total[2..3] = (ridge
    // points, components): one read-back fetches the first three
    int32_t* total;
    I2 *kept, *out_off_idx, *tmp2;
    double2* dense;
    void carve(Arena& A, int64_t n) {
        const int64_t tiles = (n + kScanTile - 1) / kScanTile;
        st = A.take<SelState>(1);
        dense = A.take<double2>(n);  // first the percentile's key list
        par = A.take<int32_t>(n);
        number = A.take<int32_t>(n);  // component number, at its root
        for (int q = 0; q < 2; ++q) {
            idx[q] = A.take<int32_t>(n);  // ridge points and their components, in turn
            comp[q] = A.take<int32_t>(n);
        }
        seg_first = A.take<int32_t>(n + 1);
        kept = A.take<I2>(n);         // (kept length, kept flag) per component
        out_off_idx = A.take<I2>(n);  // their exclusive scans
        tmp2 = A.take<I2>(tiles + 1);  // tile offsets of the pair scans
        // digit counts (scanned in place) and their tile offsets
        const int64_t digits = radix_counts(n);
        counts = A.take<int32_t>(digits);
        tmp = A.take<int32_t>((digits + kScanTile - 1) / kScanTile + 1);
        total = A.take<int32_t>(4);
    }
    // passes and bits a pass for component numbers below m
    static int radix_passes(int64_t m, int* bits) {
        int width = 1;
        while ((static_cast<int64_t>(1) << width) < m) ++width;
        const int passes = (width + kRadixBits - 1) / kRadixBits;
        *bits = (width + passes - 1) / passes;
        return passes;
    }
    static int64_t radix_counts(int64_t m) {
        // (the widest digit: a smaller m may take more bits a pass than n does)
        return (static_cast<int64_t>(1) << kRadixBits) * ((m + kRadixTile - 1) / kRadixTile);
    }
    static size_t bytes(int64_t n) {
        RidgeLayout L;
        Arena measure{nullptr, 0};
        L.carve(measure, n);
        return measure.used;
    }
};

// What a grid of n points counts against the fixed scratch: 60 bytes a point
// and 8 of the power of two that holds them, the stated limit of about 980,000
// points.  It covers RidgeLayout::bytes (68 bytes a point and 60 KB) wherever
// that could pass 64 MiB: the power of two is well above 980,000 there.
size_t noalloc_need(int64_t n) {
    const size_t p = static_cast<size_t>(n), tiles = (p + kScanTile - 1) / kScanTile;
    size_t pow2 = 1024;
    while (pow2 < p) pow2 <<= 1;
    return 6400 + 6 * align256(4 * p) + align256(16 * p) +
           align256(4 * (tiles + 1)) + align256(8 * (tiles + 1)) + align256(8 * pow2) +
           align256(4 * (p + 1)) + 2 * align256(8 * p) + 512;
}

// Count read-back without the pinned staging buffer (for callers that must
// not allocate): a copy into pageable host memory, then a wait.
int read_counts_pageable(const int32_t* dev, int count, int32_t* host, hipStream_t s) {
    NBX_HIP(hipMemcpyAsync(host, dev, sizeof(int32_t) * count, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    return 0;
}

// Counts of the asynchronous form: (ridges kept, points kept, ridge points
// before the length filter); -1 ridges if the points exceeded the grouping
// capacity m (not reachable: m bounds them, see ridges_run).
// `grouped` = 0 when the grouping stage did not run (capacity 0): its totals
// are then not this call's.
__global__ void k_counts_out(const int32_t* __restrict__ total, int64_t m, int grouped,
                             int64_t* __restrict__ counts) {
    if (threadIdx.x == 0) {
        const int32_t all = total[2];
        const int32_t kept = grouped ? total[0] : 0, ridges = grouped ? total[1] : 0;
        counts[0] = all > m ? -1 : ridges;
        counts[1] = kept;
        counts[2] = all;
    }
}

// (a kernel, not a memset: the call may be captured in a graph)
__global__ void k_counts_clear(int64_t* __restrict__ counts) {
    if (threadIdx.x < 3) counts[threadIdx.x] = 0;
}

// ftle_ridges on a scratch arena of at least RidgeLayout::bytes(nx*ny)
// bytes at `arena`; n = nx*ny > 0 and the arguments already checked.  With
// counts_dev set the counts go to device memory and nothing waits on the
// stream (then the grouping capacity without a percentile is the grid size:
// no count is read back).
int ridges_run(const double* f, const double* evec, const double* x, int nx, const double* y,
               int ny, double dx, double dy, double sdd_thresh, double percentile,
               int min_ridge_pts, double* pts, int64_t* offsets, int64_t* nridges_host,
               int64_t* npts_host, char* arena, bool pinned_counts, hipStream_t s,
               int64_t* counts_dev = nullptr) {
    const int64_t n = static_cast<int64_t>(nx) * ny;
    auto read = [&](const int32_t* dev, int count, int32_t* host) {
        return pinned_counts ? read_counts(dev, count, host, s)
                             : read_counts_pageable(dev, count, host, s);
    };
    RidgeLayout L;
    Arena A{arena, 0};
    L.carve(A, n);
    int32_t *par = L.par, *total = L.total;
    I2* const all = reinterpret_cast<I2*>(total + 2);
    const double* fmin_dev;
    if (int rc = ridge_threshold(f, n, percentile, L.st,
                                 reinterpret_cast<unsigned long long*>(L.dense), &fmin_dev, s))
        return rc;
    // ridge points and their components
    const int rows = (nx - 1) / kTileRows, cols = (ny - 1) / kTileCols;  // borders between tiles
    k_ridge_label<<<dim3(cols + 1, rows + 1), dim3(kTileCols, 4), 0, s>>>(
        f, reinterpret_cast<const double2*>(evec), x, y, nx, ny, dx, dy, sdd_thresh, fmin_dev,
        L.dense, par);
    NBX_LAUNCHED("ridge_label");
    const int64_t border = static_cast<int64_t>(rows) * ny + static_cast<int64_t>(cols) * nx;
    if (border > 0) {
        k_border_union<<<blocks_for(border, 256), 256, 0, s>>>(nx, ny, rows, cols, par);
        NBX_LAUNCHED("border_union");
    }
    // compact ridge points (raveled order) and number the components
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    k_flatten_count<<<static_cast<unsigned>(tiles), kScanThreads, 0, s>>>(n, par, L.tmp2);
    NBX_LAUNCHED("flatten_count");
    k_scan_sums<<<1, kScanThreads, 0, s>>>(L.tmp2, tiles, all);
    NBX_LAUNCHED("scan_sums");
    k_compact_roots<<<static_cast<unsigned>(tiles), kScanThreads, 0, s>>>(par, n, L.tmp2, L.idx[0],
                                                                         L.number);
    NBX_LAUNCHED("compact_roots");
    // The grouping stage works on the ridge points only (typically a few
    // percent of the grid), sized by a bound on their count; its kernels read
    // the exact count on the device.  With a percentile threshold q the bound
    // needs no read-back: a ridge point has f > f_min >= the order statistic
    // of rank floor((n-1) q/100), which at most n-1-that rank values exceed,
    // so the whole pipeline stays queued behind the work before it.  Without
    // one the count itself is read back.
    int64_t m = 0;
    if (percentile != 0) {
        const double vi = static_cast<double>(n - 1) * (percentile / 100.0);
        int64_t klo = static_cast<int64_t>(floor(vi));
        if (vi >= static_cast<double>(n - 1)) klo = n - 1;
        m = n - 1 - klo;
    } else if (counts_dev) {
        m = n;
    } else {
        int32_t cnt = 0;
        if (int rc = read(&all->a, 1, &cnt)) return rc;
        m = cnt;
    }
    if (m == 0) {
        k_offsets_zero<<<1, 1, 0, s>>>(offsets);
        NBX_LAUNCHED("offsets_zero");
        if (counts_dev) {
            // no ridge point passes (the grouping totals were not written)
            k_counts_out<<<1, 64, 0, s>>>(total, 0, 0, counts_dev);
            NBX_LAUNCHED("counts_out");
            return 0;
        }
        NBX_HIP(hipStreamSynchronize(s));
        return 0;
    }
    const unsigned nbm = blocks_for(m, 256);
    // order by (component, raveled index)
    int bits = 0;
    const int passes = RidgeLayout::radix_passes(m, &bits);
    const int64_t radix_blocks = (m + kRadixTile - 1) / kRadixTile;
    const unsigned rb = static_cast<unsigned>(radix_blocks);
    for (int q = 0; q < passes; ++q) {
        int32_t *idx = L.idx[q & 1], *comp = L.comp[q & 1];
        auto* count = q == 0 ? &k_radix_count<true> : &k_radix_count<false>;
        count<<<rb, kScanThreads, 0, s>>>(idx, par, L.number, all, m, q * bits, bits, comp,
                                          L.counts);
        NBX_LAUNCHED("radix_count");
        if (int rc = exclusive_scan_tiled(L.counts, radix_blocks << bits, L.counts, L.tmp,
                                          total, s))
            return rc;
        k_radix_move<<<rb, kScanThreads, 0, s>>>(idx, comp, all, m, q * bits, bits, L.counts,
                                                 L.tmp, L.idx[~q & 1], L.comp[~q & 1]);
        NBX_LAUNCHED("radix_move");
    }
    const int32_t *idx = L.idx[passes & 1], *comp = L.comp[passes & 1];
    // segments = components
    k_seg_first<<<nbm, 256, 0, s>>>(comp, all, m, L.seg_first);
    NBX_LAUNCHED("seg_first");
    k_seg_keep<<<nbm, 256, 0, s>>>(L.seg_first, all, m, min_ridge_pts, L.kept);
    NBX_LAUNCHED("seg_keep");
    // total and nridges are adjacent: the pair scan's total lands in both
    I2* totals = reinterpret_cast<I2*>(total);
    if (int rc = exclusive_scan_tiled(L.kept, m, L.out_off_idx, L.tmp2, totals, s)) return rc;
    // the scatter also writes offsets[nridges] = total
    k_group_scatter<<<nbm, 256, 0, s>>>(idx, comp, L.seg_first, L.kept, L.out_off_idx, L.tmp2,
                                        totals, L.dense, all, m, reinterpret_cast<double2*>(pts),
                                        offsets);
    NBX_LAUNCHED("group_scatter");
    if (counts_dev) {
        k_counts_out<<<1, 64, 0, s>>>(total, m, 1, counts_dev);
        NBX_LAUNCHED("counts_out");
        return 0;
    }
    int32_t h[3] = {0, 0, 0};  // points kept, ridges kept, ridge points (adjacent)
    if (int rc = read(total, 3, h)) return rc;
    // the grouping kernels clip to the capacity m; the percentile bound
    // guarantees count <= m, and a violation is reported, not truncated
    NBX_REQUIRE(h[2] <= m, "ridge-point count exceeds the grouping capacity");
    *nridges_host = h[1];
    *npts_host = h[0];
    return 0;
}


}  // namespace
}  // namespace nbx

using namespace nbx;

extern "C" {

int nbx_percentile(const double* f, int64_t n, double q, double* result, nbx_stream stream) {
    NBX_REQUIRE(f != nullptr && result != nullptr, "NULL array");
    hipStream_t s = as_stream(stream);
    // (one size for every n: a stream's first call allocates, and no later one
    // grows the buffer, so a call may be captured once any has run, and a captured
    // one keeps its buffer)
    Workspace ws(s, 2, align256(sizeof(SelState)) + 8 * kSelHeld);
    if (ws.error()) return ws.error();
    Arena A{ws.get(), 0};
    auto* st = A.take<SelState>(1);
    return percentile_device(f, n, q, st, A.take<unsigned long long>(kSelHeld), result, s);
}

int nbx_ridge_pts(const double* f, const double* evec, const double* x, int nx, const double* y,
                  int ny, double dx, double dy, double sdd_thresh, double percentile, double* pts,
                  int64_t* npts_host, nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(npts_host != nullptr, "npts_host is NULL");
    const int64_t n = static_cast<int64_t>(nx) * ny;
    *npts_host = 0;
    if (n == 0) return 0;
    NBX_REQUIRE(f && evec && x && y && pts, "NULL array");
    hipStream_t s = as_stream(stream);
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    const size_t bytes = align256(sizeof(SelState)) + align256(4 * n) * 2 + align256(16 * n) +
                         align256(4 * (tiles + 1)) + align256(4);
    Workspace ws(s, 1, bytes);
    if (ws.error()) return ws.error();
    Arena A{ws.get(), 0};
    auto* st = A.take<SelState>(1);
    auto* flag = A.take<int32_t>(n);
    auto* pos = A.take<int32_t>(n);
    auto* dense = A.take<double2>(n);
    auto* tmp = A.take<int32_t>(tiles + 1);
    auto* total = A.take<int32_t>(1);
    if (int rc = run_predicate(f, evec, x, y, nx, ny, dx, dy, sdd_thresh, percentile, st, flag,
                               dense, s))
        return rc;
    if (int rc = exclusive_scan(flag, n, pos, tmp, total, s)) return rc;
    k_compact<<<blocks_for(n, 256), 256, 0, s>>>(flag, pos, dense, n,
                                                 reinterpret_cast<double2*>(pts));
    NBX_LAUNCHED("compact");
    int32_t cnt = 0;
    if (int rc = read_counts(total, 1, &cnt, s)) return rc;
    *npts_host = cnt;
    return 0;
}

int nbx_ridges(const double* f, const double* evec, const double* x, int nx, const double* y,
               int ny, double dx, double dy, double sdd_thresh, double percentile,
               int min_ridge_pts, double* pts, int64_t* offsets, int64_t* nridges_host,
               int64_t* npts_host, nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(nridges_host != nullptr && npts_host != nullptr, "NULL count pointer");
    const int64_t n = static_cast<int64_t>(nx) * ny;
    *nridges_host = 0;
    *npts_host = 0;
    if (n == 0) return 0;
    NBX_REQUIRE(f && evec && x && y && pts && offsets, "NULL array");
    hipStream_t s = as_stream(stream);
    Workspace ws(s, 1, RidgeLayout::bytes(n));
    if (ws.error()) return ws.error();
    return ridges_run(f, evec, x, nx, y, ny, dx, dy, sdd_thresh, percentile, min_ridge_pts, pts,
                      offsets, nridges_host, npts_host, ws.get(), true, s);
}

int nbx_ridges_async(const double* f, const double* evec, const double* x, int nx,
                     const double* y, int ny, double dx, double dy, double sdd_thresh,
                     double percentile, int min_ridge_pts, double* pts, int64_t* offsets,
                     int64_t* counts, nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(counts != nullptr, "NULL counts");
    const int64_t n = static_cast<int64_t>(nx) * ny;
    hipStream_t s = as_stream(stream);
    if (n == 0) {
        k_counts_clear<<<1, 64, 0, s>>>(counts);
        NBX_LAUNCHED("counts_clear");
        return 0;
    }
    NBX_REQUIRE(f && evec && x && y && pts && offsets, "NULL array");
    Workspace ws(s, 1, RidgeLayout::bytes(n));
    if (ws.error()) return ws.error();
    int64_t unused_r = 0, unused_p = 0;
    return ridges_run(f, evec, x, nx, y, ny, dx, dy, sdd_thresh, percentile, min_ridge_pts, pts,
                      offsets, &unused_r, &unused_p, ws.get(), true, s, counts);
}

int nbx_ridges_noalloc(const double* f, const double* evec, const double* x, int nx,
                       const double* y, int ny, double dx, double dy, double sdd_thresh,
                       double percentile, int min_ridge_pts, double* pts, int64_t* offsets,
                       int64_t* nridges_host, int64_t* npts_host, nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(nridges_host != nullptr && npts_host != nullptr, "NULL count pointer");
    const int64_t n = static_cast<int64_t>(nx) * ny;
    *nridges_host = 0;
    *npts_host = 0;
    if (n == 0) return 0;
    NBX_REQUIRE(f && evec && x && y && pts && offsets, "NULL array");
    const size_t need = noalloc_need(n);
    if (need > kNoAllocScratchBytes) {
        set_error("nbx_ridges_noalloc: a grid of " + std::to_string(n) + " points needs " +
                  std::to_string(need) + " bytes of scratch, above its fixed " +
                  std::to_string(kNoAllocScratchBytes) + " (use nbx_ridges)");
        return -2;
    }
    char* base = nullptr;
    if (int rc = scratch_address(&base)) return rc;
    // every buffer the pipeline reads is written earlier in the same call
    // (counters and histograms are cleared by its own kernels), so the
    // previous call's contents need no clearing
    return ridges_run(f, evec, x, nx, y, ny, dx, dy, sdd_thresh, percentile, min_ridge_pts, pts,
                      offsets, nridges_host, npts_host, base, false, as_stream(stream));
}

int nbx_label8(const uint8_t* b, int nx, int ny, int32_t* labels, int32_t* nlabels_host,
               nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(nlabels_host != nullptr, "nlabels_host is NULL");
    const int64_t n = static_cast<int64_t>(nx) * ny;
    *nlabels_host = 0;
    if (n == 0) return 0;
    NBX_REQUIRE(b != nullptr && labels != nullptr, "NULL array");
    hipStream_t s = as_stream(stream);
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    const size_t bytes = align256(4 * n) * 4 + align256(4 * (tiles + 1)) + align256(4);
    Workspace ws(s, 1, bytes);
    if (ws.error()) return ws.error();
    Arena A{ws.get(), 0};
    auto* flag = A.take<int32_t>(n);
    auto* par = A.take<int32_t>(n);
    auto* isroot = A.take<int32_t>(n);
    auto* rank = A.take<int32_t>(n);
    auto* tmp = A.take<int32_t>(tiles + 1);
    auto* total = A.take<int32_t>(1);
    const unsigned nb = blocks_for(n, 256);
    k_bytes_to_flags<<<nb, 256, 0, s>>>(b, n, flag);
    NBX_LAUNCHED("bytes_to_flags");
    k_uf_init<<<nb, 256, 0, s>>>(flag, n, par);
    NBX_LAUNCHED("uf_init");
    const dim3 block(64, 4), grid((ny + 63) / 64, (nx + 3) / 4);
    k_uf_union<<<grid, block, 0, s>>>(flag, nx, ny, par);
    NBX_LAUNCHED("uf_union");
    k_uf_flatten<<<nb, 256, 0, s>>>(flag, n, par);
    NBX_LAUNCHED("uf_flatten");
    k_is_root<<<nb, 256, 0, s>>>(par, n, isroot);
    NBX_LAUNCHED("is_root");
    if (int rc = exclusive_scan(isroot, n, rank, tmp, total, s)) return rc;
    k_label_out<<<nb, 256, 0, s>>>(par, rank, n, labels);
    NBX_LAUNCHED("label_out");
    int32_t cnt = 0;
    if (int rc = read_counts(total, 1, &cnt, s)) return rc;
    *nlabels_host = cnt;
    return 0;
}

int nbx_ordered_ridges(const double* f, const double* evec, const double* x, int nx,
                       const double* y, int ny, double dist_tol, double ep_tan_ang,
                       int min_ridge_pts, double sdd_thresh, double percentile, double c,
                       double* pts_host, int64_t pts_cap, int64_t* offsets_host,
                       int64_t offsets_cap, int64_t* nridges_host, int64_t* npts_host,
                       nbx_stream stream) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(nridges_host != nullptr && npts_host != nullptr, "NULL count pointer");
    *nridges_host = 0;
    *npts_host = 0;
    const int64_t n = static_cast<int64_t>(nx) * ny;
    if (n == 0) return 0;
    NBX_REQUIRE(nx >= 2 && ny >= 2, "the ridge stencil needs at least 2 points per axis");
    NBX_REQUIRE(f && evec && x && y && pts_host && offsets_host, "NULL array");
    hipStream_t s = as_stream(stream);
    const size_t bytes = align256(sizeof(SelState)) + align256(4 * n) + align256(16 * n) +
                         align256(8 * n);
    Workspace ws(s, 1, bytes);
    if (ws.error()) return ws.error();
    Arena A{ws.get(), 0};
    auto* st = A.take<SelState>(1);
    auto* flag = A.take<int32_t>(n);
    auto* dense = A.take<double2>(n);
    auto* sdd = A.take<double>(n);
    double xh[2], yh[2];
    NBX_HIP(hipMemcpyAsync(xh, x, sizeof(xh), hipMemcpyDeviceToHost, s));
    NBX_HIP(hipMemcpyAsync(yh, y, sizeof(yh), hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    const double dx = xh[1] - xh[0], dy = yh[1] - yh[0];
    if (int rc = run_predicate(f, evec, x, y, nx, ny, dx, dy, sdd_thresh, percentile, st, flag,
                               dense, s, sdd))
        return rc;
    // the serial linking runs on the host over the dense per-point buffers
    std::vector<int32_t> fl(n);
    std::vector<double2> pt(n), ev(n);
    ordered::RidgeField F;
    F.nx = nx;
    F.ny = ny;
    F.h = dx < dy ? dx : dy;
    F.sdd.resize(n);
    NBX_HIP(hipMemcpyAsync(fl.data(), flag, 4 * n, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipMemcpyAsync(pt.data(), dense, 16 * n, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipMemcpyAsync(ev.data(), evec, 16 * n, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipMemcpyAsync(F.sdd.data(), sdd, 8 * n, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    F.px.resize(n);
    F.py.resize(n);
    F.vx.resize(n);
    F.vy.resize(n);
    for (int64_t k = 0; k < n; ++k) {
        F.px[k] = fl[k] ? pt[k].x : -1.0;
        F.py[k] = fl[k] ? pt[k].y : -1.0;
        F.vx[k] = ev[k].x;
        F.vy[k] = ev[k].y;
    }
    return link_and_join(F, dist_tol, ep_tan_ang, min_ridge_pts, sdd_thresh, c, pts_host, pts_cap,
                         offsets_host, offsets_cap, nridges_host, npts_host);
}

int nbx_ordered_ridges_link(const double* pts_dense, const double* eigvec_max, const double* sdd,
                            int nx, int ny, double h, double dist_tol, double ep_tan_ang,
                            int min_ridge_pts, double sdd_thresh, double c, double* pts_host,
                            int64_t pts_cap, int64_t* offsets_host, int64_t offsets_cap,
                            int64_t* nridges_host, int64_t* npts_host) {
    if (int rc = check_grid(nx, ny)) return rc;
    NBX_REQUIRE(nridges_host != nullptr && npts_host != nullptr, "NULL count pointer");
    *nridges_host = 0;
    *npts_host = 0;
    const int64_t n = static_cast<int64_t>(nx) * ny;
    if (n == 0) return 0;
    NBX_REQUIRE(pts_dense && eigvec_max && sdd && pts_host && offsets_host, "NULL array");
    NBX_REQUIRE(h > 0, "grid spacing must be positive");
    ordered::RidgeField F;
    F.nx = nx;
    F.ny = ny;
    F.h = h;
    F.px.resize(n);
    F.py.resize(n);
    F.vx.resize(n);
    F.vy.resize(n);
    F.sdd.assign(sdd, sdd + n);
    for (int64_t k = 0; k < n; ++k) {
        F.px[k] = pts_dense[2 * k];
        F.py[k] = pts_dense[2 * k + 1];
        F.vx[k] = eigvec_max[2 * k];
        F.vy[k] = eigvec_max[2 * k + 1];
    }
    for (int i = 0; i < nx; ++i)
        for (int j = 0; j < ny; ++j)
            NBX_REQUIRE(F.sdd[static_cast<int64_t>(i) * ny + j] >= 0 ||
                            (i >= 2 && i < nx - 2 && j >= 2 && j < ny - 2),
                        "ridge points (sdd < 0) must lie two or more points inside the grid");
    return link_and_join(F, dist_tol, ep_tan_ang, min_ridge_pts, sdd_thresh, c, pts_host, pts_cap,
                         offsets_host, offsets_cap, nridges_host, npts_host);
}

}  // extern "C"
