// Flow handles, spline prefilter and the DOP853 flow-map launches.
//
// Reference path: flowmap_grid_2D (integration.py:123-182) runs one
// numbalsoda.dop853 solve per grid point over a numba cfunc right-hand side.
// Here a lane, or a group of two or four, owns one particle: the right-hand side
// is a device functor inlined into the integrator, the state stays in registers
// (and LDS) for the whole solve, and the final position is written once.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <string>
#include <vector>

#include "common.h"
#include "dop853.h"
#include "flow_blocks.h"
#include "flow_handle.h"
#include "flows.h"
#include "queue.h"

namespace nbx {

namespace {
thread_local std::string g_last_error;
struct WsEntry {
    std::mutex m;  // held by the Workspace that uses the buffer
    void* ptr = nullptr;
    size_t bytes = 0;
};
// workspace slot of the queue launches that were not requested (never captured)
constexpr int kDefaultQueueSlot = 5;
std::mutex g_ws_mutex;  // guards the map, not the buffers
std::map<std::tuple<int, hipStream_t, int>, std::unique_ptr<WsEntry>> g_ws;
}  // namespace

void set_error(const std::string& msg) { g_last_error = msg; }

namespace {
// This thread's allocations in relaxed mode while it is in scope.
class RelaxedCapture {
   public:
    explicit RelaxedCapture(bool on) : on_(on) {
        if (on_) on_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess;
    }
    RelaxedCapture(const RelaxedCapture&) = delete;
    RelaxedCapture& operator=(const RelaxedCapture&) = delete;
    ~RelaxedCapture() {
        if (on_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }

   private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool on_;
};
}  // namespace

Workspace::Workspace(hipStream_t stream, int slot, size_t bytes, bool apart) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        set_error("hipGetDevice failed");
        err_ = -1;
        return;
    }
    WsEntry* e = nullptr;
    {
        std::lock_guard<std::mutex> g(g_ws_mutex);
        auto& slot_entry = g_ws[std::make_tuple(dev, stream, slot)];
        if (!slot_entry) slot_entry = std::make_unique<WsEntry>();
        e = slot_entry.get();
    }
    lock_ = std::unique_lock<std::mutex>(e->m);
    if (e->bytes < bytes) {
        const RelaxedCapture relaxed(apart);
        if (e->ptr) {
            // hipFree waits for the device work still using the old buffer
            (void)hipFree(e->ptr);
            e->ptr = nullptr;
            e->bytes = 0;
        }
        const size_t want = bytes < 4096 ? 4096 : bytes;
        if (device_malloc(&e->ptr, want) != hipSuccess) {
            set_error("workspace hipMalloc failed");
            err_ = -1;
            return;
        }
        e->bytes = want;
    }
    ptr_ = static_cast<char*>(e->ptr);
}

// Flow handles' memory: the blocks of closed flows (flow_blocks.h) per device.
namespace {
struct FlowMemory {
    static void* alloc(size_t bytes) {
        void* p = nullptr;
        if (hipMalloc(&p, bytes) == hipSuccess) return p;
        (void)hipGetLastError();
        return nullptr;
    }
    static void release(void* p) { (void)hipFree(p); }
};
using Blocks = FlowBlocks<FlowMemory>;
std::mutex g_blocks_mutex;
std::map<int, Blocks> g_blocks;  // per device

// A closing flow: its token is freed first, which waits for the device's work
// as freeing the arrays did, so blocks are held only when idle, whatever streams
// used them.  (hipDeviceSynchronize takes 20 us less, but invalidates every
// capture under way, another thread's of a batch among them; a free does so only
// where the capture's mode forbids frees.)
void flow_release(nbx_flow* fl) {
    int cur = fl->dev;
    (void)hipGetDevice(&cur);
    if (cur != fl->dev) (void)hipSetDevice(fl->dev);
    const bool idle = fl->token != nullptr && hipFree(fl->token) == hipSuccess;
    if (!idle) (void)hipGetLastError();
    {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        g_blocks[fl->dev].close({{fl->coef, fl->coef_bytes}, {fl->coef32, fl->coef32_bytes}}, idle);
    }
    if (cur != fl->dev) (void)hipSetDevice(cur);
}

// A new gridded flow on the current device, with its token: a small allocation
// of its own, refused where the runtime refuses allocations (during a capture),
// also when the arrays come from held blocks.
int flow_register(nbx_flow* fl) {
    if (hipGetDevice(&fl->dev) != hipSuccess) return -1;
    {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        g_blocks[fl->dev].open();
    }
    return device_malloc(&fl->token, 256) == hipSuccess ? 0 : -1;
}
template <class T>
bool flow_array(const nbx_flow* fl, T** p, size_t* bytes) {
    std::lock_guard<std::mutex> lock(g_blocks_mutex);
    const auto b = g_blocks[fl->dev].take(sizeof(T) * static_cast<size_t>(fl->ncoef));
    *p = static_cast<T*>(b.p);
    *bytes = b.bytes;
    return b.p != nullptr;
}
}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int dev = 0;
    bool any = false;
    if (hipGetDevice(&dev) == hipSuccess) {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        any = g_blocks[dev].give_back();
    }
    if (any) e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

// (u, v) pairs in FP64, and FP32 elements pairing time index t with t + 1
// (slab = one time slice of coefficients; the last slice repeats itself).
__global__ void k_interleave(const double* __restrict__ u, const double* __restrict__ v, int64_t n,
                             int64_t slab, double2* __restrict__ out,
                             float4* __restrict__ out32) {
    for (int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; k < n;
         k += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const double a = u[k], b = v[k];
        out[k] = make_double2(a, b);
        if (out32 == nullptr) continue;
        const int64_t k1 = k + slab < n ? k + slab : k;
        out32[k] = make_float4(static_cast<float>(a), static_cast<float>(b),
                               static_cast<float>(u[k1]), static_cast<float>(v[k1]));
    }
}

// 'xy' velocity samples (nt, ny, nx) to the 'ij' layout (nt, nx, ny), scaled
// (the moveaxis + unit conversion of plot_merra_ftle.py:37-41: m/s -> km/h
// is scale 3.6).  Writes are coalesced along y; the reads stride by nx.
// One 32x32 tile of one time slice per block, staged in LDS (a padding
// column keeps the column reads free of bank conflicts): the block reads 32
// rows of the 'xy' slice along x and writes 32 rows of the 'ij' slice along
// y, both coalesced.  blockIdx.y runs over (time, y-tile).
constexpr int kIngestTile = 32;
constexpr int kIngestRows = 8;  // threads per block: 32 x 8

__global__ __launch_bounds__(kIngestTile * kIngestRows) void k_ingest_xy(
    const double* __restrict__ in, int nt, int ny, int nx, double scale,
    double* __restrict__ out) {
    __shared__ double tile[kIngestTile][kIngestTile + 1];
    const int nty = (ny + kIngestTile - 1) / kIngestTile;
    const int64_t t = blockIdx.y / nty;
    const int by = static_cast<int>(blockIdx.y % nty) * kIngestTile;
    const int bx = static_cast<int>(blockIdx.x) * kIngestTile;
    const double* src = in + t * ny * static_cast<int64_t>(nx);
    double* dst = out + t * nx * static_cast<int64_t>(ny);
    const int tx = threadIdx.x, ty = threadIdx.y;
#pragma unroll
    for (int r = 0; r < kIngestTile; r += kIngestRows) {
        const int j = by + ty + r, i = bx + tx;
        if (j < ny && i < nx) tile[ty + r][tx] = src[static_cast<int64_t>(j) * nx + i];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kIngestTile; r += kIngestRows) {
        const int i = bx + ty + r, j = by + tx;
        if (i < nx && j < ny) dst[static_cast<int64_t>(i) * ny + j] = tile[tx][ty + r] * scale;
    }
}

// ---------------------------------------------------------------------------
// Flow-map kernels.

// Particle sources: a tensor grid x[i], y[j] in 'ij' order, or a point list.
// pos() returns false for a particle the source itself leaves out (its
// outputs are written as for a masked one); cell() is its mask index.
struct GridSource {
    const double* __restrict__ xs;
    const double* __restrict__ ys;
    int ny;
    int nx;
    // optional launch order of the 4 x 4 tiles (16 slots each): slot s runs
    // in tile order[s / 16] (see tile_order_edge_first)
    const int* __restrict__ order = nullptr;
    // slots of the grid launch: the tile order of tile_slots/tile_particle
    __host__ __device__ int64_t slots() const { return tile_slots(nx, ny); }
    __device__ __forceinline__ int64_t particle(int64_t slot) const {
        if (order != nullptr) slot = (static_cast<int64_t>(order[slot >> 4]) << 4) | (slot & 15);
        return tile_particle(slot, nx, ny);
    }
    __device__ __forceinline__ bool pos(int64_t p, double& px, double& py) const {
        const int64_t i = p / ny;
        px = xs[i];
        py = ys[p - i * ny];
        return true;
    }
    __device__ __forceinline__ int64_t cell(int64_t p) const { return p; }
};

struct PointSource {
    const double2* __restrict__ pts;
    __device__ __forceinline__ bool pos(int64_t p, double& px, double& py) const {
        const double2 q = pts[p];
        px = q.x;
        py = q.y;
        return true;
    }
    __device__ __forceinline__ int64_t cell(int64_t p) const { return p; }
};

// The auxiliary grid of flowmap_aux_grid_2D (integration.py:249-464):
// particle p = (i*ny + j)*naux + k starts at (x[i], y[j]) + offset k, the
// offsets being (h,0), (-h,0), (0,h), (0,-h) and, with eig_main, (0,0).
// On edge points only the centre particle runs (eig_main) or all four (not
// eig_main); without compute_edge edge points are left out.
struct AuxSource {
    const double* __restrict__ xs;
    const double* __restrict__ ys;
    int nx, ny, naux;
    double h;
    bool eig_main, compute_edge;
    __device__ __forceinline__ bool pos(int64_t p, double& px, double& py) const {
        const int64_t c = p / naux;
        const int k = static_cast<int>(p - c * naux);
        const int64_t i = c / ny;
        const int64_t j = c - i * ny;
        const bool edge = i == 0 || i == nx - 1 || j == 0 || j == ny - 1;
        if (edge && (!compute_edge || (eig_main && k != 4))) return false;
        const double ox = k == 0 ? h : (k == 1 ? -h : 0.0);
        const double oy = k == 2 ? h : (k == 3 ? -h : 0.0);
        px = xs[i] + ox;
        py = ys[j] + oy;
        return true;
    }
    __device__ __forceinline__ int64_t cell(int64_t p) const { return p / naux; }
};

// One solve per group of G lanes.  With G = 1 the lane holds both components;
// in groups of 2 or 4 even lanes hold x and odd lanes y (Solve in dop853.h), and
// the group's lanes split the right-hand side: the spline's gathers, the
// trilinear flow's time slices, the double gyre's library calls.
template <class Flow, class R, int G, class Src>
__global__ __launch_bounds__(256, (flowmap_min_waves<Flow, R, G>())) void k_flowmap(
    Flow f, Src src, int64_t P, double s0, double s1, double rtol, double atol,
    const uint8_t* __restrict__ mask, long long nmax, double2* __restrict__ out,
    int32_t* __restrict__ status, int32_t* __restrict__ nsteps) {
    f.prepare();
    const unsigned bid = xcd_block<Flow>();
    const int64_t tid = bid * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    int64_t p = tid / G;
    if (p >= P) return;  // whole groups leave together (P counts slots for grids)
    if constexpr (std::is_same<Src, GridSource>::value) {
        p = src.particle(p);
        if (p < 0) return;
    }
    const bool lead = (tid & (G - 1)) == 0;
    double px, py;
    const bool run = src.pos(p, px, py);
    if (!run || (mask != nullptr && mask[src.cell(p)])) {
        if (lead) {
            out[p] = make_double2(0.0, 0.0);
            if (status) status[p] = NBX_ST_MASKED;
            if (nsteps) nsteps[p] = 0;
        }
        return;
    }
    Solve<Flow, R, G> sv;
    auto& s = sv.s;
    sv.init(f, s0, s1, px, py, rtol, atol);
    while (sv.step(f, rtol, atol, nmax)) {
    }
    sv.store(out + p);
    if (lead) {
        if (status) status[p] = s.idid;
        if (nsteps) nsteps[p] = s.nstep;
    }
}

// Spline coefficients staged through LDS, 4 lanes per particle, one
// wavefront per 64-thread block (16 particles, a 4 x 4 tile of the grid).
// Before every attempted step the wavefront bounds where its stencils will
// fall -- times p0*[x, x+h] of its particles, positions from the current
// point along h times the current derivative with half that displacement
// as margin on either side, in the spline's lookup coordinates -- copies
// that box of coefficient elements (bt x bx x by, at most kStageElems of 16
// bytes) from HBM/L2 into LDS with row-contiguous loads, and every stencil
// inside it is then read from LDS (Spline3<..., S = true>); stencils outside
// (a stage that strays, a box too large) are gathered from global memory as
// in k_flowmap.  Per step a wavefront's stencils span a few hours and a few
// grid cells: median box 8 KiB, 23 KiB at the largest step of a typical
// tile on the gridded workload, against 192 KiB of gathered coefficients.
// The integrator's arithmetic is that of k_flowmap, so results are equal.
constexpr int kStageElems = 1280;  // 20 KiB: 8 one-wave blocks per CU

// One global_load_lds_dwordx4: lane l's 16 bytes at src go to LDS at
// dst + 16 l (dst wavefront-uniform).  The builtin exists only in the device
// compilation pass.
__device__ __forceinline__ void load_lds16(const void* src, void* dst) {
#if __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0,
                                     0);
#endif
}

__device__ __forceinline__ double wave_min_groups(double v) {
    // the four lanes of a group hold equal values: reduce over groups
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ double wave_max_groups(double v) {
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

template <class R>
__global__ __launch_bounds__(64) void k_flowmap_staged(
    Spline3<R, 4, false, true> f, GridSource src, int64_t P, double s0, double s1, double rtol,
    double atol, const uint8_t* __restrict__ mask, long long nmax, double2* __restrict__ out,
    int32_t* __restrict__ status, int32_t* __restrict__ nsteps) {
    using Pt = typename CoefPair<R>::type;
    __shared__ Pt stage[kStageElems];
    f.prepare();
    const int lane = static_cast<int>(threadIdx.x);
    const int64_t slot = static_cast<int64_t>(blockIdx.x) * 16 + (lane >> 2);
    const int64_t p = slot < P ? src.particle(slot) : -1;
    const bool lead = (lane & 3) == 0;
    bool running = p >= 0;
    if (running && mask != nullptr && mask[p]) {
        if (lead) {
            out[p] = make_double2(0.0, 0.0);
            if (status) status[p] = NBX_ST_MASKED;
            if (nsteps) nsteps[p] = 0;
        }
        running = false;
    }
    f.box.lds = stage;
    f.box.on = false;
    Solve<Spline3<R, 4, false, true>, R, 4> sv;
    auto& s = sv.s;
    if (running) {
        double px, py;
        src.pos(p, px, py);
        sv.init(f, s0, s1, px, py, rtol, atol);
    }
    auto finish = [&]() {
        sv.store(out + p);
        if (lead) {
            if (status) status[p] = s.idid;
            if (nsteps) nsteps[p] = s.nstep;
        }
    };
    const double inf = __builtin_inf();
    for (;;) {
        bool stepping = false;
        if (running) {
            stepping = dop853_step_begin(s, nmax);
            if (!stepping) {
                finish();
                running = false;
            }
        }
        if (!__any(stepping)) break;
        // ---- the step's box (wavefront-uniform)
        double tlo = inf, thi = -inf, xlo = inf, xhi = -inf, ylo = inf, yhi = -inf;
        if (stepping) {
            const double t0 = f.p0 * s.x, t1 = f.p0 * (s.x + s.h);
            tlo = fmin(t0, t1);
            thi = fmax(t0, t1);
            const double e = s.h * static_cast<double>(s.k1);
            const double ex = quad_move<kPairEven>(e), ey = quad_move<kPairOdd>(e);
            const double m = 0.5 * (fabs(ex) + fabs(ey));
            const double px = quad_move<kPairEven>(s.y), py = quad_move<kPairOdd>(s.y);
            const double a = f.lookup_x(px + fmin(0.0, ex) - m);
            const double b = f.lookup_x(px + fmax(0.0, ex) + m);
            if (a <= b) {
                xlo = a;
                xhi = b;
            } else {  // the box straddles the longitude wrap: no staging
                xlo = -inf;
                xhi = inf;
            }
            ylo = py + fmin(0.0, ey) - m;
            yhi = py + fmax(0.0, ey) + m;
        }
        tlo = wave_min_groups(tlo);
        thi = wave_max_groups(thi);
        xlo = wave_min_groups(xlo);
        xhi = wave_max_groups(xhi);
        ylo = wave_min_groups(ylo);
        yhi = wave_max_groups(yhi);
        int c0[3], c1[3];
        const double q0[3] = {tlo, xlo, ylo}, q1[3] = {thi, xhi, yhi};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            R fr;
            f.cell(d, fmin(fmax(q0[d], f.lo[d]), f.hi[d]), c0[d], fr);
            f.cell(d, fmin(fmax(q1[d], f.lo[d]), f.hi[d]), c1[d], fr);
        }
        const int bt = c1[0] - c0[0] + 4, bx = c1[1] - c0[1] + 4, by = c1[2] - c0[2] + 4;
        const int size = bt * bx * by;
        const bool fits = xlo > -inf && by <= 64 && ((size + 63) & ~63) <= kStageElems;
        f.box.it0 = c0[0];
        f.box.ix0 = c0[1];
        f.box.iy0 = c0[2];
        f.box.bt = bt;
        f.box.bx = bx;
        f.box.by = by;
        f.box.on = fits;
        if (fits) {
            // element e = (a*bx + b)*by + c of the box, 64 a pass: each
            // global_load_lds_dwordx4 writes the wavefront's 64 elements to
            // consecutive LDS slots, the loads all in flight at once.  Lanes
            // past the end (last pass) reload the last element into slots
            // below the rounded-up size, which no stencil reads.
            const float rby = __builtin_amdgcn_rcpf(static_cast<float>(by));
            const float rbx = __builtin_amdgcn_rcpf(static_cast<float>(bx));
            const int passes = (size + 63) >> 6;
            for (int k = 0; k < passes; ++k) {
                const int e = min(k * 64 + lane, size - 1);
                const int r = static_cast<int>((static_cast<float>(e) + 0.5f) * rby);
                const int c = e - r * by;
                const int a = static_cast<int>((static_cast<float>(r) + 0.5f) * rbx);
                const int b = r - a * bx;
                const Pt* src_e = f.C + (static_cast<long>(c0[0] + a) * f.st +
                                         static_cast<long>(c0[1] + b) * f.sx + (c0[2] + c));
                load_lds16(src_e, stage + k * 64);
            }
            __builtin_amdgcn_s_waitcnt(0);
        }
        __syncthreads();
        if (stepping) {
            running = sv.body(f, rtol, atol);
            if (!running) finish();
        }
        __syncthreads();  // every read of the box is done before the next copy
    }
}

template <class Flow, class R>
__global__ void k_flow_eval(Flow f, const double* __restrict__ t, const double2* __restrict__ pts,
                            int64_t n, double2* __restrict__ out) {
    f.prepare();
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k >= n) return;
    R a, b;
    f(t[k], pts[k].x, pts[k].y, a, b);
    out[k] = make_double2(static_cast<double>(a), static_cast<double>(b));
}

// defaults: the best shapes measured on the gridded-velocity, double-gyre
// and Bickley workloads; the autotuner overrides them per workload.  One-wave
// blocks let each wavefront's slot go to the next as it ends (double gyre,
// 3,321 particles: 320 us with 256 threads, 187 with 64; 2 M: 2.87, 2.80 ms).
// The Bickley jet's long trajectories leave a third of the grid launch idle
// behind its last wavefronts, so it runs the tile queue at its kernels'
// occupancy (2 and 3 wavefronts per SIMD): 401,401 particles 17.1 -> 14.0 ms,
// float 10.0 -> 8.0; 1.6 M 49.6 -> 46.4 ms.
constexpr LaunchCfg kDefaultCfg[4][2] = {{{1, 64, 0}, {1, 64, 0}},
                                         {{1, 64, 8}, {1, 64, 12}},
                                         {{4, 128, 0}, {4, 128, 0}},
                                         {{1, 64, 0}, {1, 64, 0}}};
LaunchCfg g_cfg[4][2] = {{kDefaultCfg[0][0], kDefaultCfg[0][1]},
                         {kDefaultCfg[1][0], kDefaultCfg[1][1]},
                         {kDefaultCfg[2][0], kDefaultCfg[2][1]},
                         {kDefaultCfg[3][0], kDefaultCfg[3][1]}};
// edge-first tile order of the spline grid launch, per precision
int g_edge_first[2] = {1, 1};
std::mutex g_cfg_mutex;

LaunchCfg launch_cfg(int kind, int precision) {
    std::lock_guard<std::mutex> lock(g_cfg_mutex);
    return g_cfg[kind][precision];
}

struct SolveArgs {
    int64_t P;
    double s0, s1, rtol, atol;
    const uint8_t* mask;
    long long nmax;
    double2* out;
    int32_t* status;
    int32_t* nsteps;
};

int device_cu_count() {
    static std::mutex mu;
    static std::vector<int> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(mu);
    if (static_cast<int>(cache.size()) <= dev) cache.resize(dev + 1, 0);
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        cache[dev] = n;
    }
    return cache[dev];
}

// The single-grid request as a queue entry (grid sources only).
inline ReqDev single_request(const GridSource& src, const SolveArgs& a) {
    return ReqDev{a.s0, a.s1, src.xs, src.ys, static_cast<int>(a.P / src.ny), src.ny, a.mask,
                  a.out, a.status, a.nsteps};
}

// One launch with a group of G lanes for every particle.
template <class Flow, class R, int G, class Src>
int launch_grid(const Flow& f, const Src& src, const SolveArgs& a, int block, hipStream_t s) {
    int64_t slots = a.P;
    if constexpr (std::is_same<Src, GridSource>::value) slots = src.slots();
    k_flowmap<Flow, R, G, Src><<<blocks_for(slots * G, block), block,
                                 solve_lds_bytes<Flow, R, G>(block), s>>>(
        f, src, slots, a.s0, a.s1, a.rtol, a.atol, a.mask, a.nmax, a.out, a.status, a.nsteps);
    NBX_LAUNCHED("flowmap");
    return 0;
}

template <class Flow, class R, int G, class Src>
int launch_solve(const Flow& f, const Src& src, const SolveArgs& a, const LaunchCfg& cfg,
                 hipStream_t s) {
    const int block = cfg.block;
    if constexpr (std::is_same<Src, GridSource>::value) {
        if (cfg.persistent > 0) {  // persistent grid over the queue of particle tiles
            const int cus = device_cu_count();
            NBX_REQUIRE(cus > 0, "cannot query the compute-unit count");
            const int64_t slots = src.slots();
            if (slots == 0) return 0;
            const int64_t ntiles = slots / (64 / G);
            NBX_REQUIRE(ntiles < (int64_t(1) << 31), "too many particle tiles for the queue");
            const int64_t want = (ntiles * 64 + block - 1) / block;
            const int64_t most = static_cast<int64_t>(cus) * cfg.persistent;
            // The queue as a kind's default: with a wavefront for every tile
            // there is nothing to hand on; from 16 rounds of them the tail is a
            // few percent and not worth the states' memory.  A stream under
            // capture takes the grid launch too (the queue's workspace may have
            // to be allocated), and so do a call that cannot have it and one
            // that allows solves of any length.
            if (!cfg.requested) {
                hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
                (void)hipStreamIsCapturing(s, &capture);
                if (want <= most || want > 16 * most || a.nmax > kDefaultQueueSteps ||
                    capture != hipStreamCaptureStatusNone)
                    return launch_grid<Flow, R, G>(f, src, a, block, s);
            }
            const unsigned long long ring = chunk_ring(ntiles);
            const size_t state_off = ring * sizeof(unsigned long long) + 256;
            // (a slot of its own for the default: a captured queue's workspace
            // is grown by requested queues only)
            Workspace ws(s, cfg.requested ? 3 : kDefaultQueueSlot,
                         state_off + solve_state_bytes<R, G>() * static_cast<size_t>(slots),
                         !cfg.requested);
            if (ws.error()) {
                if (cfg.requested) return ws.error();
                return launch_grid<Flow, R, G>(f, src, a, block, s);
            }
            char* w = ws.get();
            const ChunkQueue q{reinterpret_cast<unsigned long long*>(w),
                               reinterpret_cast<unsigned long long*>(w + state_off - 256),
                               reinterpret_cast<unsigned long long*>(w + state_off - 128),
                               reinterpret_cast<unsigned long long*>(w + state_off - 64),
                               ring - 1, static_cast<unsigned long long>(ntiles)};
            k_chunk_init<<<blocks_for(static_cast<int64_t>(ring), 256), 256, 0, s>>>(q, ntiles);
            NBX_LAUNCHED("chunk_init");
            k_flowmap_chunks<Flow, R, G><<<static_cast<unsigned>(std::min(want, most)), block,
                                           solve_lds_bytes<Flow, R, G>(block), s>>>(
                f, single_request(src, a), nullptr, nullptr, 1, q,
                reinterpret_cast<decltype(Solve<Flow, R, G>::s)*>(w + state_off), a.rtol, a.atol,
                a.nmax);
            NBX_LAUNCHED("flowmap_chunks");
            return 0;
        }
    }
    return launch_grid<Flow, R, G>(f, src, a, block, s);
}

// Edge-first launch order of a grid's 4 x 4 particle tiles.  A particle
// that leaves the velocity box crosses the step from the spline's values to
// zero (extrapolation 0), where DOP853 cuts its steps and rejects some, so
// tiles near the box's edge take the most steps (gridded workload: 29.5
// steps per particle within 2 degrees of the edge, 21 beyond 10); launched
// in plain tile order some of them start last and form the launch's tail.
// The tiles are counted into 64 buckets by the distance of their centre
// particle to the box edge in velocity-grid cells (the last bucket also
// takes 63 cells and more, and the tiles past the particle grid's edge) and
// scattered bucket by bucket: order[k] is the tile launched k-th.  Within a
// bucket the order is whatever the atomics give; the launch order never
// changes a particle's result.
// Edge-first order: a counting sort of the tiles by bucket (distance of the
// centre of the tile's block of kOrderBlock x kOrderBlock particles to the
// nearest edge of the velocity box, in grid cells, clipped to 0..63).  Each block histograms its tiles in LDS and stores its
// 64 counts; the scatter derives every block's offsets from those counts
// (no global atomics: nearly every interior tile falls in the last bucket,
// and a shared global counter serialised them).
constexpr int kOrderThreads = 256;
#ifndef NBX_ORDER_BLOCK
#define NBX_ORDER_BLOCK 32
#endif
constexpr int64_t kOrderBlock = NBX_ORDER_BLOCK;  // particles per side, a multiple of 8

template <class Flow>
__global__ __launch_bounds__(kOrderThreads) void k_tile_order_keys(
    Flow f, GridSource src, int64_t tiles, int* __restrict__ bucket,
    unsigned* __restrict__ block_count) {
    __shared__ unsigned hist[64];
    if (threadIdx.x < 64) hist[threadIdx.x] = 0u;
    __syncthreads();
    const int64_t u = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (u < tiles) {
        const int64_t T = u >> 2, q = u & 3, ntj = (src.ny + 7) / 8;
        const int64_t i0 = (T / ntj) * 8 + (q >> 1) * 4, j0 = (T % ntj) * 8 + (q & 1) * 4;
        int b = 63;
        if (i0 < src.nx && j0 < src.ny) {
            // the centre of the tile's block of kOrderBlock x kOrderBlock
            // particles: whole blocks share a bucket, so each bucket is swept
            // band by band in tile order (compact working sets in L2)
            const int64_t ib = (i0 / kOrderBlock) * kOrderBlock + kOrderBlock / 2;
            const int64_t jb = (j0 / kOrderBlock) * kOrderBlock + kOrderBlock / 2;
            const int64_t i = ib < src.nx ? ib : src.nx - 1;
            const int64_t j = jb < src.ny ? jb : src.ny - 1;
            const double x = f.lookup_x(src.xs[i]), y = src.ys[j];
            const double d = fmin(fmin((x - f.lo[1]) * f.dinv[1], (f.hi[1] - x) * f.dinv[1]),
                                  fmin((y - f.lo[2]) * f.dinv[2], (f.hi[2] - y) * f.dinv[2]));
            b = d > 0 ? (d < 63 ? static_cast<int>(d) : 63) : 0;
        }
        bucket[u] = b;
        atomicAdd(&hist[b], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) block_count[blockIdx.x * 64 + threadIdx.x] = hist[threadIdx.x];
}

__global__ __launch_bounds__(kOrderThreads) void k_tile_order_scatter(
    const int* __restrict__ bucket, const unsigned* __restrict__ block_count, int nblocks,
    int64_t tiles, int* __restrict__ order) {
    // per bucket: the tiles of all blocks (total) and of the blocks before
    // this one (before), four partial sums per bucket over the block counts
    __shared__ unsigned total[4][64], before[4][64];
    __shared__ unsigned base[64], cursor[64];
    const int bk = threadIdx.x & 63, part = threadIdx.x >> 6;
    unsigned tot = 0u, bef = 0u;
    for (int k = part; k < nblocks; k += 4) {
        const unsigned c = block_count[k * 64 + bk];
        tot += c;
        bef += k < static_cast<int>(blockIdx.x) ? c : 0u;
    }
    total[part][bk] = tot;
    before[part][bk] = bef;
    __syncthreads();
    if (threadIdx.x < 64) {
        base[bk] = total[0][bk] + total[1][bk] + total[2][bk] + total[3][bk];
        cursor[bk] = before[0][bk] + before[1][bk] + before[2][bk] + before[3][bk];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned acc = 0u;
        for (int b = 0; b < 64; ++b) {
            const unsigned n = base[b];
            base[b] = acc;
            acc += n;
        }
    }
    __syncthreads();
    const int64_t u = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (u >= tiles) return;
    const int b = bucket[u];
    order[base[b] + atomicAdd(&cursor[b], 1u)] = static_cast<int>(u);
}

inline int64_t tile_order_blocks(int64_t tiles) {
    return (tiles + kOrderThreads - 1) / kOrderThreads;
}

// Enqueue the edge-first order of src's tiles into the stream's workspace
// and return src with it (src unchanged for an empty grid).
template <class Flow>
int tile_order_edge_first(const Flow& f, const GridSource& src, hipStream_t s, Workspace& ws,
                          GridSource& out) {
    out = src;
    const int64_t tiles = src.slots() / 16;
    if (tiles == 0) return 0;
    NBX_REQUIRE(tiles < (int64_t(1) << 31), "too many particle tiles");
    if (ws.error()) return ws.error();
    const int64_t nb = tile_order_blocks(tiles);
    char* w = ws.get();
    unsigned* block_count = reinterpret_cast<unsigned*>(w);  // 64 per block
    int* bucket = reinterpret_cast<int*>(w + 256 * nb);
    int* order = bucket + tiles;
    k_tile_order_keys<<<static_cast<unsigned>(nb), kOrderThreads, 0, s>>>(f, src, tiles, bucket,
                                                                          block_count);
    NBX_LAUNCHED("tile_order_keys");
    k_tile_order_scatter<<<static_cast<unsigned>(nb), kOrderThreads, 0, s>>>(
        bucket, block_count, static_cast<int>(nb), tiles, order);
    NBX_LAUNCHED("tile_order_scatter");
    out.order = order;
    return 0;
}

inline size_t tile_order_bytes(const GridSource& src) {
    const int64_t tiles = src.slots() / 16;
    return 256 * static_cast<size_t>(tile_order_blocks(tiles)) +
           2 * sizeof(int) * static_cast<size_t>(tiles);
}

template <class R, class Src>
int dispatch_solve(const nbx_flow* fl, const double* params, int np, const Src& src,
                   const SolveArgs& a, int precision, hipStream_t s) {
    const LaunchCfg cfg = launch_cfg(fl->kind, precision);
    if (fl->kind == NBX_FLOW_SPLINE3) {
        // linear extrapolation: the kernel with the gradient path, one lane
        // per particle (the lane-group setting is not used for such flows)
        if (fl->extrap == 1)
            return launch_solve<Spline3<R, 1, true>, R, 1>(make_spline<R, true>(fl, params[0]),
                                                           src, a, cfg, s);
        const Spline3<R, 1> sp = make_spline<R, false>(fl, params[0]);
        if constexpr (std::is_same<Src, GridSource>::value) {
            if (cfg.persistent < 0) {  // LDS-staged coefficients, 4 lanes, one-wave blocks
                const int64_t slots = src.slots();
                if (slots == 0) return 0;
                k_flowmap_staged<R><<<blocks_for(slots * 4, 64), 64, 0, s>>>(
                    regroup<4, R, true>(sp), src, slots, a.s0, a.s1, a.rtol, a.atol, a.mask,
                    a.nmax, a.out, a.status, a.nsteps);
                NBX_LAUNCHED("flowmap_staged");
                return 0;
            }
        }
        Src run_src = src;
        std::unique_ptr<Workspace> order_ws;  // held until the launch is enqueued
        if constexpr (std::is_same<Src, GridSource>::value) {
            bool edge_first;
            {
                std::lock_guard<std::mutex> lock(g_cfg_mutex);
                edge_first = g_edge_first[precision == NBX_FP32_DISP ? 1 : 0] != 0;
            }
            if (edge_first && cfg.persistent == 0) {
                order_ws = std::make_unique<Workspace>(s, 4, tile_order_bytes(src));
                if (int rc = tile_order_edge_first(sp, src, s, *order_ws, run_src)) return rc;
            }
        }
        if (cfg.lanes == 4) {
            NBX_REQUIRE(sp.cbytes != 0, "the 4-lane spline kernel needs a coefficient array "
                                        "under 4 GiB (set 1 or 2 lanes per particle)");
            return launch_solve<Spline3<R, 4>, R, 4>(regroup<4>(sp), run_src, a, cfg, s);
        }
        if (cfg.lanes == 2)
            return launch_solve<Spline3<R, 2>, R, 2>(regroup<2>(sp), run_src, a, cfg, s);
        return launch_solve<Spline3<R, 1>, R, 1>(sp, run_src, a, cfg, s);
    }
    // (the auxiliary grid's one-lane kernels of these flows contract a few
    // operations differently from the grid's: they stay, for the same results)
    int64_t slots = a.P;
    if constexpr (std::is_same<Src, GridSource>::value) slots = src.slots();
    const bool pair = !std::is_same<Src, AuxSource>::value && pair_lanes<R>(fl, a.P, slots);
    if (fl->kind == NBX_FLOW_LINEAR3)
        return pair ? launch_solve<Linear3Pair<R>, R, 2>(
                          pair_linear(make_linear<R>(fl, params[0])), src, a, cfg, s)
                    : launch_solve<Linear3<R>, R, 1>(make_linear<R>(fl, params[0]), src, a, cfg,
                                                     s);
    if (fl->kind == NBX_FLOW_DOUBLE_GYRE) {
        NBX_REQUIRE(np >= 6, "double_gyre needs 6 parameters [dir, A, eps, alpha, omega, psi]");
        const DoubleGyre<R> dg{params[0], params[1], params[2], params[3], params[4], params[5]};
        if (pair)
            return launch_solve<DoubleGyrePair<R>, R, 2>(DoubleGyrePair<R>{dg}, src, a, cfg, s);
        return launch_solve<DoubleGyre<R>, R, 1>(dg, src, a, cfg, s);
    }
    if (fl->kind == NBX_FLOW_BICKLEY_JET) {
        NBX_REQUIRE(np >= 12, "bickley_jet needs 12 parameters");
        BickleyJet<R> bj;
        for (int k = 0; k < 12; ++k) bj.p[k] = params[k];
        return launch_solve<BickleyJet<R>, R, 1>(bj, src, a, cfg, s);
    }
    set_error("unknown flow kind");
    return -2;
}

template <class Src>
int solve(const nbx_flow* fl, const double* params, int np, const Src& src, const SolveArgs& a,
          int precision, hipStream_t s) {
    if (precision == NBX_FP32_DISP) return dispatch_solve<float>(fl, params, np, src, a, precision, s);
    return dispatch_solve<double>(fl, params, np, src, a, precision, s);
}

}  // namespace nbx

using namespace nbx;

extern "C" {

const char* nbx_last_error(void) { return nbx::g_last_error.c_str(); }

int nbx_version(void) { return 1; }

int nbx_flow_create_analytic(int kind, nbx_flow** out) {
    NBX_REQUIRE(out != nullptr, "out is NULL");
    NBX_REQUIRE(kind == NBX_FLOW_DOUBLE_GYRE || kind == NBX_FLOW_BICKLEY_JET,
                "unknown analytic flow kind");
    nbx_flow* fl = new nbx_flow();
    fl->kind = kind;
    *out = fl;
    return 0;
}

int nbx_flow_create_spline3(const double* grid9_host, const double* Cu, const double* Cv,
                            int spherical, int extrap, double r, nbx_flow** out,
                            nbx_stream stream) {
    NBX_REQUIRE(out != nullptr && grid9_host != nullptr && Cu != nullptr && Cv != nullptr,
                "NULL argument");
    NBX_REQUIRE(spherical >= 0 && spherical <= 2, "spherical must be 0, 1 or 2");
    NBX_REQUIRE(extrap >= 0 && extrap <= 2, "unknown extrapolation mode");
    int n[3];
    for (int d = 0; d < 3; ++d) {
        n[d] = static_cast<int>(grid9_host[3 * d + 2]);
        NBX_REQUIRE(n[d] >= 2 && n[d] == grid9_host[3 * d + 2],
                    "spline grids need at least 2 points per axis");
        NBX_REQUIRE(grid9_host[3 * d + 1] > grid9_host[3 * d], "grid axes must be ascending");
    }
    const int64_t ncoef = static_cast<int64_t>(n[0] + 2) * (n[1] + 2) * (n[2] + 2);
    nbx_flow* fl = new nbx_flow();
    fl->kind = NBX_FLOW_SPLINE3;
    std::memcpy(fl->grid9, grid9_host, sizeof(fl->grid9));
    fl->spherical = spherical;
    fl->extrap = extrap;
    fl->r = r;
    fl->ncoef = ncoef;
    if (flow_register(fl) != 0 || !flow_array(fl, &fl->coef, &fl->coef_bytes) ||
        !flow_array(fl, &fl->coef32, &fl->coef32_bytes)) {
        nbx_flow_destroy(fl);
        set_error("hipMalloc of spline coefficients failed");
        return -1;
    }
    hipStream_t s = as_stream(stream);
    k_interleave<<<blocks_for(ncoef, 256) < 4096 ? blocks_for(ncoef, 256) : 4096, 256, 0, s>>>(
        Cu, Cv, ncoef, static_cast<int64_t>(n[1] + 2) * (n[2] + 2), fl->coef, fl->coef32);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        nbx_flow_destroy(fl);
        set_error(std::string("interleave launch: ") + hipGetErrorString(e));
        return -1;
    }
    *out = fl;
    return 0;
}

int nbx_flow_create_linear3(const double* grid9_host, const double* U, const double* V,
                            int spherical, int extrap, double r, nbx_flow** out,
                            nbx_stream stream) {
    NBX_REQUIRE(out != nullptr && grid9_host != nullptr && U != nullptr && V != nullptr,
                "NULL argument");
    NBX_REQUIRE(spherical >= 0 && spherical <= 2, "spherical must be 0, 1 or 2");
    NBX_REQUIRE(extrap >= 0 && extrap <= 2, "unknown extrapolation mode");
    int n[3];
    for (int d = 0; d < 3; ++d) {
        n[d] = static_cast<int>(grid9_host[3 * d + 2]);
        NBX_REQUIRE(n[d] >= 2 && n[d] == grid9_host[3 * d + 2],
                    "trilinear grids need at least 2 points per axis");
        NBX_REQUIRE(grid9_host[3 * d + 1] > grid9_host[3 * d], "grid axes must be ascending");
    }
    const int64_t nval = static_cast<int64_t>(n[0]) * n[1] * n[2];
    nbx_flow* fl = new nbx_flow();
    fl->kind = NBX_FLOW_LINEAR3;
    std::memcpy(fl->grid9, grid9_host, sizeof(fl->grid9));
    fl->spherical = spherical;
    fl->extrap = extrap;
    fl->r = r;
    fl->ncoef = nval;
    if (flow_register(fl) != 0 || !flow_array(fl, &fl->coef, &fl->coef_bytes)) {
        nbx_flow_destroy(fl);
        set_error("hipMalloc of velocity samples failed");
        return -1;
    }
    hipStream_t s = as_stream(stream);
    k_interleave<<<blocks_for(nval, 256) < 4096 ? blocks_for(nval, 256) : 4096, 256, 0, s>>>(
        U, V, nval, 0, fl->coef, nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        nbx_flow_destroy(fl);
        set_error(std::string("interleave launch: ") + hipGetErrorString(e));
        return -1;
    }
    *out = fl;
    return 0;
}

int nbx_ingest_xy(const double* U_xy, int nt, int ny, int nx, double scale, double* U_ij,
                  nbx_stream stream) {
    NBX_REQUIRE(nt >= 0 && ny >= 0 && nx >= 0, "negative size");
    const int64_t n = static_cast<int64_t>(nt) * ny * nx;
    if (n == 0) return 0;
    NBX_REQUIRE(U_xy != nullptr && U_ij != nullptr && U_xy != U_ij, "NULL or aliased array");
    const unsigned tiles_x = static_cast<unsigned>((nx + kIngestTile - 1) / kIngestTile);
    const int64_t tiles_ty = static_cast<int64_t>(nt) * ((ny + kIngestTile - 1) / kIngestTile);
    // the dispatch's y extent in work-items (tiles x 8 rows) must fit 32 bits
    NBX_REQUIRE(tiles_ty * kIngestRows <= 4294967295LL, "too many time slices for one launch");
    k_ingest_xy<<<dim3(tiles_x, static_cast<unsigned>(tiles_ty)), dim3(kIngestTile, kIngestRows),
                  0, as_stream(stream)>>>(U_xy, nt, ny, nx, scale, U_ij);
    NBX_LAUNCHED("ingest_xy");
    return 0;
}

void nbx_flow_destroy(nbx_flow* fl) {
    if (!fl) return;
    if (fl->dev >= 0) flow_release(fl);
    delete fl;
}

int nbx_release_memory(void) {
    int dev = 0;
    NBX_HIP(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        (void)g_blocks[dev].give_back();
    }
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    for (auto& w : g_ws) {
        if (std::get<0>(w.first) != dev || std::get<2>(w.first) != kDefaultQueueSlot) continue;
        const std::unique_lock<std::mutex> unused(w.second->m, std::try_to_lock);
        if (!unused.owns_lock() || w.second->ptr == nullptr) continue;
        (void)hipFree(w.second->ptr);  // (waits for the device work that uses it)
        w.second->ptr = nullptr;
        w.second->bytes = 0;
    }
    return 0;
}

int nbx_flow_eval(const nbx_flow* fl, const double* params, int np, const double* t,
                  const double* pts, int64_t n, double* out, nbx_stream stream) {
    NBX_REQUIRE(fl != nullptr && params != nullptr && np >= 1, "flow and params are required");
    if (n == 0) return 0;
    NBX_REQUIRE(t != nullptr && pts != nullptr && out != nullptr, "NULL array");
    hipStream_t s = as_stream(stream);
    const auto* P = reinterpret_cast<const double2*>(pts);
    auto* O = reinterpret_cast<double2*>(out);
    const unsigned nb = blocks_for(n, 256);
    if (fl->kind == NBX_FLOW_SPLINE3) {
        k_flow_eval<Spline3<double, 1, true>, double><<<nb, 256, 0, s>>>(
            make_spline<double, true>(fl, params[0]), t, P, n, O);
    } else if (fl->kind == NBX_FLOW_LINEAR3) {
        k_flow_eval<Linear3<double>, double><<<nb, 256, 0, s>>>(
            make_linear<double>(fl, params[0]), t, P, n, O);
    } else if (fl->kind == NBX_FLOW_DOUBLE_GYRE) {
        NBX_REQUIRE(np >= 6, "double_gyre needs 6 parameters");
        const DoubleGyre<double> dg{params[0], params[1], params[2], params[3], params[4], params[5]};
        k_flow_eval<DoubleGyre<double>, double><<<nb, 256, 0, s>>>(dg, t, P, n, O);
    } else {
        NBX_REQUIRE(np >= 12, "bickley_jet needs 12 parameters");
        BickleyJet<double> bj;
        for (int k = 0; k < 12; ++k) bj.p[k] = params[k];
        k_flow_eval<BickleyJet<double>, double><<<nb, 256, 0, s>>>(bj, t, P, n, O);
    }
    NBX_LAUNCHED("flow_eval");
    return 0;
}

static int check_solve_args(const nbx_flow* fl, const double* params, int np, double rtol,
                            double atol, int64_t max_steps, int precision) {
    NBX_REQUIRE(fl != nullptr, "flow handle is NULL");
    NBX_REQUIRE(params != nullptr && np >= 1, "params must hold at least the direction");
    NBX_REQUIRE(rtol > 0 && atol >= 0, "tolerances must be positive");
    NBX_REQUIRE(max_steps >= 1, "max_steps must be >= 1");
    NBX_REQUIRE(precision == NBX_FP64 || precision == NBX_FP32_DISP, "unknown precision");
    return 0;
}

int nbx_flowmap_grid_2d(const nbx_flow* fl, double t0, double T, const double* x, int nx,
                        const double* y, int ny, const double* params, int np, double rtol,
                        double atol, const uint8_t* mask, int64_t max_steps, int precision,
                        double* out, int32_t* status, int32_t* nsteps, nbx_stream stream) {
    if (int rc = check_solve_args(fl, params, np, rtol, atol, max_steps, precision)) return rc;
    NBX_REQUIRE(nx >= 0 && ny >= 0, "negative grid size");
    const int64_t P = static_cast<int64_t>(nx) * ny;
    if (P == 0) return 0;
    NBX_REQUIRE(x != nullptr && y != nullptr && out != nullptr, "NULL array");
    SolveArgs a{P, params[0] * t0, params[0] * (t0 + T), rtol, atol, mask, max_steps,
                reinterpret_cast<double2*>(out), status, nsteps};
    return solve(fl, params, np, GridSource{x, y, ny, nx}, a, precision, as_stream(stream));
}

int nbx_flowmap_aux_grid_2d(const nbx_flow* fl, double t0, double T, const double* x, int nx,
                            const double* y, int ny, double h, int eig_main, int compute_edge,
                            const double* params, int np, double rtol, double atol,
                            const uint8_t* mask, int64_t max_steps, int precision, double* out,
                            int32_t* status, int32_t* nsteps, nbx_stream stream) {
    if (int rc = check_solve_args(fl, params, np, rtol, atol, max_steps, precision)) return rc;
    NBX_REQUIRE(nx >= 0 && ny >= 0, "negative grid size");
    const int naux = eig_main ? 5 : 4;
    const int64_t P = static_cast<int64_t>(nx) * ny * naux;
    if (P == 0) return 0;
    NBX_REQUIRE(x != nullptr && y != nullptr && out != nullptr, "NULL array");
    SolveArgs a{P, params[0] * t0, params[0] * (t0 + T), rtol, atol, mask, max_steps,
                reinterpret_cast<double2*>(out), status, nsteps};
    const AuxSource src{x, y, nx, ny, naux, h, eig_main != 0, compute_edge != 0};
    return solve(fl, params, np, src, a, precision, as_stream(stream));
}

int nbx_flowmap_pts(const nbx_flow* fl, double t0, double T, const double* pts, int64_t npts,
                    const double* params, int np, double rtol, double atol, const uint8_t* mask,
                    int64_t max_steps, int precision, double* out, int32_t* status,
                    int32_t* nsteps, nbx_stream stream) {
    if (int rc = check_solve_args(fl, params, np, rtol, atol, max_steps, precision)) return rc;
    NBX_REQUIRE(npts >= 0, "negative point count");
    if (npts == 0) return 0;
    NBX_REQUIRE(pts != nullptr && out != nullptr, "NULL array");
    SolveArgs a{npts, params[0] * t0, params[0] * (t0 + T), rtol, atol, mask, max_steps,
                reinterpret_cast<double2*>(out), status, nsteps};
    return solve(fl, params, np, PointSource{reinterpret_cast<const double2*>(pts)}, a, precision,
                 as_stream(stream));
}

int nbx_set_launch_config(int kind, int precision, int lanes_per_particle, int block_threads,
                          int persistent_blocks_per_cu) {
    NBX_REQUIRE(kind >= 0 && kind <= 3, "unknown flow kind");
    NBX_REQUIRE(precision == NBX_FP64 || precision == NBX_FP32_DISP, "unknown precision");
    NBX_REQUIRE(lanes_per_particle == 1 || lanes_per_particle == 2 || lanes_per_particle == 4,
                "lanes_per_particle must be 1, 2 or 4");
    NBX_REQUIRE(block_threads == 64 || block_threads == 128 || block_threads == 256,
                "block_threads must be 64, 128 or 256");
    NBX_REQUIRE(kind == NBX_FLOW_SPLINE3 || lanes_per_particle == 1,
                "analytic flows run one lane per particle");
    NBX_REQUIRE(persistent_blocks_per_cu >= -1 && persistent_blocks_per_cu <= 64,
                "persistent_blocks_per_cu must be in [-1, 64]");
    NBX_REQUIRE(persistent_blocks_per_cu != -1 ||
                    (kind == NBX_FLOW_SPLINE3 && lanes_per_particle == 4 && block_threads == 64),
                "the LDS-staged launch (-1) is for spline flows at 4 lanes, 64-thread blocks");
    const LaunchCfg& d = kDefaultCfg[kind][precision];
    const bool requested = lanes_per_particle != d.lanes || block_threads != d.block ||
                           persistent_blocks_per_cu != d.persistent;
    std::lock_guard<std::mutex> lock(g_cfg_mutex);
    g_cfg[kind][precision] =
        LaunchCfg{lanes_per_particle, block_threads, persistent_blocks_per_cu, requested};
    return 0;
}

int nbx_set_tile_order(int precision, int edge_first) {
    NBX_REQUIRE(precision == NBX_FP64 || precision == NBX_FP32_DISP, "unknown precision");
    NBX_REQUIRE(edge_first == 0 || edge_first == 1, "edge_first must be 0 or 1");
    std::lock_guard<std::mutex> lock(g_cfg_mutex);
    g_edge_first[precision == NBX_FP32_DISP ? 1 : 0] = edge_first;
    return 0;
}

int nbx_get_tile_order(int precision, int* edge_first) {
    NBX_REQUIRE(precision == NBX_FP64 || precision == NBX_FP32_DISP, "unknown precision");
    NBX_REQUIRE(edge_first != nullptr, "NULL output");
    std::lock_guard<std::mutex> lock(g_cfg_mutex);
    *edge_first = g_edge_first[precision == NBX_FP32_DISP ? 1 : 0];
    return 0;
}

int nbx_get_launch_config(int kind, int precision, int* lanes_per_particle, int* block_threads,
                          int* persistent_blocks_per_cu) {
    NBX_REQUIRE(kind >= 0 && kind <= 3, "unknown flow kind");
    NBX_REQUIRE(precision == NBX_FP64 || precision == NBX_FP32_DISP, "unknown precision");
    NBX_REQUIRE(lanes_per_particle != nullptr && block_threads != nullptr &&
                    persistent_blocks_per_cu != nullptr,
                "NULL output");
    const LaunchCfg c = launch_cfg(kind, precision);
    *lanes_per_particle = c.lanes;
    *block_threads = c.block;
    *persistent_blocks_per_cu = c.persistent;
    return 0;
}

}  // extern "C"
