// Device velocity fields ("flows").  Each flow is a small trivially-copyable
// functor passed by value in the kernel arguments and inlined into the
// integrator; it evaluates dy = p0 * v(p0 * t, y), the sign-flipped
// right-hand side convention of the reference (params[0] = integration
// direction, flows.py:1146-1158, docs userguide.rst:216-227).
//
// Call form: f(t, px, py, f0, f1) with time and position in double and the
// velocity returned in the stage precision R of the integrator.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "lanes.h"

namespace nbx {

constexpr double kPi = 3.141592653589793;

// Double gyre, flows.py:1146-1158.  p = [dir, A, eps, alpha, omega, psi].
// The float form evaluates the same expression in float.
template <class R>
struct DoubleGyre {
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ void prepare_factors() {}
    double p0, A, eps, alpha, omega, psi;

    __device__ __forceinline__ void operator()(double t, double y0d, double y1d, R& f0,
                                               R& f1) const {
        if constexpr (sizeof(R) == sizeof(double)) {
            const double y0 = y0d, y1 = y1d;
            const double tt = p0 * t;
            const double a = eps * sin(omega * tt + psi);
            const double b = 1 - 2 * a;
            const double f = a * (y0 * y0) + b * y0;
            const double df = 2 * a * y0 + b;
            double sf, cf, sy, cy;
            sincos(kPi * f, &sf, &cf);
            sincos(kPi * y1, &sy, &cy);
            f0 = p0 * (-kPi * A * sf * cy - alpha * y0);
            f1 = p0 * (kPi * A * cf * sy * df - alpha * y1);
        } else {
            // time enters through sin(omega*tt + psi): keep that argument in
            // double, the rest in float
            const float y0 = static_cast<float>(y0d), y1 = static_cast<float>(y1d);
            const double tt = p0 * t;
            const float a = static_cast<float>(eps * sin(omega * tt + psi));
            const float b = 1.0f - 2.0f * a;
            const float f = a * (y0 * y0) + b * y0;
            const float df = 2.0f * a * y0 + b;
            const float pi = static_cast<float>(kPi);
            float sf, cf, sy, cy;
            sincosf(pi * f, &sf, &cf);
            sincosf(pi * y1, &sy, &cy);
            const float q0 = static_cast<float>(p0), qA = static_cast<float>(A),
                        qal = static_cast<float>(alpha);
            f0 = q0 * (-pi * qA * sf * cy - qal * y0);
            f1 = q0 * (pi * qA * cf * sy * df - qal * y1);
        }
    }
};

// The double gyre on a pair of lanes (x in the even one, y in the odd one):
// the even lane takes sin and cos of pi f, the odd lane of pi y, and each lane
// the time factor eps sin(omega t + psi) of every other stage, so a lane runs
// one and a half library calls an evaluation instead of three.  By the
// operations of DoubleGyre.
template <class R>
struct DoubleGyrePair {
    static constexpr bool kStagesInLds = false;
    static constexpr bool kFusedC2 = true;
    DoubleGyre<R> g;
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ void prepare_factors() {}

    using Time = R;
    __device__ __forceinline__ R time_of(double t) const {
        const double tt = g.p0 * t;
        return static_cast<R>(g.eps * sin(g.omega * tt + g.psi));
    }
    __device__ __forceinline__ void times_of(double ta, double tb, R& a, R& b) const {
        const R v = time_of((__lane_id() & 1) ? tb : ta);
        a = quad_move<kPairEven>(v);
        b = quad_move<kPairOdd>(v);
    }

    // the lane's component but for the direction's factor
    template <class Ahead>
    __device__ __forceinline__ R undirected(R a, double yc, Ahead&& ahead) const {
        const bool odd = __lane_id() & 1;
        const R y = static_cast<R>(yc), y0 = quad_move<kPairEven>(y);
        // (the contractions of DoubleGyre's expressions, written out)
        const R b = fma(a, R(-2), R(1));
        const R f = fma(a, y0 * y0, b * y0);
        const R df = fma(2 * a, y0, b);
        const R pi = static_cast<R>(kPi), A = static_cast<R>(g.A), alpha = static_cast<R>(g.alpha);
        ahead();
        R sn, cs;
        if constexpr (sizeof(R) == sizeof(double)) sincos(pi * (odd ? y : f), &sn, &cs);
        else sincosf(pi * (odd ? y : f), &sn, &cs);
        const R other = quad_move<kPairSwap>(cs);  // cos(pi y) in the even lane, cos(pi f) in the odd
        const R w = (odd ? pi * A * other : -pi * A) * sn;
        return fma(w, odd ? df : other, -(alpha * y));
    }
    template <class Ahead>
    __device__ __forceinline__ R component(R a, double yc, Ahead&& ahead) const {
        return static_cast<R>(g.p0) * undirected(a, yc, ahead);
    }
    // component - f0 as the solver's initial step contracts it
    __device__ __forceinline__ double component_change(R a, double yc, double f0) const {
        if constexpr (sizeof(R) == sizeof(double))
            return fma(g.p0, undirected(a, yc, [] {}), -f0);
        return static_cast<double>(component(a, yc, [] {})) - f0;
    }
};

// Bickley jet with three travelling modes, flows.py:1182-1213.
// p = [dir, U0, L, A1, A2, A3, k1, k2, k3, c1, c2, c3].
template <class R>
struct BickleyJet {
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ void prepare_factors() {}
    double p[12];

    __device__ __forceinline__ void operator()(double t, double y0, double y1, R& f0,
                                               R& f1) const {
        const double tt = p[0] * t;
        if constexpr (sizeof(R) == sizeof(double)) {
            const double Y = y1 / p[2];
            const double ch = cosh(Y);
            const double sech2 = 1 / (ch * ch);
            double s1, c1, s2, c2, s3, c3;
            sincos(p[6] * (y0 - p[9] * tt), &s1, &c1);
            sincos(p[7] * (y0 - p[10] * tt), &s2, &c2);
            sincos(p[8] * (y0 - p[11] * tt), &s3, &c3);
            f0 = p[0] * (p[1] * sech2 +
                         2 * p[1] * tanh(Y) * sech2 * (p[3] * c1 + p[4] * c2 + p[5] * c3));
            f1 = -p[0] * (p[1] * p[2] * sech2 *
                          (p[3] * p[6] * s1 + p[4] * p[7] * s2 + p[5] * p[8] * s3));
        } else {
            // phase arguments k (x - c t) reduced in double, the rest in float
            const float Y = static_cast<float>(y1 / p[2]);
            const float ch = coshf(Y);
            const float sech2 = 1.0f / (ch * ch);
            float s1, c1, s2, c2, s3, c3;
            sincosf(static_cast<float>(fmod(p[6] * (y0 - p[9] * tt), 2 * kPi)), &s1, &c1);
            sincosf(static_cast<float>(fmod(p[7] * (y0 - p[10] * tt), 2 * kPi)), &s2, &c2);
            sincosf(static_cast<float>(fmod(p[8] * (y0 - p[11] * tt), 2 * kPi)), &s3, &c3);
            const float q0 = static_cast<float>(p[0]), U0 = static_cast<float>(p[1]),
                        L = static_cast<float>(p[2]);
            const float A1 = static_cast<float>(p[3]), A2 = static_cast<float>(p[4]),
                        A3 = static_cast<float>(p[5]);
            const float K1 = static_cast<float>(p[6]), K2 = static_cast<float>(p[7]),
                        K3 = static_cast<float>(p[8]);
            f0 = q0 * (U0 * sech2 + 2.0f * U0 * tanhf(Y) * sech2 * (A1 * c1 + A2 * c2 + A3 * c3));
            f1 = -q0 * (U0 * L * sech2 * (A1 * K1 * s1 + A2 * K2 * s2 + A3 * K3 * s3));
        }
    }
};

// Uniform cubic B-spline basis at local coordinate s in [0, 1].
// The 1/6 scaling is a multiplication by the rounded reciprocal (within one
// rounding of the quotient), which spares twelve IEEE divisions per
// evaluation; the 1/2 of the derivative weights is exact either way.
template <class R>
__device__ __forceinline__ void bspline_weights(R s, R w[4]) {
    constexpr R sixth = R(1) / R(6);
    const R s2 = s * s, s3 = s2 * s, u = R(1) - s;
    w[0] = u * u * u * sixth;
    w[1] = (R(3) * s3 - R(6) * s2 + R(4)) * sixth;
    w[2] = (R(-3) * s3 + R(3) * s2 + R(3) * s + R(1)) * sixth;
    w[3] = s3 * sixth;
}

// The same weights times 6 (no scaling: the 4-lane gather applies the
// three axes' 1/6 once, as 1/216 on its y-weight)
template <class R>
__device__ __forceinline__ void bspline_weights6(R s, R w[4]) {
    const R s2 = s * s, s3 = s2 * s, u = R(1) - s;
    w[0] = u * u * u;
    w[1] = R(3) * s3 - R(6) * s2 + R(4);
    w[2] = R(-3) * s3 + R(3) * s2 + R(3) * s + R(1);
    w[3] = s3;
}

template <class R>
__device__ __forceinline__ void bspline_dweights(R s, R dw[4]) {
    const R s2 = s * s, u = R(1) - s;
    dw[0] = -u * u * R(0.5);
    dw[1] = (R(3) * s2 - R(4) * s) * R(0.5);
    dw[2] = (R(-3) * s2 + R(2) * s + R(1)) * R(0.5);
    dw[3] = s2 * R(0.5);
}

// w[i] for a lane-dependent i without dynamic register indexing
template <class R>
__device__ __forceinline__ R pick4(const R w[4], int i) {
    return i == 0 ? w[0] : (i == 1 ? w[1] : (i == 2 ? w[2] : w[3]));
}

// Python's float modulo (result takes the sign of the divisor).
__device__ __forceinline__ double py_mod(double a, double m) {
    // fmod(a, m) == a exactly when |a| < |m|: the library call only runs for
    // arguments a full period or more away
    double r = fabs(a) < fabs(m) ? a : fmod(a, m);
    if (r != 0.0) {
        if ((m < 0) != (r < 0)) r += m;
    } else {
        r = copysign(0.0, m);
    }
    return r;
}

// py_mod out of line, for arguments a period or more away
__device__ __attribute__((noinline)) static double py_mod_far(double a, double m) {
    return py_mod(a, m);
}

// py_mod(a, 360): within a period the sum needs no branch (a zero keeps the
// divisor's sign, as copysign gives it: -0.0 + 0.0 is +0.0)
__device__ __forceinline__ double wrap360(double a) {
    double r = a + (a < 0 ? 360.0 : 0.0);
    if (__builtin_expect(!(fabs(a) < 360.0), 0)) r = py_mod_far(a, 360.0);
    return r;
}

// Degrees to radians as the reference writes it, (deg * pi) / 180: the
// quotient by 180 is the product with the rounded reciprocal plus one FMA
// correction (Markstein), which is the correctly rounded quotient -- equal
// to the IEEE division on 2e8 sampled latitudes and random doubles -- at
// four instructions instead of a dozen for the division sequence.
__device__ __forceinline__ double deg_to_rad(double deg) {
    constexpr double inv180 = 1.0 / 180.0;
    const double a = deg * kPi;
    const double q = a * inv180;
    return fma(fma(-q, 180.0, a), inv180, q);
}

// Cosine of a latitude x in radians as sin(pi/2 - |x|): pi/2 in two parts
// (Cody-Waite) keeps the reduced argument u accurate to the last bits, and
// sin(u) for |u| <= pi/2 is its Taylor series to u^25 (truncation below
// 3e-23) by Horner in u^2: within 2.2e-16 relative of the exact cosine on
// all latitudes (5e7 samples against long-double cos; the library cosine
// agrees with it bit for bit on 71%), without the library's range reduction
// (the spherical RHS takes one cosine per evaluation; the library's took ~50
// instructions of it).  Valid for |x| <= pi; larger arguments (no latitude)
// take the library cosine.
// fma(a, b, c) for a coefficient c, taken as a scalar-register operand of
// v_fma_f64.  Written as fma(), the compiler picks v_fmac_f64, whose addend
// is also its destination, and first copies each 64-bit coefficient into
// vector registers: two extra vector instructions per Horner step.  The
// result is the same fused multiply-add.
__device__ __forceinline__ double fma_coef(double a, double b, double c) {
#if __HIP_DEVICE_COMPILE__
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
#else
    return fma(a, b, c);
#endif
}

// The library cosine, out of line: inlined into the flow-map kernels, its
// polynomial constants were held in 18 vector registers through the whole
// solve for a path that no latitude takes.
__device__ __attribute__((noinline)) static double cos_far(double x) { return cos(x); }

__device__ __forceinline__ double cos_lat(double x) {
    constexpr double pio2_hi = 1.5707963267948966;      // double nearest pi/2
    constexpr double pio2_lo = 6.123233995736766e-17;   // pi/2 - pio2_hi
    const double ax = fabs(x);
    const double u = (pio2_hi - ax) + pio2_lo;
    const double s = u * u;
    double p = 1.0 / 15511210043330985984000000.0;      // 1/25!
    p = fma_coef(p, s, -1.0 / 25852016738884976640000.0);    // -1/23!
    p = fma_coef(p, s, 1.0 / 51090942171709440000.0);        // 1/21!
    p = fma_coef(p, s, -1.0 / 121645100408832000.0);         // -1/19!
    p = fma_coef(p, s, 1.0 / 355687428096000.0);             // 1/17!
    p = fma_coef(p, s, -1.0 / 1307674368000.0);              // -1/15!
    p = fma_coef(p, s, 1.0 / 6227020800.0);                  // 1/13!
    p = fma_coef(p, s, -1.0 / 39916800.0);                   // -1/11!
    p = fma_coef(p, s, 1.0 / 362880.0);                      // 1/9!
    p = fma_coef(p, s, -1.0 / 5040.0);                       // -1/7!
    p = fma_coef(p, s, 1.0 / 120.0);                         // 1/5!
    p = fma_coef(p, s, -1.0 / 6.0);                          // -1/3!
    double r = fma(u * s, p, u);
    if (__builtin_expect(ax > 2 * pio2_hi, 0)) r = cos_far(x);
    return r;
}

// The float form's latitude cosine: the same reduction in float, Taylor to
// u^13 (truncation below 7e-10), within 1.3e-7 relative.
__device__ __forceinline__ float cos_lat(float x) {
    constexpr float pio2_hi = 1.57079637f;              // float nearest pi/2
    constexpr float pio2_lo = -4.37113900e-8f;          // pi/2 - pio2_hi
    const float ax = fabsf(x);
    if (ax > 2 * pio2_hi) return cosf(x);
    const float u = (pio2_hi - ax) + pio2_lo;
    const float s = u * u;
    float p = 1.0f / 6227020800.0f;                     // 1/13!
    p = fmaf(p, s, -1.0f / 39916800.0f);
    p = fmaf(p, s, 1.0f / 362880.0f);
    p = fmaf(p, s, -1.0f / 5040.0f);
    p = fmaf(p, s, 1.0f / 120.0f);
    p = fmaf(p, s, -1.0f / 6.0f);
    return fmaf(u * s, p, u);
}

// Coefficient storage element.  FP64: one (u, v) pair, so one gather serves
// both velocity components.  FP32: (u, v) at time index t and at t + 1 in one
// 16-byte element, so one gather serves two time slices of the stencil and a
// stencil is 8 rows of 4 elements instead of 16 rows (the gathers are bound
// by distinct cache lines, not bytes).
template <class R> struct CoefPair;
template <> struct CoefPair<double> { using type = double2; };
template <> struct CoefPair<float> { using type = float4; };

// Sums of u and of v over the G lanes of an aligned lane group, the sum of u
// left in the even lanes and that of v in the odd ones (a reduce-scatter of
// DPP quad permutations: each lane keeps the component it integrates and sends
// the other).  Every lane of a parity ends with the same bits: the additions
// are commutative pairwise, and each level combines the same two partial sums.
// The empty asm materialises u and v first: otherwise the compiler may fuse
// the multiply that produced them into the first add (fma(a, b, other lane's
// rounded a*b)), and the lanes of a group would then round differently and
// take different step-size decisions.
template <int G, class R>
__device__ __forceinline__ R group_component(R u, R v, bool odd) {
    asm volatile("" : "+v"(u));
    asm volatile("" : "+v"(v));
    R s = (odd ? v : u) + quad_move<kPairSwap>(odd ? u : v);
    if constexpr (G == 4) s += quad_move<kQuadCross>(s);
    return s;
}

// Tricubic natural B-spline velocity on a uniform (t, x, y) grid (the
// reference's get_flow_2D over interpolation.eval_spline, flows.py:121-258).
// C holds (nt+2, nx+2, ny+2) (u, v) pairs, y fastest.  R is the coefficient
// and evaluation precision (double for the plain path, float for the
// FP32-displacement form).  G lanes (1, 2 or 4, aligned in the wavefront)
// share one evaluation and combine partial sums with group_component:
//   G = 2: lane g gathers the t-slices a with a % 2 == g (whole 4-pair rows);
//   G = 4: lane g gathers y-coefficient g of all 16 rows, so one load
//          instruction covers one contiguous row per particle -- a third of
//          the distinct cache lines per instruction of the row-per-lane
//          forms, and the vector L1's tag rate (one line per clock) is what
//          bounds these gathers.
//
// Out-of-box queries: extrap 0 ("constant") is zero outside the grid box,
// the rule of the reference dependency's eval_linear (pinned by the
// reference's composition fixture) carried over to its spline evaluation
// (inferred: no reference test leaves the grid); extrap 2 ("nearest") clamps
// the query into the box per axis; extrap 1 ("linear") adds the gradient at
// the clamped point times the outward offset.  L says whether that gradient
// path is compiled in: it is the register-heaviest code of the functor, and
// kernels built without it (L = false) serve modes 0 and 2 with fewer
// registers (one lane per particle: FP64 142 instead of 250, FP32 192 instead
// of 238).

// A uniform double moved into a vector register pair.  The flow kernels hold
// the spline's box and spacing for their whole solve; in scalar registers
// (next to the solver's constants and the kernel's pointers) they spill to
// vector-register lanes and every evaluation reloads them one lane read at
// a time.  The copy cannot be folded back into the scalar value.
__device__ __forceinline__ double in_vgpr(double x) {
    double y;
    asm volatile("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
    return y;
}

// Bare minimum and maximum: fmin and fmax first quiet each operand whose
// origin the compiler cannot see (a v_max_f64 apiece).  Same values, NaN
// included: a quiet NaN yields the other operand.
__device__ __forceinline__ double raw_min(double a, double b) {
#if __HIP_DEVICE_COMPILE__
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmin(a, b);
#endif
}
__device__ __forceinline__ double raw_max(double a, double b) {
#if __HIP_DEVICE_COMPILE__
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmax(a, b);
#endif
}
__device__ __forceinline__ double clamped(double q, double lo, double hi) {
    return raw_min(raw_max(q, lo), hi);
}

// Byte offset of the element g past the key-th, in an array of up to 4 GiB: beyond
// 2 GiB only unsigned arithmetic holds it.
__host__ __device__ constexpr unsigned element_offset(double key, int g, unsigned size) {
    return (static_cast<unsigned>(key) + static_cast<unsigned>(g)) * size;
}
static_assert(element_offset((1 << 28) - 4, 3, 16) == 0xfffffff0u,
              "the last element below 4 GiB (a signed product overflows: no constant)");

// A box of coefficient elements copied to LDS by a one-wavefront block for
// the stencils of one DOP853 step (cells it0.., ix0.., iy0.. of the
// coefficient array, bt x bx x by elements, y fastest): a stencil whose 4 x 4
// x 4 elements all lie inside is read from LDS, any other from HBM/L2.
template <class P>
struct StageBox {
    const P* lds = nullptr;
    int it0 = 0, ix0 = 0, iy0 = 0, bt = 0, bx = 0, by = 0;
    bool on = false;
    __device__ __forceinline__ bool covers(int it, int ix, int iy) const {
        return on && static_cast<unsigned>(it - it0) <= static_cast<unsigned>(bt - 4) &&
               static_cast<unsigned>(ix - ix0) <= static_cast<unsigned>(bx - 4) &&
               static_cast<unsigned>(iy - iy0) <= static_cast<unsigned>(by - 4);
    }
};
struct NoStageBox {};

template <class R, int G = 1, bool L = false, bool S = false>
struct Spline3 {
    using P = typename CoefPair<R>::type;
    const P* __restrict__ C;
    // S (4-lane form only): stencils inside the step's LDS box are read there
    std::conditional_t<S, StageBox<P>, NoStageBox> box;
    double lo[3], hi[3], dinv[3];
    int nm2[3];   // n - 2 per axis: the largest cell index
    double nm2d[3], sxd, std_;  // nm2, sx and st as doubles (the held form's cells)
    int sx, st;   // strides (in pairs) of the x and t axes
    int spherical, extrap;
    double r;     // sphere radius (km) for spherical = 1, 2
    double p0;    // integration direction
    double kdeg;  // p0 * (180 / (pi r)): km/h -> degrees/h, set with p0 and r
    // 4-lane unstaged form: the lane's column of the last stencil it
    // gathered and that stencil's origin (element offset), so a query in
    // the same cell as the particle's previous one reads registers instead
    // of the cache hierarchy (the kernel's own copy of the functor holds it)
    static constexpr bool kReuse = (G == 4) && !S;
    // the FP64 form has no vector registers left for the solver's stages (at
    // three wavefronts per SIMD)
    static constexpr bool kStagesInLds = kReuse && sizeof(R) == sizeof(double);
    static constexpr bool kFusedC2 = false;
    static constexpr int kRows = sizeof(R) == sizeof(double) ? 16 : 8;
    mutable P cst[kReuse ? kRows : 1];
    mutable double ckey = -1;
    // bytes of C (the 4-lane form's buffer loads: under 4 GiB, checked by
    // the dispatcher)
    unsigned cbytes = 0;

    // at the start of a kernel, on its own copy of the functor
    __device__ __forceinline__ void prepare() {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = in_vgpr(lo[d]);
            hi[d] = in_vgpr(hi[d]);
            dinv[d] = in_vgpr(dinv[d]);
        }
        prepare_factors();
    }
    // the direction and the degree factor only (for kernels with no
    // vector registers to spare for the box)
    __device__ __forceinline__ void prepare_factors() {
        p0 = in_vgpr(p0);
        kdeg = in_vgpr(kdeg);
    }

    __device__ __forceinline__ void cell(int d, double q, int& i, R& s) const {
        const double u = (q - lo[d]) * dinv[d];
        int k = static_cast<int>(floor(u));
        k = k > nm2[d] ? nm2[d] : k;
        k = k < 0 ? 0 : k;
        i = k;
        s = static_cast<R>(u - k);
    }

    // position u in cells of coordinate d, clamped into the box (so u >= 0 and
    // truncation is floor), and its cell k as a whole double: no conversions
    // to and from integers
    __device__ __forceinline__ void locate(int d, double q, double& u, double& k) const {
        u = (q - lo[d]) * dinv[d];
        k = raw_min(trunc(u), nm2d[d]);
    }

    // kReuse: have the lane hold its y-column of the stencil at element `key`
    // (a whole double, below 2^28)
    __device__ __forceinline__ void hold(double key, bool skip) const {
        if (skip | (key == ckey)) return;
        ckey = key;
        // buffer loads: the lane's origin is the vector offset, each row's
        // offset a scalar one (no per-load address arithmetic, and no 64-bit
        // row pointers held in scalar registers)
        const int g = static_cast<int>(__lane_id() & 3);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<P*>(C), 0, static_cast<int>(cbytes), 0x00020000);
        // (time slices step the vector offset, x rows are the scalar offsets:
        // three live scalars, not sixteen)
        const unsigned vo = element_offset(key, g, sizeof(P));
        const unsigned tstep =
            (sizeof(R) == sizeof(double) ? 1u : 2u) * static_cast<unsigned>(st) * sizeof(P);
        const unsigned xstep = static_cast<unsigned>(sx) * sizeof(P);
#pragma unroll
        for (int a = 0; a < kRows / 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const auto raw = __builtin_amdgcn_raw_buffer_load_b128(rsrc, vo + a * tstep,
                                                                       b * xstep, 0);
                __builtin_memcpy(&cst[a * 4 + b], &raw, sizeof(P));
            }
    }

    // the lane's component of the stencil sum over the held column: the sums
    // of column_sums, the y-weight applied last
    __device__ __forceinline__ R held_sum(const double u[3], const double k[3], bool odd) const {
        R wt[4], wx[4], wy[4];
        bspline_weights6(static_cast<R>(u[0] - k[0]), wt);
        bspline_weights6(static_cast<R>(u[1] - k[1]), wx);
        bspline_weights6(static_cast<R>(u[2] - k[2]), wy);
        R au = 0, av = 0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            R ru = 0, rv = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                R cu, cv;
                if constexpr (sizeof(R) == sizeof(double)) {
                    const P e = cst[a * 4 + b];
                    cu = e.x;
                    cv = e.y;
                } else {
                    const P e = cst[(a >> 1) * 4 + b];
                    cu = (a & 1) ? e.z : e.x;
                    cv = (a & 1) ? e.w : e.y;
                }
                ru = fma(wx[b], cu, ru);
                rv = fma(wx[b], cv, rv);
            }
            au = fma(wt[a], ru, au);
            av = fma(wt[a], rv, av);
        }
        const R wc = pick4(wy, static_cast<int>(__lane_id() & 3)) * R(1.0 / 216.0);
        return group_component<G>(au * wc, av * wc, odd);
    }

    // (u, v) of stencil time slice a (0..3), x row b, y column c, relative
    // to the stencil origin base
    __device__ __forceinline__ void coef(const P* base, int a, int b, int c, R& u, R& v) const {
        if constexpr (sizeof(R) == sizeof(double)) {
            const P e = base[a * st + b * sx + c];
            u = e.x;
            v = e.y;
        } else {
            const P e = base[(a & ~1) * st + b * sx + c];
            u = (a & 1) ? e.z : e.x;
            v = (a & 1) ? e.w : e.y;
        }
    }

    // y-weighted sum of one stencil row (slice a, x row b)
    __device__ __forceinline__ void row_sum(const P* base, int a, int b, const R wy[4], R& ru,
                                            R& rv) const {
        R cu, cv;
        coef(base, a, b, 0, cu, cv);
        ru = wy[0] * cu;
        rv = wy[0] * cv;
#pragma unroll
        for (int c = 1; c < 4; ++c) {
            coef(base, a, b, c, cu, cv);
            ru = fma(wy[c], cu, ru);
            rv = fma(wy[c], cv, rv);
        }
    }

    // sum over the 4 x 4 (t, x) rows of one y-column starting at lbase (time
    // and x strides ts, xs in elements) weighted by wt, wx -- the 4-lane
    // gather of one lane, from HBM/L2 or from the LDS box
    __device__ __forceinline__ static void column_sums(const P* lbase, int ts, int xs,
                                                       const R wt[4], const R wx[4], R& au,
                                                       R& av) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            R ru = 0, rv = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                R cu, cv;
                if constexpr (sizeof(R) == sizeof(double)) {
                    const P e = lbase[a * ts + b * xs];
                    cu = e.x;
                    cv = e.y;
                } else {
                    const P e = lbase[(a & ~1) * ts + b * xs];
                    cu = (a & 1) ? e.z : e.x;
                    cv = (a & 1) ? e.w : e.y;
                }
                ru = fma(wx[b], cu, ru);
                rv = fma(wx[b], cv, rv);
            }
            au = fma(wt[a], ru, au);
            av = fma(wt[a], rv, av);
        }
    }

    // (u, v) at an in-box point; in a lane group the lane's own component
    // (u in even lanes, v in odd ones), as su
    __device__ __forceinline__ void eval_in(double qt, double qx, double qy, R& su,
                                            R& sv) const {
        int it, ix, iy;
        R s0, s1, s2;
        cell(0, qt, it, s0);
        cell(1, qx, ix, s1);
        cell(2, qy, iy, s2);
        R wt[4], wx[4], wy[4];
        if constexpr (G == 4) {
            bspline_weights6(s0, wt);
            bspline_weights6(s1, wx);
            bspline_weights6(s2, wy);
        } else {
            bspline_weights(s0, wt);
            bspline_weights(s1, wx);
            bspline_weights(s2, wy);
        }
        const P* base = C + (static_cast<long>(it) * st + static_cast<long>(ix) * sx + iy);
        // explicit fma: the accumulation order and rounding do not depend on
        // how the compiler contracts each kernel instantiation
        R au = 0, av = 0;
        if constexpr (G == 1) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    R ru, rv;
                    row_sum(base, a, b, wy, ru, rv);
                    const R wab = wt[a] * wx[b];
                    au = fma(wab, ru, au);
                    av = fma(wab, rv, av);
                }
            }
        } else if constexpr (G == 4) {
            // lane g of the group takes y-coefficient g of all 16 rows, so
            // the group's four lanes read each 4-pair row in one load; the
            // y-weight is applied last, once per lane
            const int g = static_cast<int>(__lane_id() & 3);
            bool staged = false;
            if constexpr (S) staged = box.covers(it, ix, iy);
            if (staged) {
                if constexpr (S) {
                    const P* lb = box.lds + ((it - box.it0) * box.bx + (ix - box.ix0)) * box.by +
                                  (iy - box.iy0) + g;
                    column_sums(lb, box.bx * box.by, box.by, wt, wx, au, av);
                }
            } else {
                column_sums(base + g, st, sx, wt, wx, au, av);
            }
            const R wc = pick4(wy, g) * R(1.0 / 216.0);
            au *= wc;
            av *= wc;
        } else {
            static_assert(G == 2, "lane groups of 1, 2 or 4");
            // lane g of the group takes the t-slices a = 2g, 2g+1 (one element
            // row pair in FP32): each lane reads whole 4-element rows
            const int g = static_cast<int>(__lane_id() & (G - 1));
#pragma unroll
            for (int aa = 0; aa < 2; ++aa) {
                const int a = 2 * g + aa;
                const R wa = pick4(wt, a);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    R ru, rv;
                    row_sum(base, a, b, wy, ru, rv);
                    const R wab = wa * wx[b];
                    au = fma(wab, ru, au);
                    av = fma(wab, rv, av);
                }
            }
        }
        if constexpr (G == 1) {
            su = au;
            sv = av;
        } else {
            su = group_component<G>(au, av, __lane_id() & 1);
            sv = 0;
        }
    }

    // value and gradient (d/dt, d/dx, d/dy) at an in-box point; every lane
    // of the group evaluates the whole stencil (rare: out-of-box queries
    // with linear extrapolation only)
    __device__ __forceinline__ void eval_grad(double qt, double qx, double qy, R& su, R& sv,
                              R g[3][2]) const {
        int it, ix, iy;
        R s0, s1, s2;
        cell(0, qt, it, s0);
        cell(1, qx, ix, s1);
        cell(2, qy, iy, s2);
        R wt[4], wx[4], wy[4], dt[4], dx[4], dy[4];
        bspline_weights(s0, wt);
        bspline_weights(s1, wx);
        bspline_weights(s2, wy);
        bspline_dweights(s0, dt);
        bspline_dweights(s1, dx);
        bspline_dweights(s2, dy);
        const P* base = C + (static_cast<long>(it) * st + static_cast<long>(ix) * sx + iy);
        R au = 0, av = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) g[d][0] = g[d][1] = 0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                R ru = 0, rv = 0, du = 0, dv = 0;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    R cu, cv;
                    coef(base, a, b, c, cu, cv);
                    ru += wy[c] * cu;
                    rv += wy[c] * cv;
                    du += dy[c] * cu;
                    dv += dy[c] * cv;
                }
                au += wt[a] * wx[b] * ru;
                av += wt[a] * wx[b] * rv;
                g[0][0] += dt[a] * wx[b] * ru;
                g[0][1] += dt[a] * wx[b] * rv;
                g[1][0] += wt[a] * dx[b] * ru;
                g[1][1] += wt[a] * dx[b] * rv;
                g[2][0] += wt[a] * wx[b] * du;
                g[2][1] += wt[a] * wx[b] * dv;
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            g[d][0] *= static_cast<R>(dinv[d]);
            g[d][1] *= static_cast<R>(dinv[d]);
        }
        su = au;
        sv = av;
    }

    __device__ __forceinline__ void eval(double qt, double qx, double qy, R& su, R& sv) const {
        const double ct = fmin(fmax(qt, lo[0]), hi[0]);
        const double cx = fmin(fmax(qx, lo[1]), hi[1]);
        const double cy = fmin(fmax(qy, lo[2]), hi[2]);
        const bool inside = (ct == qt) & (cx == qx) & (cy == qy);
        if (inside || extrap == 2) {
            eval_in(ct, cx, cy, su, sv);
        } else if (!L || extrap == 0) {
            // without the gradient path only modes 0 and 2 are dispatched
            su = 0;
            sv = 0;
        } else if constexpr (L) {
            R g[3][2];
            eval_grad(ct, cx, cy, su, sv, g);
            su += g[0][0] * static_cast<R>(qt - ct) + g[1][0] * static_cast<R>(qx - cx) +
                  g[2][0] * static_cast<R>(qy - cy);
            sv += g[0][1] * static_cast<R>(qt - ct) + g[1][1] * static_cast<R>(qx - cx) +
                  g[2][1] * static_cast<R>(qy - cy);
        }
    }

    // the x lookup coordinate of a position: the longitude wrapped into
    // [-180, 180) (spherical=1) or [0, 360) (spherical=2), else itself
    __device__ __forceinline__ double lookup_x(double y0) const {
        if (spherical == 1) return wrap360(y0 - 180) - 180;
        if (spherical != 0) return wrap360(y0);
        return y0;
    }

    // the latitude's cosine, in R
    __device__ __forceinline__ static R lat_cos(double y) {
        if constexpr (sizeof(R) == sizeof(double)) return cos_lat(deg_to_rad(y));
        else return cos_lat(static_cast<float>(y) * static_cast<float>(kPi / 180));
    }

    // What a lane of a group of 2 or 4 brings to its component of the
    // right-hand side at time t (yc: the lane's coordinate): the spline sum s
    // and the divisor of the degree conversion (one for the meridional
    // component, which is exact) with its reciprocal.  By the operations of
    // operator().  In the held form everything that does not need the
    // stencil -- the caller's `ahead`, the cosine, the reciprocal -- stands
    // between the gathers and the sums.
    struct Parts {
        R s, den;
        double recip;
    };
    template <class Ahead>
    __device__ __forceinline__ Parts parts(double t, double yc, Ahead&& ahead) const {
        static_assert(G > 1 && !L, "one lane holds both components");
        const bool odd = __lane_id() & 1;
        const double y1 = quad_move<kPairOdd>(yc);
        const double tt = p0 * t, xx = lookup_x(quad_move<kPairEven>(yc));
        Parts r;
        if constexpr (kReuse) {
            const double ct = clamped(tt, lo[0], hi[0]);
            const double cx = clamped(xx, lo[1], hi[1]);
            const double cy = clamped(y1, lo[2], hi[2]);
            const bool zero = extrap != 2 && !((ct == tt) & (cx == xx) & (cy == y1));
            double u[3], k[3];
            locate(0, ct, u[0], k[0]);
            locate(1, cx, u[1], k[1]);
            locate(2, cy, u[2], k[2]);
            hold(fma(k[0], std_, fma(k[1], sxd, k[2])), zero);
            ahead();
            if (spherical != 0) divide_by(odd, y1, r);
            // Outside the box the sums run on the held column and are dropped (a
            // divergent branch costs more than they do), but a wavefront with no
            // particle inside skips them: a launch of few steps ends with the
            // particles that cross the box's edge, in 25 to 57 steps that a
            // wavefront mostly takes alone (676 x 251 particles, one step but
            // for those: 240 -> 180 us; 72 time units 1.48 -> 1.45 ms).
            R v = 0;
            if (__ballot(!zero) != 0ull) v = held_sum(u, k, odd);
            r.s = zero ? R(0) : v;
        } else {
            R unused;
            eval(tt, xx, y1, r.s, unused);
            ahead();
            if (spherical != 0) divide_by(odd, y1, r);
        }
        return r;
    }
    __device__ __forceinline__ void divide_by(bool odd, double y1, Parts& r) const {
        const R c = lat_cos(y1);
        r.den = odd ? R(1) : c;
        if constexpr (sizeof(R) == sizeof(double)) r.recip = div_recip(r.den);
    }
    __device__ __forceinline__ R degrees(const Parts& r) const {
        if constexpr (sizeof(R) == sizeof(double)) return div_with(kdeg * r.s, r.den, r.recip);
        else return (static_cast<float>(kdeg) * r.s) / r.den;
    }

    // (a stage's time enters as it is)
    using Time = double;
    __device__ __forceinline__ double time_of(double t) const { return t; }
    __device__ __forceinline__ void times_of(double ta, double tb, double& a, double& b) const {
        a = ta;
        b = tb;
    }

    // the lane's component of the right-hand side
    template <class Ahead>
    __device__ __forceinline__ R component(double t, double yc, Ahead&& ahead) const {
        const Parts r = parts(t, yc, ahead);
        if (spherical == 0) return static_cast<R>(p0 * static_cast<double>(r.s));
        return degrees(r);
    }
    // component(t, yc) - f0, rounded as operator()'s result is where the
    // solver's initial step subtracts it in place (the meridional product
    // contracted with the subtraction)
    __device__ __forceinline__ double component_change(double t, double yc, double f0) const {
        const Parts r = parts(t, yc, [] {});
        if (spherical == 0) return static_cast<double>(static_cast<R>(p0 * static_cast<double>(r.s))) - f0;
        const double d = static_cast<double>(degrees(r)) - f0;
        if constexpr (sizeof(R) == sizeof(double))
            return (__lane_id() & 1) ? fma(kdeg, r.s, -f0) : d;
        return d;
    }

    __device__ __forceinline__ void operator()(double t, double y0, double y1, R& f0,
                                               R& f1) const {
        const double tt = p0 * t;
        // one inlined spline evaluation per call for every coordinate mode
        const double xx = lookup_x(y0);
        R su, sv;
        eval(tt, xx, y1, su, sv);
        if (spherical == 0) {
            f0 = static_cast<R>(p0 * static_cast<double>(su));
            f1 = static_cast<R>(p0 * static_cast<double>(sv));
        } else if constexpr (sizeof(R) == sizeof(double)) {
            // km/h -> degrees/h with one factor p0 * 180 / (pi r) per flow,
            // computed on the host (left to the device, the compiler
            // recomputed it, a division included, at every evaluation), so
            // the meridional component needs no division: within a few ulps
            // of dividing each by pi r
            f0 = (kdeg * su) / cos_lat(deg_to_rad(y1));
            f1 = kdeg * sv;
        } else {
            // the float form converts km/h to degrees/h in float too: the
            // velocity is already float, and the cosine of a float latitude
            // is good to ~1e-7, below the form's own rounding
            const float k = static_cast<float>(kdeg);
            f0 = (k * su) / cos_lat(static_cast<float>(y1) * static_cast<float>(kPi / 180));
            f1 = k * sv;
        }
    }
};

// Trilinear velocity on a uniform (t, x, y) grid (the reference's
// get_flow_linear_2D over interpolation.eval_linear, flows.py:418-506).
// V holds the (nt, nx, ny) samples as (u, v) pairs, y fastest.  Cell index
// floor((q - lo)/step) clamped to [0, n-2], weights q/step - index, the
// three linear stages in source order with contraction off.  Out-of-box
// queries: extrap 0 ("constant") is zero, pinned for eval_linear by the
// reference's composition fixture; 2 ("nearest") clamps the query into the
// box; 1 ("linear") continues the boundary cell's trilinear function.  The
// evaluation is FP64 in both precision forms (8 gathers of 16 B: not the
// bottleneck), rounded to R at the end.
template <class R>
struct Linear3 {
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ void prepare_factors() {}
    const double2* __restrict__ V;
    double lo[3], hi[3], step[3];
    int n[3];
    int sx, st;  // strides (in pairs) of the x and t axes
    int spherical, extrap;
    double r, p0;

    __device__ __forceinline__ void eval(double qt, double qx, double qy, double& su,
                                         double& sv) const {
#pragma clang fp contract(off)
        const double q[3] = {qt, qx, qy};
        bool out = false;
#pragma unroll
        for (int d = 0; d < 3; ++d) out |= (q[d] < lo[d]) | (q[d] > hi[d]);
        if (out && extrap == 0) {
            su = 0.0;
            sv = 0.0;
            return;
        }
        int i[3];
        double w[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double qq = extrap == 2 ? fmin(fmax(q[d], lo[d]), hi[d]) : q[d];
            const double u = (qq - lo[d]) / step[d];
            int k = static_cast<int>(floor(u));
            k = k > n[d] - 2 ? n[d] - 2 : k;
            k = k < 0 ? 0 : k;
            i[d] = k;
            w[d] = u - k;
        }
        const double2* c = V + (static_cast<long>(i[0]) * st + static_cast<long>(i[1]) * sx + i[2]);
        const double2 a00 = c[0], a01 = c[1], a10 = c[sx], a11 = c[sx + 1];
        const double2 b00 = c[st], b01 = c[st + 1], b10 = c[st + sx], b11 = c[st + sx + 1];
        const double w1 = w[1], w2 = w[2], w0 = w[0];
        const double bu0 = (1 - w1) * ((1 - w2) * a00.x + w2 * a01.x) + w1 * ((1 - w2) * a10.x + w2 * a11.x);
        const double bv0 = (1 - w1) * ((1 - w2) * a00.y + w2 * a01.y) + w1 * ((1 - w2) * a10.y + w2 * a11.y);
        const double bu1 = (1 - w1) * ((1 - w2) * b00.x + w2 * b01.x) + w1 * ((1 - w2) * b10.x + w2 * b11.x);
        const double bv1 = (1 - w1) * ((1 - w2) * b00.y + w2 * b01.y) + w1 * ((1 - w2) * b10.y + w2 * b11.y);
        su = (1 - w0) * bu0 + w0 * bu1;
        sv = (1 - w0) * bv0 + w0 * bv1;
    }

    __device__ __forceinline__ void operator()(double t, double y0, double y1, R& f0,
                                               R& f1) const {
        const double tt = p0 * t;
        double xx = y0;
        if (spherical == 1) xx = py_mod(y0 - 180, 360) - 180;
        else if (spherical != 0) xx = py_mod(y0, 360);
        double su, sv;
        eval(tt, xx, y1, su, sv);
        if (spherical == 0) {
            f0 = static_cast<R>(p0 * su);
            f1 = static_cast<R>(p0 * sv);
        } else {
            f0 = static_cast<R>(((p0 * su) * 180) / (kPi * r * cos_lat(deg_to_rad(y1))));
            f1 = static_cast<R>(((p0 * sv) * 180) / (kPi * r));
        }
    }
};

// The trilinear flow on a pair of lanes (x in the even one, y in the odd one):
// the even lane gathers and sums time slice it, the odd lane slice it + 1 (four
// samples each instead of eight), and each finishes its own component.  By the
// operations of Linear3, its three quotients by the grid steps taken with
// their reciprocals (div_with: an IEEE division's result, for offsets from the
// box's edge down to 2^-969).
template <class R>
struct Linear3Pair {
    static constexpr bool kStagesInLds = false;
    static constexpr bool kFusedC2 = false;
    Linear3<R> f;
    double rstep[3];  // 1 / step, correctly rounded
    // the lane's four samples of the cell it read last and that cell: a step
    // cut at a cell face makes most of its evaluations inside one cell
    mutable double2 held[4];
    mutable double hkey = -1;
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ void prepare_factors() {}

    using Time = double;
    __device__ __forceinline__ double time_of(double t) const { return t; }
    __device__ __forceinline__ void times_of(double ta, double tb, double& a, double& b) const {
        a = ta;
        b = tb;
    }

    template <class Ahead>
    __device__ __forceinline__ R component(double t, double yc, Ahead&& ahead) const {
#pragma clang fp contract(off)
        const bool odd = __lane_id() & 1;
        const double y1 = quad_move<kPairOdd>(yc);
        double xx = quad_move<kPairEven>(yc);
        if (f.spherical == 1) xx = wrap360(xx - 180) - 180;
        else if (f.spherical != 0) xx = wrap360(xx);
        const double q[3] = {f.p0 * t, xx, y1};
        bool out = false;
        double k[3], w[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            out |= (q[d] < f.lo[d]) | (q[d] > f.hi[d]);
            const double qq = f.extrap == 2 ? clamped(q[d], f.lo[d], f.hi[d]) : q[d];
            const double u = div_with(qq - f.lo[d], f.step[d], rstep[d]);
            k[d] = clamped(floor(u), 0.0, f.n[d] - 2);
            w[d] = u - k[d];
        }
        // (out-of-box points read the boundary cell and are dropped)
        const double key = fma(k[0], static_cast<double>(f.st),
                               fma(k[1], static_cast<double>(f.sx), k[2]));
        if (key != hkey) {
            hkey = key;
            const double2* c = f.V + (static_cast<unsigned>(key) + (odd ? f.st : 0));
            held[0] = c[0];
            held[1] = c[1];
            held[2] = c[f.sx];
            held[3] = c[f.sx + 1];
        }
        ahead();
        double den = 1.0, recip = 1.0;
        if (f.spherical != 0) {
            const double pr = kPi * f.r, cl = cos_lat(deg_to_rad(y1));
            den = odd ? pr : pr * cl;
            recip = div_recip(den);
        }
        const double2 a00 = held[0], a01 = held[1], a10 = held[2], a11 = held[3];
        const double w1 = w[1], w2 = w[2], w0 = w[0];
        const double bu = (1 - w1) * ((1 - w2) * a00.x + w2 * a01.x) + w1 * ((1 - w2) * a10.x + w2 * a11.x);
        const double bv = (1 - w1) * ((1 - w2) * a00.y + w2 * a01.y) + w1 * ((1 - w2) * a10.y + w2 * a11.y);
        const double got = quad_move<kPairSwap>(odd ? bu : bv);
        double s = (1 - w0) * (odd ? got : bu) + w0 * (odd ? bv : got);
        if (out && f.extrap == 0) s = 0.0;
        if (f.spherical == 0) return static_cast<R>(f.p0 * s);
        return static_cast<R>(div_with((f.p0 * s) * 180, den, recip));
    }
    __device__ __forceinline__ double component_change(double t, double yc, double f0) const {
        return static_cast<double>(component(t, yc, [] {})) - f0;
    }
};

}  // namespace nbx
