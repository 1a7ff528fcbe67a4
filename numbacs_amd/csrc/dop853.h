// DOP853 for a two-component state, one solve per GPU thread (or per group
// of G cooperating lanes, see flows.h), written as an init + step state
// machine so that a persistent kernel can refill finished lanes.
//
// Method: Dormand-Prince 8(5,3) as published by Hairer, Norsett & Wanner
// ("Solving Ordinary Differential Equations I", 2nd ed., sec. II.10), with
// the default step-size control of Hairer's dop853 code -- the integrator
// behind numbalsoda.dop853 (integration.py:169-171):
//   safety 0.9, fac1 0.333, fac2 6, beta 0, initial step from HINIT,
//   hmax = |xend - x|, last step clipped to xend, blended err5/err3 norm.
// Stiffness detection (every 1000 accepted steps) and dense output are not
// part of the flow-map path and are omitted.
//
// Precision forms (R = stage precision):
//   R = double: the state is the absolute position (anchor 0), every
//               operation in the order of Hairer's code;
//   R = float : the stored stages (velocities) and the velocity evaluation
//               (spline gathers and sums) are float; the position is a double
//               anchor, moved to each accepted point, plus the step's
//               displacement h * sum(b k) formed from the float stages; time,
//               step size, the stage sums, the error norm and the step-size
//               control stay double.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "lanes.h"

namespace nbx {
namespace dop {

constexpr double c2 = 0.526001519587677318785587544488e-01;
constexpr double c3 = 0.789002279381515978178381316732e-01;
constexpr double c4 = 0.118350341907227396726757197510e+00;
constexpr double c5 = 0.281649658092772603273242802490e+00;
constexpr double c6 = 0.333333333333333333333333333333e+00;
constexpr double c7 = 0.25e+00;
constexpr double c8 = 0.307692307692307692307692307692e+00;
constexpr double c9 = 0.651282051282051282051282051282e+00;
constexpr double c10 = 0.6e+00;
constexpr double c11 = 0.857142857142857142857142857142e+00;

constexpr double a21 = 5.26001519587677318785587544488e-2;
constexpr double a31 = 1.97250569845378994544595329183e-2;
constexpr double a32 = 5.91751709536136983633785987549e-2;
constexpr double a41 = 2.95875854768068491816892993775e-2;
constexpr double a43 = 8.87627564304205475450678981324e-2;
constexpr double a51 = 2.41365134159266685502369798665e-1;
constexpr double a53 = -8.84549479328286085344864962717e-1;
constexpr double a54 = 9.24834003261792003115737966543e-1;
constexpr double a61 = 3.7037037037037037037037037037e-2;
constexpr double a64 = 1.70828608729473871279604482173e-1;
constexpr double a65 = 1.25467687566822425016691814123e-1;
constexpr double a71 = 3.7109375e-2;
constexpr double a74 = 1.70252211019544039314978060272e-1;
constexpr double a75 = 6.02165389804559606850219397283e-2;
constexpr double a76 = -1.7578125e-2;
constexpr double a81 = 3.70920001185047927108779319836e-2;
constexpr double a84 = 1.70383925712239993810214054705e-1;
constexpr double a85 = 1.07262030446373284651809199168e-1;
constexpr double a86 = -1.53194377486244017527936158236e-2;
constexpr double a87 = 8.27378916381402288758473766002e-3;
constexpr double a91 = 6.24110958716075717114429577812e-1;
constexpr double a94 = -3.36089262944694129406857109825e+0;
constexpr double a95 = -8.68219346841726006818189891453e-1;
constexpr double a96 = 2.75920996994467083049415600797e+1;
constexpr double a97 = 2.01540675504778934086186788979e+1;
constexpr double a98 = -4.34898841810699588477366255144e+1;
constexpr double a101 = 4.77662536438264365890433908527e-1;
constexpr double a104 = -2.48811461997166764192642586468e+0;
constexpr double a105 = -5.90290826836842996371446475743e-1;
constexpr double a106 = 2.12300514481811942347288949897e+1;
constexpr double a107 = 1.52792336328824235832596922938e+1;
constexpr double a108 = -3.32882109689848629194453265587e+1;
constexpr double a109 = -2.03312017085086261358222928593e-2;
constexpr double a111 = -9.3714243008598732571704021658e-1;
constexpr double a114 = 5.18637242884406370830023853209e+0;
constexpr double a115 = 1.09143734899672957818500254654e+0;
constexpr double a116 = -8.14978701074692612513997267357e+0;
constexpr double a117 = -1.85200656599969598641566180701e+1;
constexpr double a118 = 2.27394870993505042818970056734e+1;
constexpr double a119 = 2.49360555267965238987089396762e+0;
constexpr double a1110 = -3.0467644718982195003823669022e+0;
constexpr double a121 = 2.27331014751653820792359768449e+0;
constexpr double a124 = -1.05344954667372501984066689879e+1;
constexpr double a125 = -2.00087205822486249909675718444e+0;
constexpr double a126 = -1.79589318631187989172765950534e+1;
constexpr double a127 = 2.79488845294199600508499808837e+1;
constexpr double a128 = -2.85899827713502369474065508674e+0;
constexpr double a129 = -8.87285693353062954433549289258e+0;
constexpr double a1210 = 1.23605671757943030647266201528e+1;
constexpr double a1211 = 6.43392746015763530355970484046e-1;

constexpr double b1 = 5.42937341165687622380535766363e-2;
constexpr double b6 = 4.45031289275240888144113950566e+0;
constexpr double b7 = 1.89151789931450038304281599044e+0;
constexpr double b8 = -5.8012039600105847814672114227e+0;
constexpr double b9 = 3.1116436695781989440891606237e-1;
constexpr double b10 = -1.52160949662516078556178806805e-1;
constexpr double b11 = 2.01365400804030348374776537501e-1;
constexpr double b12 = 4.47106157277725905176885569043e-2;

constexpr double bhh1 = 0.244094488188976377952755905512e+00;
constexpr double bhh2 = 0.733846688281611857341361741547e+00;
constexpr double bhh3 = 0.220588235294117647058823529412e-01;

constexpr double er1 = 0.1312004499419488073250102996e-01;
constexpr double er6 = -0.1225156446376204440720569753e+01;
constexpr double er7 = -0.4957589496572501915214079952e+00;
constexpr double er8 = 0.1664377182454986536961530415e+01;
constexpr double er9 = -0.3503288487499736816886487290e+00;
constexpr double er10 = 0.3341791187130174790297318841e+00;
constexpr double er11 = 0.8192320648511571246570742613e-01;
constexpr double er12 = -0.2235530786388629525884427845e-01;

constexpr double uround = 2.3e-16;
constexpr double safe = 0.9;
constexpr double facc1 = 1.0 / 0.333;
constexpr double facc2 = 1.0 / 6.0;
// x^(1/8) (x >= 0) for the step-size factor err^expo1, expo1 = 1/8, and the
// initial step's (0.01/der12)^(1/8): three correctly rounded square roots,
// within about one ulp of the exact root, as pow is.  pow's inlined log/exp
// polynomials kept ~37 VGPRs of hoisted constants live through the whole
// solve (4-lane FP64 spline kernel: 221 -> 184 VGPRs; 3-8% faster across the
// flow-map kernels).
__device__ __forceinline__ double root8(double x) { return sqrt(sqrt(sqrt(x))); }

}  // namespace dop

// Per-solve state.  Position = (ax, ay) + (dx, dy).
template <class R>
struct Dop853State {
    double x, xend, h, hmax, posneg, facold;
    double ax, ay;
    R dx, dy;
    R k1x, k1y;
    int nstep;
    bool last, reject;
    int idid;  // 0 while running; 1 ok, -2 step budget exhausted, -3 step underflow

    __device__ __forceinline__ double px() const { return ax + static_cast<double>(dx); }
    __device__ __forceinline__ double py() const { return ay + static_cast<double>(dy); }
};

// Start a solve at (x0, y0) from time x to xend: first derivative and the
// initial step (Hairer's HINIT, order 8).
template <class R, class Flow>
__device__ __forceinline__ void dop853_init(const Flow& f, Dop853State<R>& s, double x,
                                            double xend, double p0x, double p0y, double rtol,
                                            double atol) {
    s.x = x;
    s.xend = xend;
    s.posneg = (xend - x) >= 0 ? 1.0 : -1.0;
    s.hmax = fabs(xend - x);
    s.facold = 1.0e-4;
    s.last = false;
    s.reject = false;
    s.nstep = 0;
    s.idid = 0;
    if constexpr (sizeof(R) == sizeof(double)) {
        s.ax = 0.0;
        s.ay = 0.0;
        s.dx = p0x;
        s.dy = p0y;
    } else {
        s.ax = p0x;
        s.ay = p0y;
        s.dx = R(0);
        s.dy = R(0);
    }
    const double y0 = s.px(), y1 = s.py();
    f(x, y0, y1, s.k1x, s.k1y);
    const double f00 = static_cast<double>(s.k1x), f01 = static_cast<double>(s.k1y);
    const double sk0 = atol + rtol * fabs(y0);
    const double sk1 = atol + rtol * fabs(y1);
    const double dnf = (f00 / sk0) * (f00 / sk0) + (f01 / sk1) * (f01 / sk1);
    const double dny = (y0 / sk0) * (y0 / sk0) + (y1 / sk1) * (y1 / sk1);
    double h = (dnf <= 1.0e-10 || dny <= 1.0e-10) ? 1.0e-6 : sqrt(dny / dnf) * 0.01;
    h = fmin(h, s.hmax);
    h = s.posneg >= 0 ? fabs(h) : -fabs(h);
    R f10, f11;
    f(x + h, y0 + h * f00, y1 + h * f01, f10, f11);
    const double d0 = (static_cast<double>(f10) - f00) / sk0;
    const double d1 = (static_cast<double>(f11) - f01) / sk1;
    const double der2 = sqrt(d0 * d0 + d1 * d1) / h;
    const double der12 = fmax(fabs(der2), sqrt(dnf));
    const double h1 =
        der12 <= 1.0e-15 ? fmax(1.0e-6, fabs(h) * 1.0e-3) : dop::root8(0.01 / der12);
    h = fmin(fmin(100 * fabs(h), h1), s.hmax);
    s.h = s.posneg >= 0 ? h : -h;
}

// The head of one attempted step: the step budget and underflow checks and
// the clipping of the last step to xend.  Sets s.idid != 0 and returns false
// when the solve ends here; otherwise s.h is the step about to be taken.
template <class State>
__device__ __forceinline__ bool dop853_step_begin(State& s, long long nmax) {
    using namespace dop;
    if (s.nstep > nmax) {
        s.idid = -2;
        return false;
    }
    if (0.1 * fabs(s.h) <= fabs(s.x) * uround) {
        s.idid = -3;
        return false;
    }
    if ((s.x + 1.01 * s.h - s.xend) * s.posneg > 0.0) {
        s.h = s.xend - s.x;
        s.last = true;
    }
    return true;
}

// The stages, error estimate and step-size control of the attempted step
// that dop853_step_begin prepared.
template <class R, class Flow>
__device__ __forceinline__ bool dop853_step_body(const Flow& f, Dop853State<R>& s, double rtol,
                                                 double atol) {
    using namespace dop;
    ++s.nstep;
    const double x = s.x, h = s.h;
    // Stage sums in double for both forms: DOP853's coefficients are large
    // and cancel (|a98| = 43.5), so float sums would cost ~1e-6 relative per
    // stage, the size of the tolerance itself.  In the float form only the
    // stored stages, the stored displacement and the velocity evaluation are
    // float.
    auto D = [](R v) { return static_cast<double>(v); };
    const double ax = s.ax, ay = s.ay;
    const double y0 = ax + D(s.dx), y1 = ay + D(s.dy);  // = s.dx, s.dy exactly for double
    const double K1x = D(s.k1x), K1y = D(s.k1y);
    R k2x, k2y, k3x, k3y, k4x, k4y, k5x, k5y, k6x, k6y, k7x, k7y, k8x, k8y, k9x, k9y, k10x, k10y;
#define NBX_K(n) const double K##n##x = D(k##n##x), K##n##y = D(k##n##y)
    f(x + c2 * h, y0 + h * a21 * K1x, y1 + h * a21 * K1y, k2x, k2y);
    NBX_K(2);
    f(x + c3 * h, y0 + h * (a31 * K1x + a32 * K2x), y1 + h * (a31 * K1y + a32 * K2y), k3x, k3y);
    NBX_K(3);
    f(x + c4 * h, y0 + h * (a41 * K1x + a43 * K3x), y1 + h * (a41 * K1y + a43 * K3y), k4x, k4y);
    NBX_K(4);
    f(x + c5 * h, y0 + h * (a51 * K1x + a53 * K3x + a54 * K4x),
      y1 + h * (a51 * K1y + a53 * K3y + a54 * K4y), k5x, k5y);
    NBX_K(5);
    f(x + c6 * h, y0 + h * (a61 * K1x + a64 * K4x + a65 * K5x),
      y1 + h * (a61 * K1y + a64 * K4y + a65 * K5y), k6x, k6y);
    NBX_K(6);
    f(x + c7 * h, y0 + h * (a71 * K1x + a74 * K4x + a75 * K5x + a76 * K6x),
      y1 + h * (a71 * K1y + a74 * K4y + a75 * K5y + a76 * K6y), k7x, k7y);
    NBX_K(7);
    f(x + c8 * h, y0 + h * (a81 * K1x + a84 * K4x + a85 * K5x + a86 * K6x + a87 * K7x),
      y1 + h * (a81 * K1y + a84 * K4y + a85 * K5y + a86 * K6y + a87 * K7y), k8x, k8y);
    NBX_K(8);
    f(x + c9 * h,
      y0 + h * (a91 * K1x + a94 * K4x + a95 * K5x + a96 * K6x + a97 * K7x + a98 * K8x),
      y1 + h * (a91 * K1y + a94 * K4y + a95 * K5y + a96 * K6y + a97 * K7y + a98 * K8y), k9x,
      k9y);
    NBX_K(9);
    f(x + c10 * h,
      y0 + h * (a101 * K1x + a104 * K4x + a105 * K5x + a106 * K6x + a107 * K7x + a108 * K8x +
                a109 * K9x),
      y1 + h * (a101 * K1y + a104 * K4y + a105 * K5y + a106 * K6y + a107 * K7y + a108 * K8y +
                a109 * K9y),
      k10x, k10y);
    NBX_K(10);
    // stage 11 reuses k2, stage 12 reuses k3 (as in Hairer's code)
    f(x + c11 * h,
      y0 + h * (a111 * K1x + a114 * K4x + a115 * K5x + a116 * K6x + a117 * K7x + a118 * K8x +
                a119 * K9x + a1110 * K10x),
      y1 + h * (a111 * K1y + a114 * K4y + a115 * K5y + a116 * K6y + a117 * K7y + a118 * K8y +
                a119 * K9y + a1110 * K10y),
      k2x, k2y);
    const double L2x = D(k2x), L2y = D(k2y);
    const double xph = x + h;
    f(xph,
      y0 + h * (a121 * K1x + a124 * K4x + a125 * K5x + a126 * K6x + a127 * K7x + a128 * K8x +
                a129 * K9x + a1210 * K10x + a1211 * L2x),
      y1 + h * (a121 * K1y + a124 * K4y + a125 * K5y + a126 * K6y + a127 * K7y + a128 * K8y +
                a129 * K9y + a1210 * K10y + a1211 * L2y),
      k3x, k3y);
    const double L3x = D(k3x), L3y = D(k3y);
#undef NBX_K
    const double k4nx = b1 * K1x + b6 * K6x + b7 * K7x + b8 * K8x + b9 * K9x + b10 * K10x +
                        b11 * L2x + b12 * L3x;
    const double k4ny = b1 * K1y + b6 * K6y + b7 * K7y + b8 * K8y + b9 * K9y + b10 * K10y +
                        b11 * L2y + b12 * L3y;
    const double pnx = y0 + h * k4nx;
    const double pny = y1 + h * k4ny;
    // error estimate: blended 5th/3rd order norms
    const double skx = atol + rtol * fmax(fabs(y0), fabs(pnx));
    const double sky = atol + rtol * fmax(fabs(y1), fabs(pny));
    const double e2x = (k4nx - bhh1 * K1x - bhh2 * K9x - bhh3 * L3x) / skx;
    const double e2y = (k4ny - bhh1 * K1y - bhh2 * K9y - bhh3 * L3y) / sky;
    const double e5x = (er1 * K1x + er6 * K6x + er7 * K7x + er8 * K8x + er9 * K9x +
                        er10 * K10x + er11 * L2x + er12 * L3x) / skx;
    const double e5y = (er1 * K1y + er6 * K6y + er7 * K7y + er8 * K8y + er9 * K9y +
                        er10 * K10y + er11 * L2y + er12 * L3y) / sky;
    const double err2 = e2x * e2x + e2y * e2y;
    double err = e5x * e5x + e5y * e5y;
    double deno = err + 0.01 * err2;
    if (deno <= 0.0) deno = 1.0;
    err = fabs(h) * err * sqrt(1.0 / (2 * deno));
    const double fac11 = dop::root8(err);
    const double fac = fmax(facc2, fmin(facc1, fac11 / safe));
    double hnew = h / fac;
    if (err <= 1.0) {
        s.facold = fmax(err, 1.0e-4);
        // new state, then the derivative at the stored point.  The float
        // form moves its double anchor to the accepted position: a float
        // displacement from the initial point loses increments below its
        // resolution (~1e-7 of the distance travelled), and a particle whose
        // steps shrink at a velocity discontinuity (the grid edge under zero
        // extrapolation) would stop moving while time crawls on.
        if constexpr (sizeof(R) == sizeof(double)) {
            s.dx = pnx;
            s.dy = pny;
        } else {
            s.ax = pnx;
            s.ay = pny;
            s.dx = R(0);
            s.dy = R(0);
        }
        f(xph, s.px(), s.py(), s.k1x, s.k1y);
        s.x = xph;
        if (s.last) {
            s.idid = 1;
            return false;
        }
        if (fabs(hnew) > s.hmax) hnew = s.posneg * s.hmax;
        if (s.reject) hnew = s.posneg * fmin(fabs(hnew), fabs(h));
        s.reject = false;
    } else {
        hnew = h / fmin(facc1, fac11 / safe);
        s.reject = true;
        s.last = false;
    }
    s.h = hnew;
    return true;
}

// One attempted step (accepted or rejected).  Sets s.idid != 0 when the
// solve has ended; returns true while it is still running.
template <class R, class Flow>
__device__ __forceinline__ bool dop853_step(const Flow& f, Dop853State<R>& s, double rtol,
                                            double atol, long long nmax) {
    if (!dop853_step_begin(s, nmax)) return false;
    return dop853_step_body(f, s, rtol, atol);
}

// ---------------------------------------------------------------------------
// Component-per-lane form, for G = 2 or 4 lanes per particle: even lanes
// hold x, odd lanes y (a 4-lane group holds each component twice), so a stage
// sum is one chain of FMAs instead of two and a lane keeps ten stage values
// instead of twenty.  A lane's flow evaluation takes its own coordinate and
// returns its own velocity component; the functor exchanges what it needs
// inside the group (Flow::component).  The error norms combine the two
// components with one DPP exchange.  Every value is formed by the operations
// of dop853_step_body in their order and as the compiler contracts them there
// (written out as fma here: of each sum's first pair the second product is
// rounded, but in stage 11 the first), so the two forms agree bit for bit.

// x*x + y*y of a pair's components: the even lane forms fma(x, x, y*y), as
// the two-component form's contracted sum, and both lanes take its result
__device__ __forceinline__ double pair_sumsq(double e) {
    return quad_move<kPairEven>(fma(e, e, quad_move<kPairOdd>(e * e)));
}

// The step's error norm from a pair's scaled errors of third and fifth order
__device__ __forceinline__ double pair_norm(double e2, double e5, double h) {
    const double err2 = pair_sumsq(e2), err = pair_sumsq(e5);
    double deno = fma(0.01, err2, err);
    if (deno <= 0.0) deno = 1.0;
    return fabs(h) * err * sqrt(1.0 / (2 * deno));
}
// ... and from the errors by the divisions themselves, out of line
[[maybe_unused]] __device__ __attribute__((noinline)) static double pair_norm_far(double n2, double n5,
                                                                                 double sk,
                                                                                 double h) {
    return pair_norm(n2 / sk, n5 / sk, h);
}

template <class R>
struct Dop853Lane {
    double x, xend, h, hmax, posneg;
    double y;  // the lane's coordinate
    R k1;
    int nstep;
    bool last, reject;
    int idid;  // as Dop853State
};

template <class R, class Flow>
__device__ __forceinline__ void dop853_init(const Flow& f, Dop853Lane<R>& s, double x,
                                            double xend, double p0, double rtol, double atol) {
    s.x = x;
    s.xend = xend;
    s.posneg = (xend - x) >= 0 ? 1.0 : -1.0;
    s.hmax = fabs(xend - x);
    s.last = false;
    s.reject = false;
    s.nstep = 0;
    s.idid = 0;
    s.y = p0;
    s.k1 = f.component(f.time_of(x), p0, [] {});
    const double f0 = static_cast<double>(s.k1);
    const double sk = atol + rtol * fabs(p0);
    const double dnf = pair_sumsq(f0 / sk);
    const double dny = pair_sumsq(p0 / sk);
    double h = (dnf <= 1.0e-10 || dny <= 1.0e-10) ? 1.0e-6 : sqrt(dny / dnf) * 0.01;
    h = fmin(h, s.hmax);
    h = s.posneg >= 0 ? fabs(h) : -fabs(h);
    const double df = f.component_change(f.time_of(x + h), p0 + h * f0, f0);
    const double der2 = sqrt(pair_sumsq(df / sk)) / h;
    const double der12 = fmax(fabs(der2), sqrt(dnf));
    const double h1 =
        der12 <= 1.0e-15 ? fmax(1.0e-6, fabs(h) * 1.0e-3) : dop::root8(0.01 / der12);
    h = fmin(fmin(100 * fabs(h), h1), s.hmax);
    s.h = s.posneg >= 0 ? h : -h;
}

// Where a lane keeps its ten stage values (index 0..9: stages 1, 4..10, 11 and
// 12; stages 2 and 3 are used once, at once).
struct StageRegs {
    double k[10];
    __device__ __forceinline__ void put(int i, double v) { k[i] = v; }
    __device__ __forceinline__ double get(int i) const { return k[i]; }
};
// In LDS, 512 bytes a stage and wavefront (kStageLdsBytes a wavefront, the
// launch's dynamic LDS): each value is written once and read back where a sum
// needs it, so the 20 vector registers it would hold stay free.  volatile, or
// the compiler forwards the stores and keeps the registers.
constexpr unsigned kStageLdsBytes = 10 * 64 * sizeof(double);
extern __shared__ double stage_lds[];
struct StageLds {
    // (an LDS pointer: volatile accesses through a generic one stay flat)
    using Slot = __attribute__((address_space(3))) volatile double;
    Slot* at;
    __device__ __forceinline__ StageLds()
        : at((Slot*)stage_lds + (threadIdx.x >> 6) * 640 + (threadIdx.x & 63)) {}
    __device__ __forceinline__ void put(int i, double v) const { at[64 * i] = v; }
    __device__ __forceinline__ double get(int i) const { return at[64 * i]; }
};

__device__ __forceinline__ double unfused_add(double a, double b) {
#pragma clang fp contract(off)
    return a + b;
}

// A stage's evaluation and, in the time its gathers are in flight, the part
// of the next stage's sum that does not need it (`ahead`).
template <class R, class Stages, class Flow>
__device__ __forceinline__ bool dop853_step_body(const Flow& f, Dop853Lane<R>& s, Stages& ks,
                                                 double rtol, double atol) {
    using namespace dop;
    ++s.nstep;
    const double x = s.x, h = s.h, y = s.y;
    auto F = [&](typename Flow::Time t, double q, auto&& ahead) {
        return static_cast<double>(f.component(t, q, ahead));
    };
    auto none = [] {};
    double P;  // the next stage's sum but for its last term
    const double K1 = static_cast<double>(s.k1);
    ks.put(0, K1);
    typename Flow::Time ta, tb;  // of a pair of stages (a pair of lanes forms one each)
    // (c2 = a21: gridded flows' kernels form h a21 once and add it to x)
    const double ha = h * a21;
    f.times_of(Flow::kFusedC2 ? fma(c2, h, x) : unfused_add(x, ha), fma(c3, h, x), ta, tb);
    double K = F(ta, fma(ha, K1, y), none);
    K = F(tb, fma(h, fma(a31, K1, a32 * K), y), none);
    f.times_of(fma(c4, h, x), fma(c5, h, x), ta, tb);
    K = F(ta, fma(h, fma(a41, K1, a43 * K), y), [&, K3 = K] { P = fma(a51, K1, a53 * K3); });
    ks.put(1, K);
    K = F(tb, fma(h, fma(a54, K, P), y),
          [&] { P = fma(a61, ks.get(0), a64 * ks.get(1)); });
    ks.put(2, K);
    f.times_of(fma(c6, h, x), fma(c7, h, x), ta, tb);
    K = F(ta, fma(h, fma(a65, K, P), y),
          [&] { P = fma(a75, ks.get(2), fma(a71, ks.get(0), a74 * ks.get(1))); });
    ks.put(3, K);
    K = F(tb, fma(h, fma(a76, K, P), y), [&] {
        P = fma(a86, ks.get(3),
                fma(a85, ks.get(2), fma(a81, ks.get(0), a84 * ks.get(1))));
    });
    ks.put(4, K);
    f.times_of(fma(c8, h, x), fma(c9, h, x), ta, tb);
    K = F(ta, fma(h, fma(a87, K, P), y), [&] {
        P = fma(a97, ks.get(4),
                fma(a96, ks.get(3),
                    fma(a95, ks.get(2), fma(a91, ks.get(0), a94 * ks.get(1)))));
    });
    ks.put(5, K);
    K = F(tb, fma(h, fma(a98, K, P), y), [&] {
        P = fma(a108, ks.get(5),
                fma(a107, ks.get(4),
                    fma(a106, ks.get(3),
                        fma(a105, ks.get(2), fma(a101, ks.get(0), a104 * ks.get(1))))));
    });
    ks.put(6, K);
    f.times_of(fma(c10, h, x), fma(c11, h, x), ta, tb);
    K = F(ta, fma(h, fma(a109, K, P), y), [&] {
        P = fma(a119, ks.get(6),
                fma(a118, ks.get(5),
                    fma(a117, ks.get(4),
                        fma(a116, ks.get(3), fma(a115, ks.get(2), fma(a114, ks.get(1), a111 * ks.get(0)))))));
    });
    ks.put(7, K);
    K = F(tb, fma(h, fma(a1110, K, P), y), [&] {
        P = fma(a1210, ks.get(7),
                fma(a129, ks.get(6),
                    fma(a128, ks.get(5),
                        fma(a127, ks.get(4),
                            fma(a126, ks.get(3),
                                fma(a125, ks.get(2),
                                    fma(a121, ks.get(0), a124 * ks.get(1))))))));
    });
    ks.put(8, K);
    const double xph = x + h;
    const typename Flow::Time tn = f.time_of(xph);
    double B, E;  // the update's and the fifth-order error's sums but for the last term
    K = F(tn, fma(h, fma(a1211, K, P), y), [&] {
        const double k1 = ks.get(0), k6 = ks.get(3), k7 = ks.get(4), k8 = ks.get(5),
                     k9 = ks.get(6), k10 = ks.get(7), k11 = ks.get(8);
        B = fma(b11, k11,
                fma(b10, k10, fma(b9, k9, fma(b8, k8, fma(b7, k7, fma(b1, k1, b6 * k6))))));
        E = fma(er11, k11,
                fma(er10, k10,
                    fma(er9, k9, fma(er8, k8, fma(er7, k7, fma(er1, k1, er6 * k6))))));
    });
    const double k4n = fma(b12, K, B);
    const double pn = fma(h, k4n, y);
    const double sk = fma(rtol, fmax(fabs(y), fabs(pn)), atol);
    const double rsk = div_recip(sk);
    const double n2 = fma(-bhh3, K, fma(-bhh2, ks.get(6), fma(-bhh1, ks.get(0), k4n)));
    const double n5 = fma(er12, K, E);
    double err = pair_norm(div_with(n2, sk, rsk), div_with(n5, sk, rsk), h);
    // (no number: also where the scale is subnormal -- an absolute tolerance of
    // zero and a coordinate near zero -- and has no reciprocal)
    if (__builtin_expect(err != err, 0)) err = pair_norm_far(n2, n5, sk, h);
    const double fac = dop::root8(err) / safe;
    const bool accept = err <= 1.0;
    double hnew = h / (accept ? fmax(facc2, fmin(facc1, fac)) : fmin(facc1, fac));
    if (accept) {
        s.y = pn;
        s.k1 = f.component(tn, pn, none);
        s.x = xph;
        if (s.last) {
            s.idid = 1;
            return false;
        }
        if (fabs(hnew) > s.hmax) hnew = s.posneg * s.hmax;
        if (s.reject) hnew = s.posneg * fmin(fabs(hnew), fabs(h));
        s.reject = false;
    } else {
        s.reject = true;
        s.last = false;
    }
    s.h = hnew;
    return true;
}


// The solver of a group of G lanes, as the launches use it: one lane holds
// both components, two or four lanes one component each.
template <class Flow, class R, int G>
struct Solve {
    static constexpr int kStates = 2;  // states a group hands on (one per component)
    static constexpr unsigned kLdsBytes = Flow::kStagesInLds ? kStageLdsBytes : 0;  // a wavefront
    Dop853Lane<R> s;
    std::conditional_t<Flow::kStagesInLds, StageLds, StageRegs> ks;
    __device__ __forceinline__ void init(const Flow& f, double x, double xend, double px,
                                         double py, double rtol, double atol) {
        dop853_init(f, s, x, xend, (__lane_id() & 1) ? py : px, rtol, atol);
    }
    __device__ __forceinline__ bool body(const Flow& f, double rtol, double atol) {
        return dop853_step_body(f, s, ks, rtol, atol);
    }
    // one attempted step: false when the solve has ended (s.idid says how)
    __device__ __forceinline__ bool step(const Flow& f, double rtol, double atol, long long nmax) {
        return dop853_step_begin(s, nmax) && body(f, rtol, atol);
    }
    // the group's final position: lanes 0 and 1 write x and y
    __device__ __forceinline__ void store(double2* out) const {
        const unsigned g = __lane_id() & (G - 1);
        if (g < 2) reinterpret_cast<double*>(out)[g] = s.y;
    }
};
template <class Flow, class R>
struct Solve<Flow, R, 1> {
    static constexpr int kStates = 1;
    static constexpr unsigned kLdsBytes = 0;
    Dop853State<R> s;
    __device__ __forceinline__ void init(const Flow& f, double x, double xend, double px,
                                         double py, double rtol, double atol) {
        dop853_init(f, s, x, xend, px, py, rtol, atol);
    }
    __device__ __forceinline__ bool step(const Flow& f, double rtol, double atol, long long nmax) {
        return dop853_step(f, s, rtol, atol, nmax);
    }
    __device__ __forceinline__ void store(double2* out) const {
        *out = make_double2(s.px(), s.py());
    }
};
// dynamic LDS of a launch with `block` threads a block
template <class Flow, class R, int G>
constexpr unsigned solve_lds_bytes(int block) {
    return block / 64 * Solve<Flow, R, G>::kLdsBytes;
}
// what the launches' hand-over buffers hold per particle slot
template <class R, int G>
constexpr size_t solve_state_bytes() {
    return G == 1 ? sizeof(Dop853State<R>) : 2 * sizeof(Dop853Lane<R>);
}

}  // namespace nbx
