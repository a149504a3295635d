// vah_face.h -- signed speed of one reconstructed face state, in closed form.
//
// The KT flux needs v = u^DIR / u^tau of the two states of a face, which the
// reference finds by Newton's method on
//     f(u) = U g - xM,   U = u / sqrt(1 + u^2),  g = bL + b (e - P_L) / 2,
//     e = c0 - U xM      (EnergyMomentumTensor.cpp:30-72 with Pi = 0)
// from M^mu = T^{tau mu} - pi^{tau mu}, F = M^3 / (M^0 + P_L), Ft = tau F,
// x^2 = |1 - Ft^2|, xM = x M_T, b = x^2 + Ft^2, bL = x^2 M^0 - Ft^2 P_L,
// c0 = M^0 - Ft^2 (M^0 + P_L).  For Ft^2 < 1, b = 1 and f is the quadratic
//     f = -(xM / 2) U^2 + B U - xM,   B = bL + (c0 - P_L) / 2,
// increasing and concave in u left of its vertex U = B / xM.
//
// face_speed takes the quadratic's smaller root U* (the physical one) when
// the Newton path from the start u0 must end there, which it does if
//   (a) f(1) > 0: the one root in [0, 1) is U*, and the vertex lies right of 1;
//   (b) c0 > xM: e stays positive for every U in [0, 1], so no iterate fails
//       the reference's e < 0 test;
//   (c) the first update is clearly positive.  Left of the root an update of a
//       concave increasing function moves up towards the root and never past
//       it, so only the first update (from a start right of the root) can
//       leave [0, u*]; every later one climbs towards the root.
// (c) needs no division: u1 = u0 - f/f' >= eps u0  <=>  f <= (1 - eps) u0 f',
// and u0 f' = U0 (B - U0 xM) / (1 + u0^2).  The tests keep a margin of 1e-9,
// far above rounding.  A state that fails one of them (an unphysical or NaN
// state, or a path that may fall back) gets `false`, and the caller runs the
// reference's iteration; every decision is then the full path's.
//
// The root gives the speed without its square roots and quotients by M_T:
//     v = U* x M^DIR / M_T = 2 x^2 M^DIR / (B + sqrt(B^2 - 2 xM^2)),
// and v = F for the eta direction.  The states' Newton setup, one update, the
// root and the speed took 245 issue slots per side (a reciprocal or reciprocal
// square root counting as four), this takes 86 (55 for eta).
#pragma once


#include "vah_sqrt.h"

namespace vah {

// hardware estimates on the device, the plain quotients on the host
__host__ __device__ inline double rcp_estimate(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return 1.0 / x;
#endif
}

__host__ __device__ inline double rsq_estimate(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return 1.0 / __builtin_sqrt(x);
#endif
}

// a / b: the estimate refined twice, then a residual correction (~1 ulp for
// normal operands)
__host__ __device__ inline double quotient(double a, double b) {
    double r = rcp_estimate(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// sqrt(x) for x >= 0 to about 2^-45, for the tests only (their margin is 1e-9)
__host__ __device__ inline double sqrt_coarse(double x) {
    const double m = __builtin_fmax(x, 1e-300);
    const double y = rsq_estimate(m), g = m * y;
    return __builtin_fma(__builtin_fma(-g, g, m), 0.5 * y, g);
}

// The start of a face's two solves: U0 = u0 / sqrt(1 + u0^2) and 1 / (1 + u0^2)
// from u0^2 (coarse: used by the tests only).
struct FaceStart {
    double U0, w;
};

__host__ __device__ inline FaceStart face_start(double u0sq) {
    const double d = 1.0 + u0sq;
    const double y = rsq_estimate(d);
    const double rs = __builtin_fma(y, __builtin_fma(-0.5 * d * y, y, 0.5), y);
    FaceStart s;
    s.U0 = sqrt_coarse(u0sq) * rs;
    s.w = rs * rs;
    return s;
}

// true: *v is the speed the reference's path from s gives; false: run the path
template <int DIR>
__host__ __device__ inline bool face_speed(double t, double M0, double M1, double M2, double M3, double PL,
                                           const FaceStart &s, double *v) {
    constexpr double kMargin = 1.0 + 1e-9;
    const double F = quotient(M3, M0 + PL);
    const double Ft = t * F;
    const double Ft2 = Ft * Ft;
    const double x2 = __builtin_fma(-Ft, Ft, 1.0);
    const double m2 = x2 * __builtin_fma(M1, M1, M2 * M2);  // xM^2
    const double xM = sqrt_coarse(m2);
    const double bL = __builtin_fma(x2, M0, -Ft2 * PL);
    const double c0 = __builtin_fma(-t * Ft, M3, M0);
    const double B = __builtin_fma(0.5, c0 - PL, bL);
    const double f0 = __builtin_fma(s.U0, __builtin_fma(-0.5 * s.U0, xM, B), -xM);
    const double h = s.U0 * s.w * __builtin_fma(-s.U0, xM, B);
    const bool ok = (Ft2 < 1.0 - 1e-6) & (B > 1.5 * kMargin * xM) & (c0 > kMargin * xM) & (f0 <= (1.0 - 1e-9) * h);
    if (DIR == 3) {
        *v = F;
    } else {
        const double disc = __builtin_fmax(__builtin_fma(B, B, -2.0 * m2), 1e-300);
        const double D = B + sqrt_refine(disc, rsq_estimate(disc));
        *v = quotient(2.0 * x2 * (DIR == 1 ? M1 : M2), D);
    }
    return ok;
}

}  // namespace vah
