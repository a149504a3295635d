// vah_face.h -- signed speed of one reconstructed face state, and the primitive
// variables of a cell, in closed form.
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
// far above rounding.  B < 1e140 as well, so that its square does not overflow; the
// floor of sqrt_coarse keeps it above 1.5e-140, where the root's square is far above
// its own floor.  A state that fails one of the tests (an unphysical or NaN state, or a
// path that may fall back) gets `false`, and the caller runs the reference's iteration;
// every decision is then the full path's.
//
// The root gives the speed without its square roots and quotients by M_T:
//     v = U* x M^DIR / M_T = 2 x^2 M^DIR / (B + sqrt(B^2 - 2 xM^2)),
// and v = F for the eta direction.  The states' Newton setup, one update, the
// root and the speed took 245 issue slots per side (a reciprocal or reciprocal
// square root counting as four), this takes 86 (55 for eta).
#pragma once

#include "vah_div.h"
#include "vah_sqrt.h"

namespace vah {

// sqrt(x) for x >= 0 to 2^-43, at least 1e-140, for the tests only (their margin
// is 1e-9)
__host__ __device__ inline double sqrt_coarse(double x) {
    const double m = __builtin_fmax(x, 1e-280);
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

// What the tests and the root need of a state.
struct FaceSetup {
    double F, x2, m2, c0, B;  // m2 = xM^2
    bool ok;                  // the path from the start ends on the root
};

__host__ __device__ inline FaceSetup face_setup(double t, double M0, double M1, double M2, double M3, double PL,
                                                const FaceStart &s) {
    constexpr double kMargin = 1.0 + 1e-9;
    FaceSetup r;
    r.F = quotient(M3, M0 + PL);
    const double Ft = t * r.F;
    const double Ft2 = Ft * Ft;
    r.x2 = __builtin_fma(-Ft, Ft, 1.0);
    r.m2 = r.x2 * __builtin_fma(M1, M1, M2 * M2);
    const double xM = sqrt_coarse(r.m2);
    const double bL = __builtin_fma(r.x2, M0, -Ft2 * PL);
    r.c0 = __builtin_fma(-t * Ft, M3, M0);
    r.B = __builtin_fma(0.5, r.c0 - PL, bL);
    const double f0 = __builtin_fma(s.U0, __builtin_fma(-0.5 * s.U0, xM, r.B), -xM);
    const double h = s.U0 * s.w * __builtin_fma(-s.U0, xM, r.B);
    r.ok = (Ft2 < 1.0 - 1e-6) & (r.B > 1.5 * kMargin * xM) & (r.B < 1e140) & (r.c0 > kMargin * xM) &
           (f0 <= (1.0 - 1e-9) * h);
    return r;
}

// B + sqrt(B^2 - 2 xM^2), the denominator of the root
__host__ __device__ inline double root_denominator(const FaceSetup &r) {
    const double disc = __builtin_fmax(__builtin_fma(r.B, r.B, -2.0 * r.m2), 1e-300);
    return r.B + sqrt_refine(disc, rsq_estimate(disc));
}

// true: *v is the speed the reference's path from s gives; false: run the path
template <int DIR>
__host__ __device__ inline bool face_speed(double t, double M0, double M1, double M2, double M3, double PL,
                                           const FaceStart &s, double *v) {
    const FaceSetup r = face_setup(t, M0, M1, M2, M3, PL, s);
    *v = DIR == 3 ? r.F : quotient(2.0 * r.x2 * (DIR == 1 ? M1 : M2), root_denominator(r));
    return r.ok;
}

// 1 / sqrt(x), the estimate refined twice (~1 ulp)
__host__ __device__ inline double inverse_sqrt(double x) {
    double y = rsq_estimate(x);
    const double h = 0.5 * x;
    y = __builtin_fma(y, __builtin_fma(-h * y, y, 0.5), y);
    return __builtin_fma(y, __builtin_fma(-h * y, y, 0.5), y);
}

// The primitive variables of a cell from the same root: with W = 1 / (B + sqrt(..)),
// U* = 2 xM W and C = 1 / sqrt(1 - U*^2) = sqrt(1 + u_T^2),
//     u^tau = C / x, u^i = 2 x W C M^i, u^eta = F C / x, e = c0 - 2 xM^2 W,
// without the three Newton passes (each a reciprocal square root and a
// reciprocal in sequence) and the quotients by x and M_T of the iteration.  The
// cell waves are one long dependent chain: with the regulator's quotients taken
// from reciprocal square roots and p(e) read early, 261x243 went from 38.6 to
// 37.7 us per step, 611x587 from 147 to 143, 101x101x30 from 182 to 179.  Against
// 80-bit arithmetic u is off by 3.4e-16 rms (the iteration: 9.6e-16).
struct CellRoot {
    double e, ut, ux, uy, un;
};

__host__ __device__ inline bool cell_root(double t, double M0, double M1, double M2, double M3, double PL,
                                          const FaceStart &s, CellRoot *c) {
    const FaceSetup r = face_setup(t, M0, M1, M2, M3, PL, s);
    const double W = quotient(1.0, root_denominator(r));
    const double ix = inverse_sqrt(__builtin_fmax(r.x2, 1e-300));
    const double mW = 2.0 * r.m2 * W;
    const double C = inverse_sqrt(__builtin_fmax(__builtin_fma(-2.0 * mW, W, 1.0), 1e-300));
    const double k = 2.0 * (r.x2 * ix) * (W * C);
    c->e = r.c0 - mW;
    c->ut = C * ix;
    c->ux = k * M1;
    c->uy = k * M2;
    c->un = r.F * c->ut;
    return r.ok;
}

}  // namespace vah
