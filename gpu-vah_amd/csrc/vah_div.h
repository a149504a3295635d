// vah_div.h -- quotients from the hardware's reciprocal estimate, about half the
// instructions of the correctly rounded sequence, whose range scaling the callers'
// operands do not need.
#pragma once

namespace vah {

// The hardware estimates on the device (relative error up to 2^-23); on the host the
// plain quotients, which a test build can put off by as much through VAH_SEED.
#ifndef VAH_SEED
#define VAH_SEED(s) (s)
#endif

__host__ __device__ inline double rcp_estimate(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return VAH_SEED(1.0 / x);
#endif
}

__host__ __device__ inline double rsq_estimate(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return VAH_SEED(1.0 / __builtin_sqrt(x));
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

// sqrt(x) and 1 / sqrt(x), rounded as the square root and the division are, from one
// estimate: a Goldschmidt step, a residual correction of the root and one of the
// inverse.  For x between 1e-280 and 1e280 (the residuals would underflow or overflow
// beyond).
struct Root {
    double root, inverse;
};

__host__ __device__ inline Root root_of(double x) {
    const double y = rsq_estimate(x);
    double g = x * y, h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    const double r = h + h;
    return {g, __builtin_fma(r, __builtin_fma(-g, r, 1.0), r)};
}

// a / r.root, rounded as the division is
__host__ __device__ inline double quotient(double a, const Root &r) {
    const double q = a * r.inverse;
    return __builtin_fma(__builtin_fma(-r.root, q, a), r.inverse, q);
}

}  // namespace vah
