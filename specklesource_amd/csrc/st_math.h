// Short forms of correctly rounded divisions and square roots
// (tests/test_gpu_math.py compares them with the full ones).
#pragma once

#include <hip/hip_runtime.h>

namespace sttrack {

// sqrtf for finite x >= 2^-96: the rounded product of x and its hardware
// reciprocal square root, then one Newton step by its exact residual (Markstein's
// correction of a root).  Correctly rounded at every such float (the test
// compares all 1.88e9); five instructions against nine for the hardware root
// with its two one-ulp tests, sixteen for sqrtf.
__device__ inline float sqrt_rn_normal(float x)
{
    const float y = __builtin_amdgcn_rsqf(x);
    const float s = x * y;
    return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
}

// Whether any of n values (sums of squares, so never negative) in the wave lies
// outside sqrt_rn_normal's range, NaN included: least and greatest of the bit
// patterns, two values an instruction.
template <int n>
__device__ inline bool sqrt_needs_full(const float (&x)[n])
{
    static_assert(n % 2 == 0, "pairs");
    unsigned lo = 0xffffffffu, hi = 0;
#pragma unroll
    for (int j = 0; j < n; j += 2) {
        const unsigned a = __float_as_uint(x[j]), b = __float_as_uint(x[j + 1]);
        lo = min(lo, min(a, b));
        hi = max(hi, max(a, b));
    }
    return __builtin_amdgcn_ballot_w64(lo < 0x0f800000u || hi >= 0x7f800000u) != 0;
}

// The classes of negative and positive, normal and subnormal numbers.
__device__ inline bool finite_nonzero(double x) { return __builtin_amdgcn_class(x, 0x198); }

// x / n, correctly rounded, from rn = 1 / n rounded (Markstein: the residual of
// the rounded product is exact).  Infinite quotients come out as NaN, negative
// zeros as zero.
__device__ inline double div_by(double x, double n, double rn)
{
    const double q = x * rn;
    return fma(fma(-q, n, x), rn, q);
}

// x / sqrt(a), both correctly rounded, for finite x and a in (1e-280, 1e280).
// From one reciprocal square root: coupled Newton steps (Goldschmidt) give the
// root g and h = 1 / (2 g), a residual step rounds g.  2 h is a few units from
// 1 / g (g has been rounded since); a Newton step rounds it, a residual step
// brings the quotient within a unit, and another (Markstein's) rounds it.
__device__ inline double div_sqrt(double x, double a)
{
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y, h = 0.5 * y;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
    }
    g = fma(fma(-g, g, a), h, g);
    const double r = h + h, rg = fma(fma(-g, r, 1.0), r, r);
    const double p = x * rg, q = fma(fma(-p, g, x), rg, p);
    return fma(fma(-q, g, x), rg, q);
}

// The normalised correlation of a lag (corrTrackFast.c:407-477, 862-899): c the
// correlation, mean and var those of the other window, s1 and s2 the sums of
// the n = 1 / rn samples under the lag and of their squares, rn1 = 1 / (n - 1).
// Short quotients where the variances' product and the numerator are finite and
// far from the range's ends: then so were the means, and no guard is needed on
// either.  All else takes full divisions: constant windows (0 / 0), overflow,
// NaN.
__device__ inline double ncc_value(double c, double mean, double var, double s1, double s2, double n, double rn,
                                   double rn1)
{
#pragma clang fp contract(off)
    const double m = div_by(s1, n, rn), sig = div_by(s2, n - 1., rn1) - m * m;
    const double num = c - mean * m, a = var * sig;
    if (a > 1e-280 && a < 1e280 && fabs(num) < 1e280)
        return div_sqrt(num, a);
    const double mf = s1 / n;
    return (c - mean * mf) / sqrt(var * (s2 / (n - 1.) - mf * mf));
}

}  // namespace sttrack
