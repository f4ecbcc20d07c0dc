// mdg_math64.h -- FP64 device functions of the pair kernels: reciprocal,
// reciprocal square root and erfc with its Gaussian, each a few operations
// from the hardware estimates instead of the library's general routines.
//
// A pair of the real-space Ewald sum needs sqrt, 1/r, erfc(a r) and
// exp(-(a r)^2).  From the library they cost about 350 FP64 instructions a
// wavefront (IEEE square root and division with their range fix-ups, an erfc
// whose argument branches diverge across the lanes, and a second exponential);
// from here about 75, with one exponential serving both terms.
#pragma once
#include <hip/hip_runtime.h>

// 1/x for normal x: the hardware estimate (about 2^-24) and one third-order
// step, y (1 + h + h^2) with h = 1 - x y: an error of h^3 before rounding.
__device__ __forceinline__ double mdg_rcp64(double x)
{
    const double y = __builtin_amdgcn_rcp(x);
    const double h = __builtin_fma(-x, y, 1.0);
    return __builtin_fma(y, __builtin_fma(h, h, h), y);
}

// a / b for normal b and quotients, from a reciprocal and one correction by the
// remainder a - q b, which is exact.  The reciprocal's error (0.5 ulp and 2^-24 of
// one) times the remainder (at most an ulp or two of q) is below 2^-51 ulp of q, so
// the result is the correctly rounded quotient unless the exact one lies that close
// to a midpoint of two doubles; then it is one of the two.
__device__ __forceinline__ double mdg_div64(double a, double b)
{
    const double y = mdg_rcp64(b);
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// 1/sqrt(x) for normal x > 0, by the same third-order step
// y (1 + h/2 + 3 h^2 / 8), h = 1 - x y^2; r receives sqrt(x), x y with one
// correction for its rounding.
__device__ __forceinline__ double mdg_rsqrt64(double x, double &r)
{
    double y = __builtin_amdgcn_rsq(x);
    const double h = __builtin_fma(-x * y, y, 1.0);
    y = __builtin_fma(y * h, __builtin_fma(h, 0.375, 0.5), y);
    const double s = x * y;
    r = __builtin_fma(__builtin_fma(-s, s, x), 0.5 * y, s);
    return y;
}

// Coefficients (low order first) of (1 + 2x) exp(x^2) erfc(x) as a polynomial
// in y = (x - 3.75) / (x + 3.75), which maps x >= 0 onto [-1, 1) (M. M.
// Shepherd and J. G. Laframboise, Math. Comp. 36, 249 (1981)); the degree-22
// truncation of the Chebyshev series, computed in 60 digits from the
// definition, leaves 8e-17.
#define MDG_ERFCX_N 23
__device__ constexpr double mdg_erfcx_c[MDG_ERFCX_N] = {
    1.2375126308378275,
    -0.14024059858554525,
    0.0035854154854790257,
    0.08227673848999506,
    -0.10880393014244462,
    0.09230432116428125,
    -0.05869339857664934,
    0.02836227737211114,
    -0.00974657968326525,
    0.0017556261651970615,
    0.00029371437804490326,
    -0.00029015535246076896,
    5.164652974193095e-05,
    2.2387565714905518e-05,
    -1.1438048033631918e-05,
    -9.79262570735844e-07,
    1.741982158951425e-06,
    -5.084465377032029e-08,
    -2.485712627127677e-07,
    1.8790823210316808e-08,
    3.197926680817349e-08,
    -1.955135883083941e-09,
    -2.6231073623858514e-09};

// erfc(x) = exp(-x^2) p(y) / (1 + 2x) for x >= 0, and ez = exp(-x^2).  The
// rounding errors of x^2, of 1/(1 + 2x) and of their product are kept (each
// from one fma) and added with the last one, and y = (x - 3.75)/(x + 3.75) is
// formed as 2x/(x + 3.75) - 1, which is exact enough where p is steep.
// Against 113-bit values over x in [0, 6]: within 4.2e-16, rms 1.1e-16
// (erfc() of the device library: 4.2e-16, 1.0e-16); ez within 2.2e-16.
__device__ __forceinline__ double mdg_erfc64(double x, double &ez)
{
    const double e = x * x, lo = __builtin_fma(x, x, -e);
    const double g = exp(-e);
    ez = __builtin_fma(-g, lo, g);
    const double a = x + 3.75, x2 = x + x, b = x2 + 1.0;
    const double inv = mdg_rcp64(a * b);
    const double y = __builtin_fma(x2, b * inv, -1.0), r = a * inv;
    double p = mdg_erfcx_c[MDG_ERFCX_N - 1];
#pragma unroll
    for (int k = MDG_ERFCX_N - 2; k >= 0; k--) p = __builtin_fma(p, y, mdg_erfcx_c[k]);
    const double bl = x2 - (b - 1.0);
    const double c = __builtin_fma(-bl, r, __builtin_fma(-b, r, 1.0));
    const double w = g * r;
    const double wl = __builtin_fma(w, c - lo, __builtin_fma(g, r, -w));
    return __builtin_fma(w, p, wl * p);
}
