// hc_arith.hpp -- FP64 building blocks of the fused kernels: reciprocals, square roots and products
// formed from the hardware seeds with as many Newton steps as full precision takes, and no range
// handling.  On the device a correctly rounded FP64 division is 11 instructions and a square root 18,
// of which the scaling of extreme exponents, the last half-ulp correction and the special cases are
// about half; here they are 5 and 9 (within 1 ulp).  Arguments are gas states and mesh metrics, far
// from 2^+-900; infinities and zero divisors give NaN instead of an infinity, which the update's
// finiteness check reports alike.  The host versions are the plain operations.
#pragma once

#include <cfloat>
#include <cmath>

#if defined(__HIPCC__)
#define HC_HD __host__ __device__ inline
#else
#define HC_HD inline
#endif

namespace hc {

HC_HD double hc_fma(double a, double b, double c) { return ::fma(a, b, c); }
HC_HD double hc_copysign(double a, double b) { return ::copysign(a, b); }

// 1 / b: hardware seed (about 2^-24), two Newton steps
HC_HD double hc_rcp(double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(b);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    return y;
#else
    return 1.0 / b;
#endif
}

// sqrt(x) and, in the second form, also its reciprocal: hardware seed of 1/sqrt, one coupled Newton
// step of g ~ sqrt(x) and h ~ 1/(2 sqrt(x)), one residual step of g (and of the reciprocal).  x = 0 gives g = 0 (the added smallest
// normal number leaves every x above 2^-969 as it is); a negative or NaN x gives NaN.
HC_HD double hc_root(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(x + DBL_MIN);
    double g = x * y, h = 0.5 * y;
    const double r = ::fma(-h, g, 0.5);
    g = ::fma(g, r, g);
    h = ::fma(h, r, h);
    return ::fma(::fma(-g, g, x), h, g);
#else
    return ::sqrt(x);
#endif
}
HC_HD double hc_root(double x, double& inv)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(x + DBL_MIN);
    double g = x * y, h = 0.5 * y;
    const double r = ::fma(-h, g, 0.5);
    g = ::fma(g, r, g);
    h = ::fma(h, r, h);
    g = ::fma(::fma(-g, g, x), h, g);
    inv = h + h;
    inv = ::fma(inv, ::fma(-inv, g, 1.0), inv);
    return g;
#else
    const double g = ::sqrt(x);
    inv = 1.0 / g;
    return g;
#endif
}

// a / b and sqrt(x) with the bits of the correctly rounded operations: Newton-Raphson on the reciprocal with
// Markstein's final quotient correction, and Goldschmidt's coupled iteration with two residual corrections of
// the root, without the scaling of extreme exponents that library sequences begin and end with (9
// instructions instead of 11, and 13 instead of 18).  The
// fixup keeps zeros, infinities and NaNs as they are; bits agree for operands and quotients of
// magnitude 2^-900 .. 2^900 and roots of 2^-767 and more.  The mixed-precision objects keep the
// compiler's sequences (their few FP64 divisions gain nothing: the 48-case batch ran 4 % slower with these).
HC_HD double hc_div(double a, double b)
{
#if defined(__HIP_DEVICE_COMPILE__) && !defined(HC_MIXED_OBJECT)
    double y = __builtin_amdgcn_rcp(b);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    const double q = a * y;
    return __builtin_amdgcn_div_fixup(::fma(::fma(-b, q, a), y, q), b, a);
#else
    return a / b;
#endif
}
template <class R> HC_HD R hc_div(R a, R b) { return a / b; }

HC_HD double hc_sqrt(double x)
{
#if defined(__HIP_DEVICE_COMPILE__) && !defined(HC_MIXED_OBJECT)
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = ::fma(-h, g, 0.5);
    g = ::fma(g, r, g);
    h = ::fma(h, r, h);
    g = ::fma(::fma(-g, g, x), h, g);
    g = ::fma(::fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // +-0 and +inf are their own roots
#else
    return ::sqrt(x);
#endif
}

}   // namespace hc
