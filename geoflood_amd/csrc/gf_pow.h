// gf_pow.h -- the two powers of the step, correctly rounded.
//
// The reference evaluates h**(7.d0/3.d0) in src2 (geoclaw_src2_fort.f90:62)
// and (q0(2)/sqrt(grav))**(2.0d0/3.0d0) for the hydrograph's inflow depth
// (geoflood_bc2_fort.f90:63 and twins, hydrograh_module.f90:245-318), i.e.
// pow(x, y) of the host libm with y the double nearest 7/3 or 2/3.  The device's own pow rounds differently from glibc's
// in about a quarter of calls (one ulp), and such differences, carried by the
// flow, move wet/dry fronts apart after O(100) steps.  These functions return
// the correctly rounded x^y (the exact real power of the double y), which is
// what glibc's pow returns too except in the rare calls it misrounds.
//
// Method.  y = k/3 + d exactly, with d = 2^-51/3 for 7/3 (k = 7) and
// d = -2^-53/3 for 2/3 (k = 2), so x^y = x^(k/3) * x^d:
//  * a cube root c good to an ulp, refined by one Newton step
//    c - (c^3 - x) / (3 c^2) with c^3 - x formed from exact products
//    (the FMA error-free transformation of a product; J.-M. Muller et al.,
//    Handbook of Floating-Point Arithmetic, 2nd ed., 2018, sections 4.4 and
//    5.3), giving cbrt(x) as a double-double to about 2^-102;
//  * x^2 (for 7/3) as an exact double-double product, x^(k/3) as the
//    double-double product with the refined root;
//  * x^d = exp(d ln x) = 1 + d ln x + (d ln x)^2 / 2 ..., without the square:
//    it is 2^-100 at |ln x| = 7 and 2^-94 at the ends of the range below, more
//    than all that the root and the logarithm leave;
//  * one final rounding of the double-double value (hi + (lo + hi d ln x)):
//    the correctly rounded result unless x^y lies within that of the midpoint
//    of two doubles.
// The host build takes c and ln x from its library.  The device forms both
// itself between 2^-100 and 2^60 (root_and_log), as good as the library's: the
// library's handle every argument, and were most of the friction term, a tenth
// of the step kernel's instructions.  Arguments outside (2^-300, 2^300) (zero,
// negatives, subnormals, Inf, NaN) go to the library pow.  GF_HOST_DEVICE lets
// a host test compile the same functions, and GF_OWN_ROOT with the four seed
// functions the device's root and logarithm.
#pragma once

#include <cmath>

#ifndef GF_HOST_DEVICE
#define GF_HOST_DEVICE __host__ __device__
#endif

namespace gf {

#if defined(__HIP_DEVICE_COMPILE__)
#define GF_OWN_ROOT
// x^(-1/3) in single precision, to 2^-17 for 2^-100 <= x <= 2^60 (the product
// that goes to exp2 reaches 33.3, where an ulp is 2^-18).
__device__ inline double root_seed(double x)
{
    return (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)x) * (-1.0f / 3.0f));
}
__device__ inline double inverse_seed(double d) { return __builtin_amdgcn_rcp(d); }
__device__ inline double mantissa_of(double x) { return __builtin_amdgcn_frexp_mant(x); }  // [1/2, 1)
__device__ inline int power_of(double x) { return __builtin_amdgcn_frexp_exp(x); }
#endif

#if defined(GF_OWN_ROOT)
// For 2^-100 <= x <= 2^60: x^(-1/3) to 2^-52, the cube root to an ulp and ln x
// to 2^-51 or an ulp.  The root: the seed r0 and one step of the fourth-order
// iteration r0 (1 + e/3 + 2 e^2/9 + 14 e^3/81), e = 1 - x r0^3 (|e| < 2^-15: the
// next term is 2^-63), then c = x r^2 with one Newton step.  The logarithm:
// x = 2^k z with z in [sqrt(1/2), sqrt(2)) and ln z = 2 atanh((z-1)/(z+1)) by
// its series (|s| <= 0.172: ten terms leave 2^-56).
GF_HOST_DEVICE inline void root_and_log(double x, double& r, double& c, double& lnx)
{
    const double r0 = root_seed(x);
    const double e = ::fma(-(x * r0), r0 * r0, 1.0);
    r = ::fma(r0 * e, ::fma(e, ::fma(e, 14.0 / 81.0, 2.0 / 9.0), 1.0 / 3.0), r0);
    c = x * (r * r);
    const double a = c * c;
    c = ::fma(-(::fma(a, c, -x) + ::fma(c, c, -a) * c), (r * r) * (1.0 / 3.0), c);
    double z = mantissa_of(x);
    int k = power_of(x);
    if (z < 0.70710678118654752) {
        z = z + z;
        k -= 1;
    }
    const double d = z + 1.0;
    double q = inverse_seed(d);
    q = ::fma(q, ::fma(-d, q, 1.0), q);
    q = ::fma(q, ::fma(-d, q, 1.0), q);
    const double s = (z - 1.0) * q, w = s * s;
    double p = 1.0 / 19.0;
    p = ::fma(p, w, 1.0 / 17.0);
    p = ::fma(p, w, 1.0 / 15.0);
    p = ::fma(p, w, 1.0 / 13.0);
    p = ::fma(p, w, 1.0 / 11.0);
    p = ::fma(p, w, 1.0 / 9.0);
    p = ::fma(p, w, 1.0 / 7.0);
    p = ::fma(p, w, 0.2);
    p = ::fma(p, w, 1.0 / 3.0);
    p = ::fma(p, w, 1.0);
    lnx = ::fma((double)k, 0.69314718055994531, (s + s) * p);
}
#endif

// cbrt(x) = hi + lo to about 2^-102 relative and ln x, x normal and > 0.
GF_HOST_DEVICE inline double cbrt_dd(double x, double& lo, double& lnx)
{
    double c, inv = 0.0;  // inv: 1 / (3 c^2) to 2^-50, or 0 to divide
#if defined(GF_OWN_ROOT)
    if (x >= 0x1p-100 && x <= 0x1p60) {
        double r;
        root_and_log(x, r, c, lnx);
        inv = (r * r) * (1.0 / 3.0);
    } else
#endif
    {
        c = ::cbrt(x);
        lnx = ::log(x);
    }
    const double a = c * c;
    const double a_lo = ::fma(c, c, -a);    // c^2 = a + a_lo exactly
    const double b = a * c;
    const double b_lo = ::fma(a, c, -b);    // a c = b + b_lo exactly
    // c^3 - x: b - x is exact (b lies within a factor 2 of x), the rest is
    // the low-order part of c^3
    const double r = (b - x) + (b_lo + a_lo * c);
    lo = inv != 0.0 ? -r * inv : -r / (3.0 * a);
    return c;
}

// x^y for y = 7.0/3.0 (the double nearest 7/3), correctly rounded.
GF_HOST_DEVICE inline double pow_7_3(double x)
{
    if (!(x > 0x1p-300 && x < 0x1p300)) return ::pow(x, 7.0 / 3.0);
    double c_lo, lnx;
    const double c = cbrt_dd(x, c_lo, lnx);
    const double p = x * x;
    const double e = ::fma(x, x, -p);         // x^2 = p + e exactly
    const double hi = p * c;
    const double lo = ::fma(p, c, -hi) + (p * c_lo + e * c);
    const double t = lnx * (1.0 / 6755399441055744.0);   // d ln x, d = 1 / (3 * 2^51)
    return hi + (lo + hi * t);
}

// x^y for y = 2.0/3.0 (the double nearest 2/3), correctly rounded.
GF_HOST_DEVICE inline double pow_2_3(double x)
{
    if (!(x > 0x1p-300 && x < 0x1p300)) return ::pow(x, 2.0 / 3.0);
    double c_lo, lnx;
    const double c = cbrt_dd(x, c_lo, lnx);
    const double hi = c * c;
    const double lo = ::fma(c, c, -hi) + 2.0 * (c * c_lo);
    const double t = lnx * (-1.0 / 27021597764222976.0);  // d ln x, d = -1 / (3 * 2^53)
    return hi + (lo + hi * t);
}

}  // namespace gf
