// gf_exact.h -- quotients and square roots of the step's inner loops with the
// bits of the general operations, without their range handling.
//
// The step kernel is bound by VALU issue, and its ~50 divisions and ~10
// square roots per cell were a third of the instructions: `a / b` costs 11
// (two scalings, the quarter-rate reciprocal, two Newton steps, the quotient
// with its residual correction, and the unscaling and special-case fixups),
// sqrt about 17.  Two things make them cheaper without changing a bit:
//
//  * inside the range below nothing can overflow or lose bits to underflow,
//    so the scaling and fixup steps have nothing to do;
//  * quotients with one denominator share its reciprocal: each further one is
//    a product and one residual correction (3 instructions).
//
// The same bits.  For `a / b` in double precision the compiler emits, between
// the two scalings and the fixup, the reciprocal's seed, two Newton steps, the
// product, its residual and the correction: the operations of recip and quot, in
// that order; for sqrt, between two scalings, those of root.  Where nothing is
// scaled or fixed up the results are therefore equal, whatever the seeds are.
// (The sequences are the published ones: P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990;
// J.-M. Muller et al., Handbook of Floating-Point Arithmetic, 2nd ed., 2018,
// sections 4.7 and 4.8.  With a seed good to 20 bits y is 1/b rounded unless 1/b
// lies within 2^-80 of the midpoint of two doubles, and q then a/b rounded: the
// residual is exact when |a| >= 2^-960 or a = 0.  Denominators one or two ulps
// below a power of two have such reciprocals; there only the equality with `a / b`
// is claimed.)  A zero quotient loses the sign of its zero.
//
// Range.  step_cell_in_range bounds a tile's cells, and
// step_params_in_range bounds the parameters; a tile that holds anything else
// (a NaN, a momentum of 1e-80, 10^9 m of water) takes the same step with the
// general operations.  Write m = 2^-240 for the smallest non-zero momentum or
// bathymetry.  A non-zero sum of two values is at least 2^-52 of the smaller,
// so, with drytol >= 2^-14, 2^-4 <= g <= 2^8, h <= 2^30, |hu|, |hv| <= 2^20:
//   u, v in {0} or [m 2^-30, 2^34]; c = sqrt(g h) in [2^-9, 2^19];
//   |u| / c <= 2^20 drytol^-3/2 g^-1/2 <= 2^43, so the differences of wave
//   speeds that divide (s2 - s0, sE2 - sE1, lam0 - lam2) never vanish;
//   speeds in {0} or [2^-68, 2^36]; |delb| in {0} or [m 2^-52, 2^31];
//   deldelh >= m 2^-205, hstarHLL (sE2 - sE1) >= m 2^-240,
//   delh - deldelh >= m 2^-354, the numerators of beta >= m 2^-714 = 2^-954,
// and every product stays below 2^800.  Two families of numerators have no
// such bound, because they multiply waves with waves: the limiter's dot
// products and rpt2's.  They are tested one by one (quotients_tiny) and
// divided in the general way when they are too small.
#pragma once

#include <cmath>

#ifndef GF_DEVICE
#define GF_DEVICE __device__ __forceinline__
#endif

namespace gf {

GF_DEVICE unsigned long long bits_of(double x) { return __builtin_bit_cast(unsigned long long, x); }

// smallest non-zero |hu|, |hv|, |b| of a fast tile: 2^-240 (zero_or_within)
constexpr double STEP_MAX_Q = 0x1p20;    // largest |hu|, |hv|
constexpr double STEP_MAX_H = 0x1p30;    // largest h, |b|
constexpr int QUOT_MIN_EXP = -900;       // numerators and denominators below 2^-901 divide in the general way

inline bool step_params_in_range(double grav, double drytol)
{
    return grav >= 0x1p-4 && grav <= 0x1p8 && drytol >= 0x1p-14 && drytol <= 0x1p10;
}

// |x| is 0 or lies in [2^-240, hi], by its high word (hi a power of two).
GF_DEVICE bool zero_or_within(double x, double hi)
{
    constexpr unsigned lo = (1023u - 240u) << 20;
    const unsigned top = (unsigned)(bits_of(hi) >> 32);
    return x == 0.0 || ((unsigned)(bits_of(x) >> 32) & 0x7fffffffu) - lo < top - lo;
}

// A cell after b4step2 that the fast quotients are made for.
GF_DEVICE bool step_cell_in_range(double h, double hu, double hv, double b)
{
    return h <= STEP_MAX_H && zero_or_within(hu, STEP_MAX_Q) && zero_or_within(hv, STEP_MAX_Q) &&
           zero_or_within(b, STEP_MAX_H);
}

#ifndef GF_SEED_FUNCTIONS
GF_DEVICE double rcp_seed(double b) { return __builtin_amdgcn_rcp(b); }
GF_DEVICE double rsq_seed(double b) { return __builtin_amdgcn_rsq(b); }
GF_DEVICE int exponent_of(double a) { return __builtin_amdgcn_frexp_exp(a); }  // 0 for 0, NaN and Inf
#endif

namespace fast {

// A denominator with its refined reciprocal.
struct Recip {
    double b, y;
};

GF_DEVICE Recip recip(double b)
{
    double y = rcp_seed(b);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    y = ::fma(y, ::fma(-b, y, 1.0), y);
    return Recip{b, y};
}

GF_DEVICE double quot(double a, const Recip& d)
{
    const double q = a * d.y;
    return ::fma(::fma(-d.b, q, a), d.y, q);
}

GF_DEVICE double quot(double a, double b) { return quot(a, recip(b)); }

// sqrt(x), x = 0 or 2^-700 <= x <= 2^700.
GF_DEVICE double root(double x)
{
    const double y = rsq_seed(::fmax(x, 0x1p-700));
    double s = x * y, h = 0.5 * y;
    const double r = ::fma(-h, s, 0.5);
    s = ::fma(s, r, s);
    h = ::fma(h, r, h);
    s = ::fma(::fma(-s, s, x), h, s);
    return ::fma(::fma(-s, s, x), h, s);
}

// Maximum and minimum of two numbers where the sign of a zero result does not
// matter: one instruction instead of a compare and two selects.  (A NaN operand
// is lost here; LLVM Flang's MAX and MIN, fmaxf64 and fminf64, return the
// second operand then.)
GF_DEVICE double vmax(double a, double b) { return ::fmax(a, b); }
GF_DEVICE double vmin(double a, double b) { return ::fmin(a, b); }

}  // namespace fast
}  // namespace gf
