// FP64 logarithm, angle, sine / cosine and reciprocal square root for the
// polar powers, written for the arguments that occur there.
//
// The device library's log, acos, exp and sincos spend most of their
// instructions on double-double carries, range reduction for huge arguments
// and special values. The map's arguments are positive normal squared norms,
// angles in [0, pi] and their products with an exponent, so a short reduction
// and one polynomial do (coefficients: fit_math64.py): log 26 instead of about
// 70 instructions, angle + sine + cosine about 65 instead of about 200.
// Largest errors, measured on gfx950 over the ranges below against 80-bit
// arithmetic (2^22 arguments each): quotient 0.5 ulp, log 0.9 ulp, angle 2.5
// ulp (the library's acos of a rounded w / |q| loses far more near 0 and pi),
// sine 1.2 ulp, cosine 1.2e-16, square root and its reciprocal 0.5 and 1.7 ulp,
// exponential 1.0 ulp, hyperbolic tangent 0.81 ulp.
//
// Callers keep arguments in range themselves (see the range stated at each
// function and polar_unit's tests); outside it the results are garbage or NaN,
// never a trap.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qj {

// kInLoop: every constant is set in a scalar register pair where it is used. The
// compiler otherwise keeps a polar power's constants in registers across the
// root loop (178 instead of 101 VGPRs in k_grid64); two scalar moves per use
// issue beside other waves' vector work. Code that runs once per point leaves
// the constants to the compiler.
template <bool kInLoop>
__device__ __forceinline__ double k64(double c) {
  if constexpr (kInLoop) asm volatile("" : "+s"(c));
  return c;
}

// n / d for normal d and quotient: reciprocal estimate, one Newton step, one
// residual correction.
__device__ __forceinline__ double div64(double n, double d) {
#pragma clang fp contract(off)
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// log(x) for normal positive x. x = 2^k m with m in [sqrt(1/2), sqrt(2)),
// f = m - 1 (exact), s = f / (2 + f): log m = 2 atanh(s) = 2 s + s R(s^2) =
// f - s (f - R), since 2 s = f - s f. This reduction, with the offset to the
// high word that splits at sqrt(1/2), and this form of the sum are the published
// method of fdlibm's e_log.c (K. C. Ng, Sun Microsystems, 1993); the polynomial
// is fit_math64.py's. Zero, denormal, infinite and NaN x give a finite result
// beyond +-700.
template <bool kInLoop = false>
__device__ __forceinline__ double log64(double x) {
#pragma clang fp contract(off)
  const uint64_t bits = __builtin_bit_cast(uint64_t, x);
  const uint32_t hi = (uint32_t)(bits >> 32) + (0x3ff00000u - 0x3fe6a09eu);
  const int k = (int)(hi >> 20) - 0x3ff;
  const uint32_t mh = (hi & 0x000fffffu) + 0x3fe6a09eu;
  const double m = __builtin_bit_cast(double, (uint64_t)mh << 32 | (uint32_t)bits);
  const double f = m - 1.0;
  const double s = div64(f, m + 1.0);
  const double z = s * s;
  double p = k64<kInLoop>(0.14616449685043406);
  p = __builtin_fma(p, z, k64<kInLoop>(0.15331721600556042));
  p = __builtin_fma(p, z, k64<kInLoop>(0.18182889125261723));
  p = __builtin_fma(p, z, k64<kInLoop>(0.2222221113479508));
  p = __builtin_fma(p, z, k64<kInLoop>(0.28571428625975487));
  p = __builtin_fma(p, z, k64<kInLoop>(0.39999999999899505));
  p = __builtin_fma(p, z, k64<kInLoop>(0.666666666666667));
  const double t = __builtin_fma(-p, z, f);  // f - R
  const double dk = (double)k;
  // ln 2 = 0x1.62e42fefa38p-1 (k times it is exact) + 0x1.ef35793c7673p-45
  const double lo = __builtin_fma(-s, t, dk * k64<kInLoop>(0x1.ef35793c7673p-45));
  return __builtin_fma(dk, k64<kInLoop>(0x1.62e42fefa38p-1), f + lo);
}

// sqrt(x) and 1 / sqrt(x) for normal x in [2^-900, 2^900] (Goldschmidt steps
// from the estimate). x = 0 gives NaN for both.
__device__ __forceinline__ void sqrt_rsqrt64(double x, double& root, double& inverse) {
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double r = __builtin_fma(-g, h, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  r = __builtin_fma(-g, h, 0.5);
  h = __builtin_fma(h, r, h);
  root = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  inverse = 2.0 * h;
}

// The angle of w + i y for y >= 0, in [0, pi] (y and w finite, not both 0,
// their larger one in [2^-450, 2^450]): octant reduction to mn / mx, beyond
// tan(pi / 8) a rotation by pi / 4, then atan(u) = u + u z P(z).
template <bool kInLoop = false>
__device__ __forceinline__ double angle64(double y, double w) {
#pragma clang fp contract(off)
  const double aw = __builtin_fabs(w);
  const bool steep = y > aw;
  const double mx = steep ? y : aw, mn = steep ? aw : y;
  const bool wide = mn > k64<kInLoop>(0.41421356237309503) * mx;
  const double n = wide ? mn - mx : mn, d = wide ? mn + mx : mx;
  const double u = div64(n, d);
  const double z = u * u;
  double p = k64<kInLoop>(0.016285756855221028);
  p = __builtin_fma(p, z, k64<kInLoop>(-0.034570561981427744));
  p = __builtin_fma(p, z, k64<kInLoop>(0.04551593220626549));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.05230454270650244));
  p = __builtin_fma(p, z, k64<kInLoop>(0.05878928997834775));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.06666424885738255));
  p = __builtin_fma(p, z, k64<kInLoop>(0.07692296375032143));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.09090908753500877));
  p = __builtin_fma(p, z, k64<kInLoop>(0.11111111105155447));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.14285714285659828));
  p = __builtin_fma(p, z, k64<kInLoop>(0.19999999999999804));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.3333333333333333));
  // +-(u + u z P) added to its multiple of pi / 4 in two parts: atan(t) = u or
  // pi / 4 + u; y steep: pi / 2 - atan(t); w < 0: pi - that
  double a = __builtin_fma(u * z, p, wide ? 0.78539816339744828 : 0.0);  // pi / 4 - 3.06e-17
  a = (wide ? u + 3.061616997868383e-17 : u) + a;
  if (steep) a = 1.5707963267948966 - (a - 6.123233995736766e-17);
  return w < 0.0 ? 3.141592653589793 - (a - 1.2246467991473532e-16) : a;
}

// (e^r - 1 - r) / r^2 for |r| <= ln 2 / 2
template <bool kInLoop>
__device__ __forceinline__ double exp_poly(double r) {
#pragma clang fp contract(off)
  double p = k64<kInLoop>(2.0914679376583935e-09);
  p = __builtin_fma(p, r, k64<kInLoop>(2.510520637395701e-08));
  p = __builtin_fma(p, r, k64<kInLoop>(2.7557273661348637e-07));
  p = __builtin_fma(p, r, k64<kInLoop>(2.7557255425746435e-06));
  p = __builtin_fma(p, r, k64<kInLoop>(2.4801587325533363e-05));
  p = __builtin_fma(p, r, k64<kInLoop>(0.00019841269874800493));
  p = __builtin_fma(p, r, k64<kInLoop>(0.0013888888888883752));
  p = __builtin_fma(p, r, k64<kInLoop>(0.008333333333326141));
  p = __builtin_fma(p, r, k64<kInLoop>(0.04166666666666667));
  p = __builtin_fma(p, r, k64<kInLoop>(0.1666666666666667));
  p = __builtin_fma(p, r, k64<kInLoop>(0.5));
  return p;
}

// exp(x) for finite x: 2^k exp(r), |r| <= ln 2 / 2. Overflow gives inf,
// underflow a denormal or 0, as the scaling by 2^k rounds them.
template <bool kInLoop = false>
__device__ __forceinline__ double exp64(double x) {
#pragma clang fp contract(off)
  const double dk = __builtin_rint(x * k64<kInLoop>(1.4426950408889634));
  double r = __builtin_fma(-dk, k64<kInLoop>(0x1.62e42fefa39efp-1), x);
  r = __builtin_fma(-dk, k64<kInLoop>(0x1.abc9e3b39803fp-56), r);
  const double p = exp_poly<kInLoop>(r);
  const double k = __builtin_fmin(__builtin_fmax(dk, -4000.0), 4000.0);
  return __builtin_amdgcn_ldexp(1.0 + __builtin_fma(r * r, p, r), (int)k);
}

// tanh(x) for every x: E / (E + 2) with E = e^(2 |x|) - 1 = (2^k - 1) + 2^k p,
// p = e^r - 1 as in exp64, which keeps small arguments' relative precision; r, p,
// E and E + 2 come each with the part that its rounding cuts off, and the
// quotient's one residual takes those in: 0.81 ulp (2.6 without them; the device
// library's 0.86). Beyond |x| = 20 the quotient rounds to 1.
template <bool kInLoop = false>
__device__ __forceinline__ double tanh64(double x) {
#pragma clang fp contract(off)
  const double ax = __builtin_fabs(x), y = 2.0 * (ax > 20.0 ? 20.0 : ax);  // a NaN stays one
  const double dk = __builtin_rint(y * k64<kInLoop>(1.4426950408889634));
  const double r1 = __builtin_fma(-dk, k64<kInLoop>(0x1.62e42fefa39efp-1), y);  // exact
  const double r = __builtin_fma(-dk, k64<kInLoop>(0x1.abc9e3b39803fp-56), r1);
  const double rl = __builtin_fma(-dk, k64<kInLoop>(0x1.abc9e3b39803fp-56), r1 - r);
  const double z = r * r, c = exp_poly<kInLoop>(r);
  const double p = __builtin_fma(z, c, r), pl = __builtin_fma(z, c, r - p) + rl;
  const double t = __builtin_amdgcn_ldexp(1.0, (int)dk), a = t - 1.0;
  const double e = __builtin_fma(t, p, a), el = __builtin_fma(t, pl, __builtin_fma(t, p, a - e));
  const double d = e + 2.0, b = d - e, dl = el + ((e - (d - b)) + (2.0 - b));
  double q = __builtin_amdgcn_rcp(d);
  q = __builtin_fma(__builtin_fma(-d, q, 1.0), q, q);
  const double q0 = e * q;
  q = __builtin_fma(__builtin_fma(-d, q0, e) + __builtin_fma(-q0, dl, el), q, q0);
  return __builtin_copysign(q, x);
}

// sin(x) and cos(x) for |x| <= 2^52: x - k pi / 2 with pi / 2 in two parts (the
// first difference is exact), then the two polynomials, swapped and signed by
// the low bits of k, which are the last ones of k + 1.5 2^52. (Its callers'
// x = e angle is rounded to half a radian and more beyond that, at exponents above
// 10^15; those are not tested for.)
template <bool kInLoop = false>
__device__ __forceinline__ void sincos64(double x, double& sn, double& cs) {
#pragma clang fp contract(off)
  const double dk = __builtin_rint(x * k64<kInLoop>(0.63661977236758138));
  double r = __builtin_fma(-dk, k64<kInLoop>(1.5707963267948966), x);
  r = __builtin_fma(-dk, k64<kInLoop>(6.123233995736766e-17), r);
  const int k = (int)(uint32_t)__builtin_bit_cast(uint64_t, dk + k64<kInLoop>(0x1.8p52));
  const double z = r * r;
  double p = k64<kInLoop>(1.5918129294866608e-10);
  p = __builtin_fma(p, z, k64<kInLoop>(-2.5051131845003624e-08));
  p = __builtin_fma(p, z, k64<kInLoop>(2.755731610255244e-06));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.00019841269836758574));
  p = __builtin_fma(p, z, k64<kInLoop>(0.008333333333330948));
  p = __builtin_fma(p, z, k64<kInLoop>(-0.16666666666666666));
  const double s = __builtin_fma(r * z, p, r);
  double c = k64<kInLoop>(-1.1382632425521717e-11);
  c = __builtin_fma(c, z, k64<kInLoop>(2.08761462684032e-09));
  c = __builtin_fma(c, z, k64<kInLoop>(-2.7557317271729793e-07));
  c = __builtin_fma(c, z, k64<kInLoop>(2.480158729876569e-05));
  c = __builtin_fma(c, z, k64<kInLoop>(-0.0013888888888887398));
  c = __builtin_fma(c, z, k64<kInLoop>(0.041666666666666664));
  c = __builtin_fma(z, __builtin_fma(z, c, -0.5), 1.0);
  const double a = (k & 1) ? c : s, b = (k & 1) ? s : c;
  sn = (k & 2) ? -a : a;
  cs = ((k + 1) & 2) ? -b : b;
}

}  // namespace qj
