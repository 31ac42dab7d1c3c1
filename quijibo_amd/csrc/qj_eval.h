// FP64 evaluation of the map at one point, shared by the field kernels and
// the non-linear mesher (OPTIMIZE_3D.cpp:1317-1362, TRIANGLE_MESH.cpp:1755-1795).
#pragma once
#include <float.h>

#include <type_traits>

#include "qj_internal.h"
#include "qj_math64.h"
#include "qj_quat.h"

namespace qj {

constexpr double kBlackHole = 10.0 * (double)FLT_MIN;  // 10 * REAL_MIN, SETTINGS.h:58, OPTIMIZE_3D.cpp:1358

// ---------------------------------------------------------------- FP64 method

// POLYNOMIAL_4D::evaluateScaledPowerFactored (POLYNOMIAL_4D.cpp:912-923)
// Once a component of the running product is NaN every later product is NaN
// in all four components (each output component reads all four inputs), and
// so are T B^-1 and |q|: the loop can stop there with the same F.
__device__ __forceinline__ bool has_nan(const q64& q) { return isnan(q.w) || isnan(q.x) || isnan(q.y) || isnan(q.z); }

// How term64 takes (q - r)^e:
//   kPolar      QUATERNION::pow's polar form as written, with the device library's
//               functions, for every exponent (QUATERNION.cpp:375-393): the Lagrange
//               order, and the sampled cross-check, whose evaluator shares nothing
//               with the other two modes but the roots
//   kExactInt   exponents exactly 1 and 2 as b and b*b, others by polar64
//   kExactOnly  every exponent is 1 or 2 (the caller checked), no polar code
// All agree to a few ulps per term and keep the polar form's special cases:
// b = 0 gives NaN, v = 0 gives (|w|^e, +0 * v).
enum PowMode { kPolar = 0, kExactInt = 1, kExactOnly = 2 };

// f on roots r[i], r[i + 1], ... r[end - 1] in order, the loads of four at once:
// the terms branch on the exponent, which keeps the compiler from hoisting the
// next root's load, which then costs its latency where few waves share a SIMD
// (40,000 points, 64+64 roots, 3 iterations: 107 to 75 us; bisection of a 256^3
// mesh's vertices 277 to 204 us a slab; 256^3 cells, 32+32 roots 3.7 to 3.3 ms).
// Only for scalar loads: per-lane pointers would hold the four in vector registers.
template <class RP, class F>
__device__ __forceinline__ void each_root(RP r, int i, int end, F f) {
#pragma unroll 1
  for (; std::is_same_v<RP, ConstRoots> && i + 4 <= end; i += 4) {  // roots in scalar registers
    const RootRec64 a = load_root64(r + i), b = load_root64(r + i + 1), c = load_root64(r + i + 2),
                    d = load_root64(r + i + 3);
    f(a);
    f(b);
    f(c);
    f(d);
  }
#pragma unroll 1
  for (; i < end; i++) f(load_root64(r + i));
}

// The exact forms' arithmetic with every rounding fixed by the source
// (explicit fused multiply-adds, contraction off), so that the fast and the
// guarded product below, and every kernel that inlines them, round alike.
__device__ __forceinline__ q64 qsub64x(const q64& a, const RootRec64& r) {
#pragma clang fp contract(off)
  return q64{a.w - r.w, a.x - r.x, a.y - r.y, a.z - r.z};
}
__device__ __forceinline__ double partial64(const q64& b) {
#pragma clang fp contract(off)
  return __builtin_fma(b.z, b.z, __builtin_fma(b.y, b.y, b.x * b.x));
}
__device__ __forceinline__ q64 square64(const q64& b, double partial) {
#pragma clang fp contract(off)
  const double t = 2.0 * b.w;
  return q64{__builtin_fma(b.w, b.w, -partial), t * b.x, t * b.y, t * b.z};
}
// operator*(QUATERNION, QUATERNION) (QUATERNION.cpp:154-162), same term order
__device__ __forceinline__ q64 qmul64x(const q64& l, const q64& r) {
#pragma clang fp contract(off)
  q64 f;
  f.x = __builtin_fma(l.w, r.x, __builtin_fma(r.w, l.x, __builtin_fma(-l.z, r.y, l.y * r.z)));
  f.y = __builtin_fma(l.w, r.y, __builtin_fma(r.w, l.y, __builtin_fma(-l.x, r.z, l.z * r.x)));
  f.z = __builtin_fma(l.w, r.z, __builtin_fma(r.w, l.z, __builtin_fma(-l.y, r.x, l.x * r.y)));
  f.w = __builtin_fma(-l.z, r.z, __builtin_fma(-r.y, l.y, __builtin_fma(-l.x, r.x, l.w * r.w)));
  return f;
}

// left * inverse(right) (QUATERNION.cpp:167-182) and magnitude, same term order
__device__ __forceinline__ double norm64x(const q64& q) {
#pragma clang fp contract(off)
  return __builtin_fma(q.z, q.z, __builtin_fma(q.y, q.y, __builtin_fma(q.x, q.x, q.w * q.w)));
}
__device__ __forceinline__ double qmag64x(const q64& q) { return sqrt(norm64x(q)); }
__device__ __forceinline__ q64 qdiv64x(const q64& l, const q64& r) {
#pragma clang fp contract(off)
  const double inv = 1.0 / norm64x(r);
  return qmul64x(l, q64{r.w * inv, -r.x * inv, -r.y * inv, -r.z * inv});
}

__device__ __forceinline__ bool is_one(double e) { return __builtin_bit_cast(unsigned long long, e) == 0x3FF0000000000000ull; }
__device__ __forceinline__ bool is_two(double e) { return __builtin_bit_cast(unsigned long long, e) == 0x4000000000000000ull; }

// QUATERNION::pow (QUATERNION.cpp:375-393) in polar form with qj_math64.h's
// functions, as the unit part (cos m, sin m v / |v|), m = e angle(|v|, w), and
// ln |b^e| = e log|b|. Its guards carry over: b = 0 gives NaN, v = 0 a positive
// real result, m <= 0 drops the imaginary part. Bases and vector parts whose
// squares would leave FP64's normal range are scaled by a power of two first.
// The angle comes from |v| and w directly where the reference takes
// acos(w / |b|), which loses half its digits next to the real axis.
// slope: m / |v|, the factor that the reference multiplies |b^e| by first.
// kPlain: outside the extended range a base whose square is 0 or infinite in
// FP64 gives what the reference's |b| of 0 or infinity gives: NaN or, where w^2
// alone is infinite, an angle of pi / 2 and a magnitude of infinity or 0.
template <bool kPlain>
__device__ __forceinline__ q64 polar_unit(q64 b, double e, double& ln, double& slope) {
#pragma clang fp contract(off)
  double partial = partial64(b);
  double n2 = __builtin_fma(b.w, b.w, partial);
  double lnoff = 0.0, vscale = 1.0;  // 1 / the scale of v
  slope = 0.0;
  if (__builtin_expect(!(partial >= 0x1p-900 && n2 <= 0x1p900), 0)) {
    if (kPlain && (n2 == 0.0 || n2 == __builtin_inf())) {
      const bool real = partial > 0.0 && partial < __builtin_inf() && e != 0.0;
      b.w = 0.0;
      lnoff = __builtin_copysign(800.0, e);
      n2 = real ? 1.0 : __builtin_nan("");
    } else if (n2 < 0x1p-900 || n2 > 0x1p900) {
      const double s = n2 < 1.0 ? 0x1p500 : 0x1p-500;
      b = q64{b.w * s, b.x * s, b.y * s, b.z * s};
      lnoff = e * (n2 < 1.0 ? -346.57359027997264 : 346.57359027997264);  // -+500 ln 2
      partial = partial64(b);
      n2 = __builtin_fma(b.w, b.w, partial);
    }
    if (!(n2 > 0.0 && n2 < __builtin_inf())) {
      const double nan = __builtin_nan("");
      ln = nan;
      return q64{nan, nan, nan, nan};
    }
    if (!(partial >= 0x1p-900)) {
      if (!(partial > 0.0)) {
        // v = 0 (or its square is): a positive real, +0 * v
        ln = __builtin_fma(e * 0.5, log64<true>(n2), lnoff);
        return q64{1.0, 0.0 * b.x, 0.0 * b.y, 0.0 * b.z};
      }
      vscale = 0x1p-500;
      b.x *= 0x1p500;
      b.y *= 0x1p500;
      b.z *= 0x1p500;
      partial = partial64(b);
    }
  }
  double vm, vi;
  sqrt_rsqrt64(partial, vm, vi);
  const double m = e * angle64<true>(vm * vscale, b.w);
  double s, c;
  sincos64<true>(m, s, c);
  ln = __builtin_fma(e * 0.5, log64<true>(n2), lnoff);
  const double f = m > 0.0 ? s * vi : 0.0;
  slope = m * vi;
  return q64{c, f * b.x, f * b.y, f * b.z};
}
// b^e itself: about 150 instructions against 350 with the device library's acos,
// log, exp, sincos, square roots and divisions. The reference's imaginary part
// is ((m / |v|) |b^e|) (1 / m) sin m v, so it overflows where (m / |v|) |b^e|
// does, some bits before |b^e|: those terms come out infinite here as well.
__device__ __forceinline__ q64 polar64(const q64& b, double e) {
#pragma clang fp contract(off)
  double ln, slope;
  const q64 u = polar_unit<true>(b, e, ln, slope);
  const double ex = exp64<true>(ln);
  const double im = slope * ex < __builtin_inf() ? ex : __builtin_inf();
  return q64{u.w * ex, u.x * im, u.y * im, u.z * im};
}

// (q - r)^e with the special cases (guarded form).
template <int kPow>
__device__ __forceinline__ q64 term64(const RootRec64& r, const q64& q) {
  if (kPow == kPolar) return qpow(qsub(q, q64{r.w, r.x, r.y, r.z}), r.e);
  const q64 b = qsub64x(q, r);
  if (kPow == kExactOnly || is_one(r.e) || is_two(r.e)) {
    const double partial = partial64(b);
    if (!(partial + b.w * b.w > 0.0)) {
      const double nan = __builtin_nan("");
      return q64{nan, nan, nan, nan};
    }
    if (!(partial > 0.0)) {
      const double m = is_one(r.e) ? fabs(b.w) : b.w * b.w;
      return q64{m, 0.0 * b.x, 0.0 * b.y, 0.0 * b.z};
    }
    if (is_one(r.e)) return b;
    return square64(b, partial);
  }
  return polar64(b, r.e);
}

// (q - r)^e without the special cases; vx keeps the smallest |b.x|. With
// |b.x| >= kExactMinX for every root, partial >= 1e-300 > 0 and term64 takes
// exactly these branches.
constexpr double kExactMinX = 1e-150;
// vx = min(vx, |x|) in one instruction (fmin would canonicalise both inputs
// first); a NaN x leaves vx unchanged, and a NaN product is caught by has_nan.
__device__ __forceinline__ void min_abs64(double& vx, double x) {
  asm("v_min_f64 %0, %1, |%2|" : "=v"(vx) : "v"(vx), "v"(x));
}
template <int kPow>
__device__ __forceinline__ q64 term64_plain(const RootRec64& r, const q64& q, double& vx) {
  const q64 b = qsub64x(q, r);
  min_abs64(vx, b.x);
  if (is_one(r.e)) return b;
  if (kPow == kExactOnly || is_two(r.e)) return square64(b, partial64(b));
  return polar64(b, r.e);
}
// t <- t * (q - r)^e, the product inside each kind's branch (no copies at the merge)
template <int kPow>
__device__ __forceinline__ void apply64_plain(q64& t, const RootRec64& r, const q64& q, double& vx) {
  const q64 b = qsub64x(q, r);
  min_abs64(vx, b.x);
  if (is_one(r.e)) {
    t = qmul64x(t, b);
  } else if (kPow == kExactOnly || is_two(r.e)) {
    t = qmul64x(t, square64(b, partial64(b)));
  } else {
    t = qmul64x(t, polar64(b, r.e));
  }
}

template <int kPow, class RP>
__device__ __forceinline__ q64 poly64_guarded(RP r, int n, const q64& q) {
  q64 res = term64<kPow>(load_root64(r), q);
  for (int i = 1; i < n; i++) {
    res = kPow == kPolar ? qmul(res, term64<kPow>(load_root64(r + i), q))
                         : qmul64x(res, term64<kPow>(load_root64(r + i), q));
    if ((i & 7) == 0 && has_nan(res)) {
      const double nan = __builtin_nan("");
      return q64{nan, nan, nan, nan};
    }
  }
  return res;
}

// The factored product. The exact modes first run it without the special
// cases (no per-term tests, no NaN stand-ins), and only a point where some
// |b.x| < kExactMinX (a special case may apply) runs the guarded form again;
// otherwise the two are the same arithmetic.
template <int kPow = kPolar, class RP = const RootRec64*>
__device__ __forceinline__ q64 poly64(RP r, int n, const q64& q) {
  if (kPow == kPolar) return poly64_guarded<kPow>(r, n, q);
  double vx = __builtin_inf();
  q64 res = term64_plain<kPow>(load_root64(r), q, vx);
  bool nan = false;
  if constexpr (kPow == kExactOnly) {
    for (int i = 1; i < n && !nan; i += 8) {
      const int end = i + 8 < n ? i + 8 : n;
      each_root(r, i, end, [&](const RootRec64& t) { apply64_plain<kPow>(res, t, q, vx); });
      nan = end == i + 8 && has_nan(res);
    }
  } else {
    for (int i = 1; i < n; i++) {
      apply64_plain<kPow>(res, load_root64(r + i), q, vx);
      if ((i & 7) == 0 && has_nan(res)) {
        nan = true;
        break;
      }
    }
  }
  if (!(vx >= kExactMinX)) return poly64_guarded<kPow>(r, n, q);
  if (nan) {
    const double n4 = __builtin_nan("");
    return q64{n4, n4, n4, n4};
  }
  return res;
}

__device__ __forceinline__ bool finite4(const q64& q) {
  return isfinite(q.w) && isfinite(q.x) && isfinite(q.y) && isfinite(q.z);
}

// ---------------------------------------------------------------- the last iteration

// The last iteration needs |q| alone, and norms are multiplicative: |T|^2 =
// prod |q - r_i|^(2 e_i). magnitude64 keeps a product of |q - r|^2 over the
// exponents 1 and 2 as N 2^E (renormalised every kMagGroup terms), the sum L of
// e log|q - r|^2 over the others, the extremes of E and the sum S of
// |e log|q - r|^2|: 10 instructions per exponent-1 term against 24 for the
// quaternion product, 40 per general term against 170. ok stays set when
// no running product can have left FP64's range, so that the product in
// reference order gives the same magnitude; the caller forms it where not.
constexpr int kMagGroup = 8;
constexpr double kMagMaxTermBits = 50.0;  // 2 x 8 x 50 bits in a group stay in range
struct Mag64 {
  double N = 1.0, L = 0.0, S = 0.0;
  int E = 0, hi = 0, lo = 0;
  bool ok = true;
};
template <int kPow, class RP>
__device__ __forceinline__ Mag64 magnitude64(RP r, int n, const q64& q, int margin) {
#pragma clang fp contract(off)
  Mag64 m;
  double big = 0.0;
  int low = 0;
  auto term = [&](const RootRec64& t) {
    const q64 b = qsub64x(q, t);
    const double n2 = __builtin_fma(b.w, b.w, partial64(b));
    if (is_one(t.e)) {
      m.N *= n2;
    } else if (kPow == kExactOnly || is_two(t.e)) {
      m.N *= n2 * n2;
    } else {
      const double l = log64<true>(n2);
      m.L = __builtin_fma(t.e, l, m.L);
      m.S = __builtin_fma(t.e, fabs(l), m.S);
      big = fabs(l) > big ? fabs(l) : big;
      m.ok = m.ok && t.e >= 0.0;  // pow drops the imaginary part of a negative power
    }
  };
  auto renorm = [&]() {
    const int k = __builtin_amdgcn_frexp_exp(m.N);
    m.N = __builtin_amdgcn_ldexp(m.N, -k);
    low = min(low, k);
    m.E += k;
    m.hi = max(m.hi, m.E);
    m.lo = min(m.lo, m.E);
  };
  int i = 0;
  // four copies where a term is a few instructions; one of the general term otherwise
  while (i < n) {
    const int end = i + kMagGroup < n ? i + kMagGroup : n;
    if (kPow == kExactOnly) {
      each_root(r, i, end, term);
    } else {
#pragma unroll 1
      for (int j = i; j < end; j++) term(load_root64(r + j));
    }
    i = end;
    renorm();
  }
  // a group that ends above 2^(margin - 1000) never fell below 2^-1000 (each of
  // its terms is at most 2^(margin / kMagGroup)); log64 of a zero, denormal or
  // infinite norm is beyond +-700
  m.ok = m.ok && m.N > 0.0 && m.N < __builtin_inf() && low > margin - 1000 && big < 600.0;
  return m;
}

// top and bottom through one copy of the loop's code
template <int kPow, class RP>
__device__ __forceinline__ void both_magnitudes(const MapArgs& a, RP roots, const q64& q, int margin, Mag64& T,
                                                Mag64& B) {
  if constexpr (kPow == kExactOnly) {
    T = magnitude64<kPow>(roots, a.nt, q, margin);
    if (a.nb > 0) B = magnitude64<kPow>(roots + a.nt, a.nb, q, margin);
    return;
  }
#pragma unroll 1
  for (int p = 0; p < 2; p++) {
    const Mag64 m = magnitude64<kPow>(p ? roots + a.nt : roots, p ? a.nb : a.nt, q, margin);
    if (p) B = m;
    else T = m;
    if (a.nb == 0) break;
  }
}

// log|q| after the last iteration from q before it; false when some product may
// leave FP64's range (or the scaling is not an ordinary positive number).
template <int kPow, class RP>
__device__ __forceinline__ bool last64(const MapArgs& a, RP roots, const q64& q, double& F) {
#pragma clang fp contract(off)
  if (!(a.term_bits <= kMagMaxTermBits && a.exp_scaling >= 0x1p-300 && a.exp_scaling <= 0x1p300)) return false;
  const int margin = (int)(2.0 * kMagGroup * a.term_bits) + 1;
  Mag64 T, B;
  both_magnitudes<kPow>(a, roots, q, margin, T, B);
  if (!T.ok || !B.ok) return false;
  // in bits of |T|^2: FP64's range less a group's growth and the general terms' share
  const double lim = 2000.0 - margin, bits = 1.4426950408889634;
  double s = T.S * bits, l = 0.5 * T.L, x = T.N;
  bool ok = T.hi + s < lim && s - T.lo < lim;
  int e = T.E;
  if (a.nb > 0) {
    const double sb = B.S * bits;
    // and |B|^2 itself, which the quotient divides by, within 2^+-950: E and L
    ok = ok && B.hi + sb < lim && sb - B.lo < lim && fabs((double)B.E + B.L * bits) < 950.0;
    if (!ok) return false;
    x = div64(x, B.N);
    e -= B.E;
    l = __builtin_fma(-0.5, B.L, l);
  }
  x = x * a.exp_scaling * a.exp_scaling;
  const int k = __builtin_amdgcn_frexp_exp(x);
  // |q|^2 likewise, from the signed logarithms: by the sum of their sizes, 24^3 with
  // 32+32 real exponents and three iterations took the products after the norms,
  // 226 us; 119 now
  const double ek = (double)(e + k);
  if (!(ok && fabs(ek) < 950.0 && fabs(__builtin_fma(2.0 * bits, l, ek)) < 950.0)) return false;
  F = __builtin_fma(0.5, log64(__builtin_amdgcn_ldexp(x, e)), l);
  return true;
}

struct Res64 {
  double F;
  int iters;
  bool written;
  bool overflow;
};

// RATIONAL_4D::evaluateLagrange (RATIONAL_4D.cpp:27-88): with bottom roots,
// r = 1, then r = (r t_i) / b_i for the paired roots, then the leftover top
// terms multiplied or bottom terms divided; the factored top product otherwise.
template <int kPow = kPolar, class RP = const RootRec64*>
__device__ __forceinline__ q64 lagrange64(RP roots, int nt, int nb, const q64& q) {
  if (nb == 0) return poly64<kPow>(roots, nt, q);
  const RP bot = roots + nt;
  q64 r{1.0, 0.0, 0.0, 0.0};
  const int same = nt < nb ? nt : nb;
  for (int i = 0; i < same; i++) {
    const RootRec64 t = load_root64(roots + i), d = load_root64(bot + i);  // d's load behind t's term
    r = qmul(r, term64<kPow>(t, q));
    r = qdiv(r, term64<kPow>(d, q));
  }
  for (int i = same; i < nt; i++) r = qmul(r, term64<kPow>(load_root64(roots + i), q));
  for (int i = same; i < nb; i++) r = qdiv(r, term64<kPow>(load_root64(bot + i), q));
  return r;
}

// One voxel of the map in Lagrange order (QJ_MAP_LAGRANGE), polar powers. The
// API takes it with neither the AP flags nor the extended range; the mesher
// evaluates it itself.
template <class RP = const RootRec64*>
__device__ __forceinline__ Res64 eval64_lagrange(const MapArgs& a, RP roots, q64 q) {
  Res64 r{0.0, 0, true, false};
  double magnitude = qmag(q);
  int it = 0;
  while (magnitude < a.escape && it < a.max_iter) {
    q = qscale(lagrange64<kPolar>(roots, a.nt, a.nb, q), a.exp_scaling);
    magnitude = qmag(q);
    it++;
    r.iters++;
    if ((a.flags & QJ_MAP_BLACK_HOLE) && magnitude < kBlackHole) it = a.max_iter;
  }
  r.F = log(magnitude);
  return r;
}

// One voxel of computeLogScaledPowerRationalMap (OPTIMIZE_3D.cpp:1317-1362) /
// computeRationalMapAP's first pass (:1423-1475). Overflow detection replaces
// fetestexcept(FE_OVERFLOW): any non-finite T, B, |B|^2, quotient or |q|.
template <int kPow = kPolar, class RP = const RootRec64*>
__device__ __forceinline__ Res64 eval64(const MapArgs& a, RP roots, q64 q) {
  Res64 r{0.0, 0, true, false};
  // the exact modes round alike in every kernel (explicit fused multiply-adds)
  auto mag = [](const q64& v) { return kPow == kPolar ? qmag(v) : qmag64x(v); };
  double magnitude = mag(q);
  if ((a.flags & QJ_MAP_SKIP_ORIGIN) && magnitude < 1e-8) {
    r.written = false;
    return r;
  }
  const bool adaptive = (a.flags & QJ_MAP_ADAPTIVE) != 0;
  int it = 0;
  // one iteration by the products
  auto step = [&]() {
    q64 T, B;
    bool nan_top = false;
    if constexpr (kPow == kExactOnly) {
      T = poly64<kPow>(roots, a.nt, q);
      if (a.nb > 0) {
        // T B^-1 is all-NaN whatever B is: B is not evaluated
        nan_top = has_nan(T) && !adaptive;
        if (!nan_top) B = poly64<kPow>(roots + a.nt, a.nb, q);
      }
    } else {
#pragma unroll 1
      for (int p = 0; p < 2; p++) {  // one copy of the loop's code
        const q64 v = poly64<kPow>(p ? roots + a.nt : roots, p ? a.nb : a.nt, q);
        if (p) B = v;
        else T = v;
        if (a.nb == 0) break;
        nan_top = has_nan(T) && !adaptive;
        if (nan_top) break;
      }
    }
    it++;
    r.iters++;
    if (a.nb > 0) {
      if (nan_top) {
        const double nan = __builtin_nan("");
        q = q64{nan, nan, nan, nan};
        magnitude = nan;
        return;
      }
      q = kPow == kPolar ? qdiv(T, B) : qdiv64x(T, B);
      if (adaptive) {
        const double m2 = B.w * B.w + B.x * B.x + B.y * B.y + B.z * B.z;
        r.overflow |= !(finite4(T) && finite4(B) && isfinite(m2) && finite4(q));
      }
    } else {
      q = T;
      if (adaptive) r.overflow |= !finite4(T);
    }
    q = qscale(q, a.exp_scaling);
    magnitude = mag(q);
    if (adaptive && !isfinite(magnitude)) r.overflow = true;
    if ((a.flags & QJ_MAP_BLACK_HOLE) && magnitude < kBlackHole) it = a.max_iter;
  };
  if constexpr (kPow == kExactOnly) {
    // the loop without the last iteration's code, each polynomial with its own
    // copy (200^3, one root, ten iterations: 321 -> 203 us)
    while (magnitude < a.escape && it + 1 < a.max_iter) step();
    if (magnitude < a.escape && it < a.max_iter) {
      if (last64<kPow>(a, roots, q, r.F)) {
        r.iters++;
        return r;
      }
      step();
    }
  } else {
    while (magnitude < a.escape && it < a.max_iter) {
      if (kPow != kPolar && it + 1 == a.max_iter && last64<kPow>(a, roots, q, r.F)) {
        r.iters++;
        return r;
      }
      step();
    }
  }
  r.F = log(magnitude);
  return r;
}


// ---------------------------------------------------------------- extended range

// A quaternion times 2^e. Normalised so the largest |component| is in [0.5, 1).
struct xq {
  q64 m;
  int e;
};
__device__ __forceinline__ void xnorm(xq& v) {
  const double mx = fmax(fmax(fabs(v.m.w), fabs(v.m.x)), fmax(fabs(v.m.y), fabs(v.m.z)));
  if (mx > 0.0 && isfinite(mx)) {
    int k;
    (void)frexp(mx, &k);
    v.m.w = ldexp(v.m.w, -k);
    v.m.x = ldexp(v.m.x, -k);
    v.m.y = ldexp(v.m.y, -k);
    v.m.z = ldexp(v.m.z, -k);
    v.e += k;
  }
}
// QUATERNION::pow (QUATERNION.cpp:375-393) with exps = exp(e log|q| + lnoff)
// kept as mantissa * 2^k (the AP map's re-pass and the cross-check); lnoff
// carries the scale of a normalised base (e k ln 2 for a base m 2^k: the angle
// does not depend on the scale).
__device__ __forceinline__ xq xpow(const q64& q, double e, double lnoff = 0.0) {
  const double partial = q.x * q.x + q.y * q.y + q.z * q.z;
  const double qMagnitude = sqrt(partial + q.w * q.w);
  const double vMagnitude = sqrt(partial);
  const double vMagnitudeInv = (vMagnitude > 0.0) ? 1.0 / vMagnitude : 0.0;
  const double scale = e * acos(q.w / qMagnitude) * vMagnitudeInv;
  const double magnitude = scale * vMagnitude;
  const double magnitudeInv = (magnitude > 0.0) ? 1.0 / magnitude : 0.0;
  const double lnE = e * log(qMagnitude) + lnoff;
  int k = 0;
  double em;
  if (isfinite(lnE)) {
    k = (int)floor(lnE * 1.4426950408889634);
    em = exp(lnE - k * 0.6931471805599453);
  } else {
    em = exp(lnE);
  }
  double s, c;
  sincos(magnitude, &s, &c);
  const double scale2 = scale * em * magnitudeInv * s;
  xq r{{em * c, scale2 * q.x, scale2 * q.y, scale2 * q.z}, k};
  xnorm(r);
  return r;
}

// v <- v e^ln: the power of two to the exponent, the rest to the mantissa
__device__ __forceinline__ void scale_ext(xq& v, double ln) {
#pragma clang fp contract(off)
  const double k = __builtin_rint(ln * 1.4426950408889634);
  v.m = qscale(v.m, exp64(__builtin_fma(-k, 0x1.abc9e3b39803fp-56, __builtin_fma(-k, 0x1.62e42fefa39efp-1, ln))));
  v.e += (int)k;
}

// (q - r)^e with a separate binary exponent, for QJ_MAP_EXTENDED_RANGE: the
// base is normalised first, so neither its square nor the polar magnitude
// leaves FP64's range; exponents 1 and 2 (kPow != kPolar) as the exact
// products with the polar form's special cases (b = 0: NaN; v = 0:
// (|w|^e, +0 v)), decided on the normalised base as long double would.
template <int kPow>
__device__ __forceinline__ xq term_ext(const RootRec64& r, const q64& q) {
  xq n{qsub64x(q, r), 0};
  xnorm(n);
  if (kPow == kPolar) return xpow(n.m, r.e, r.e * (double)n.e * 0.6931471805599453);
  if (kPow != kExactOnly && !is_one(r.e) && !is_two(r.e)) {
    double ln, slope;
    xq v{polar_unit<false>(n.m, r.e, ln, slope), 0};
    ln = __builtin_fma(r.e * (double)n.e, 0.6931471805599453, ln);
    scale_ext(v, ln);
    xnorm(v);
    return v;
  }
  const double partial = partial64(n.m);
  if (!(partial + n.m.w * n.m.w > 0.0)) {
    const double nan = __builtin_nan("");
    return xq{{nan, nan, nan, nan}, 0};
  }
  if (!(partial > 0.0)) {
    xq v = is_one(r.e) ? xq{{fabs(n.m.w), 0.0 * n.m.x, 0.0 * n.m.y, 0.0 * n.m.z}, n.e}
                       : xq{{n.m.w * n.m.w, 0.0 * n.m.x, 0.0 * n.m.y, 0.0 * n.m.z}, 2 * n.e};
    xnorm(v);
    return v;
  }
  if (is_one(r.e)) return n;
  xq v{square64(n.m, partial), 2 * n.e};
  xnorm(v);
  return v;
}

template <int kPow, class RP>
__device__ __forceinline__ xq poly_ext(RP r, int n, const q64& q) {
  xq res = term_ext<kPow>(load_root64(r), q);
  for (int i = 1; i < n; i++) {
    const xq t = term_ext<kPow>(load_root64(r + i), q);
    res.m = qmul64x(res.m, t.m);
    res.e += t.e;
    xnorm(res);
  }
  return res;
}

// The same product with the exponent taken out every kExtGroup terms instead
// of three times per term (base, square, product): 27 instead of about 75
// instructions per exponent-1 term, the same bits. In a group the terms are at
// most 2^term_bits and, with |b.x| >= kExtMinX, exponents 1 and 2 at least
// 2^-100, so a product of 8 that starts in [1/2, 2) stays within 2^-801 and
// 2^802 and scaling by a power of two loses nothing. General exponents multiply
// the unit part and add their logarithm to ln. False when some term is outside
// that (the caller takes poly_ext).
constexpr int kExtGroup = 8;
constexpr double kExtMaxTermBits = 100.0, kExtMinX = 0x1p-50;
template <int kPow, class RP>
__device__ __forceinline__ bool poly_ext_grouped(RP r, int n, const q64& q, xq& res, double& ln) {
#pragma clang fp contract(off)
  double vx = __builtin_inf();
  bool ok = true;
  q64 t{1.0, 0.0, 0.0, 0.0};
  res.e = 0;
  auto term = [&](const RootRec64& rt) {
    const q64 b = qsub64x(q, rt);
    min_abs64(vx, b.x);
    if (is_one(rt.e)) {
      t = qmul64x(t, b);
    } else if (kPow == kExactOnly || is_two(rt.e)) {
      t = qmul64x(t, square64(b, partial64(b)));
    } else {
      double l, slope;
      t = qmul64x(t, polar_unit<false>(b, rt.e, l, slope));
      ln += l;
      ok = ok && rt.e > 0.0;  // cos m of a negative power can be 0 to any depth
    }
  };
  auto renorm = [&]() {
    xq v{t, 0};
    xnorm(v);
    t = v.m;
    res.e += v.e;
  };
  // the first term without a product by 1 (it would turn -0 components into +0)
  {
    const RootRec64 r0 = load_root64(r);
    if (is_one(r0.e)) {
      t = qsub64x(q, r0);
      min_abs64(vx, t.x);
    } else {
      term(r0);
    }
  }
  int i = 1;
  renorm();
  while (i < n) {
    const int end = i + kExtGroup < n ? i + kExtGroup : n;
    if (kPow == kExactOnly) {
      each_root(r, i, end, term);
    } else {
#pragma unroll 1
      for (int j = i; j < end; j++) term(load_root64(r + j));
    }
    i = end;
    renorm();
  }
  res.m = t;
  return ok && vx >= kExtMinX;
}

// log|q| after the last iteration in the extended range (see last64): no
// product can leave the range here, only the norms have to be ordinary numbers.
template <int kPow, class RP>
__device__ __forceinline__ bool last64e(const MapArgs& a, RP roots, const q64& q, double& F) {
#pragma clang fp contract(off)
  if (!(a.term_bits <= kMagMaxTermBits && a.exp_scaling >= 0x1p-300 && a.exp_scaling <= 0x1p300)) return false;
  const int margin = (int)(2.0 * kMagGroup * a.term_bits) + 1;
  Mag64 T, B;
  both_magnitudes<kPow>(a, roots, q, margin, T, B);
  if (!T.ok || !B.ok) return false;
  double l = 0.5 * T.L, x = T.N;
  int e = T.E;
  if (a.nb > 0) {
    x = div64(x, B.N);
    e -= B.E;
    l = __builtin_fma(-0.5, B.L, l);
  }
  x = x * a.exp_scaling * a.exp_scaling;
  // a magnitude near 1 keeps its relative precision (one logarithm of the whole)
  const bool near = e > -300 && e < 300;
  l = __builtin_fma(0.5, log64(near ? __builtin_amdgcn_ldexp(x, e) : x), l);
  F = near ? l : __builtin_fma((double)e, 0.34657359027997264, l);
  return true;
}

// One voxel with the range of the reference's default build (Real = long
// double, SETTINGS.h:10; QJ_MAP_EXTENDED_RANGE): the factored products, the
// quotient and |q| are FP64 mantissas with separate binary exponents, so
// nothing overflows or underflows where x87 long double does not. The
// escape and black-hole tests compare the FP64 value of |q| (exact whenever
// it is representable; +inf or 0 beyond, which decides them the same way);
// F = log|mantissa| + exponent ln 2. An iterate that continues below FP64's
// range (no black-hole stop) continues from its FP64 value. kPolar: every term
// and product one by one, for the cross-check.
template <int kPow, class RP = const RootRec64*>
__device__ __forceinline__ Res64 eval64e(const MapArgs& a, RP roots, q64 q) {
  Res64 r{0.0, 0, true, false};
  auto mag = [](const q64& v) { return kPow == kPolar ? qmag(v) : qmag64x(v); };
  double magnitude = mag(q);
  if ((a.flags & QJ_MAP_SKIP_ORIGIN) && magnitude < 1e-8) {
    r.written = false;
    return r;
  }
  double logmag = log(magnitude);
  int it = 0;
  // one iteration by the products
  auto step = [&]() {
    xq v, B;
    double ln = 0.0;
    bool grouped = kPow != kPolar && a.term_bits <= kExtMaxTermBits;
    if constexpr (kPow == kExactOnly) {
      if (grouped) {
        grouped = poly_ext_grouped<kPow>(roots, a.nt, q, v, ln);
        if (a.nb > 0) grouped = poly_ext_grouped<kPow>(roots + a.nt, a.nb, q, B, ln) && grouped;
      }
    } else if (grouped) {
#pragma unroll 1
      for (int p = 0; p < 2; p++) {  // one copy of the loop's code
        xq w;
        double l = 0.0;
        grouped = poly_ext_grouped<kPow>(p ? roots + a.nt : roots, p ? a.nb : a.nt, q, w, l) && grouped;
        if (p) B = w;
        else v = w;
        ln += p ? -l : l;
        if (a.nb == 0) break;
      }
    }
    if (!grouped) {
      ln = 0.0;
#pragma unroll 1
      for (int p = 0; p < 2; p++) {
        const xq w = poly_ext<kPow>(p ? roots + a.nt : roots, p ? a.nb : a.nt, q);
        if (p) B = w;
        else v = w;
        if (a.nb == 0) break;
      }
    }
    if (a.nb > 0) {
      v.m = kPow == kPolar ? qdiv(v.m, B.m) : qdiv64x(v.m, B.m);
      v.e -= B.e;
    }
    v.m = qscale(v.m, a.exp_scaling);
    if (kPow == kExactInt && ln != 0.0) scale_ext(v, ln);  // the general terms' magnitude
    xnorm(v);
    const double mm = mag(v.m);
    logmag = __builtin_fma((double)v.e, 0.6931471805599453, log(mm));
    magnitude = ldexp(mm, v.e);
    q = q64{ldexp(v.m.w, v.e), ldexp(v.m.x, v.e), ldexp(v.m.y, v.e), ldexp(v.m.z, v.e)};
    it++;
    r.iters++;
    if ((a.flags & QJ_MAP_BLACK_HOLE) && magnitude < kBlackHole) it = a.max_iter;
  };
  if constexpr (kPow == kExactOnly) {
    while (magnitude < a.escape && it + 1 < a.max_iter) step();
    if (magnitude < a.escape && it < a.max_iter) {
      if (last64e<kPow>(a, roots, q, r.F)) {
        r.iters++;
        return r;
      }
      step();
    }
  } else {
    while (magnitude < a.escape && it < a.max_iter) {
      if constexpr (kPow != kPolar) {
        if (it + 1 == a.max_iter && last64e<kPow>(a, roots, q, r.F)) {
          r.iters++;
          return r;
        }
      }
      step();
    }
  }
  r.F = logmag;
  return r;
}

// eval64 or, with QJ_MAP_EXTENDED_RANGE, eval64e (a uniform branch where a
// wave's voxels share their map arguments).
template <int kPow, class RP = const RootRec64*>
__device__ __forceinline__ Res64 eval64_any(const MapArgs& a, RP roots, const q64& q) {
  if (a.flags & QJ_MAP_EXTENDED_RANGE) return eval64e<kPow>(a, roots, q);
  return eval64<kPow>(a, roots, q);
}

}  // namespace qj
