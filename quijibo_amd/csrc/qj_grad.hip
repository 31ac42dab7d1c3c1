// Gradient kernels.
//
// k_ap_fast, k_ap_grads: the one-iteration AP score and exponent gradients of
//   the optimizer (OPTIMIZE_3D.cpp computeScoreAP :3563, computeExpGradientAP
//   :3589-3625, computeTopGradientAP :8905-9106, computeBottomGradientAP
//   :10012, computeTop/BottomBulkScalarGradientAP :9250/:10360).
//   With one iteration only magnitudes matter. |T| = prod |b_i|^e_i, so F is a
//   sum of logarithms. Each gradient term is dSdF Re(R^-1 R'): with R = L P S B^-1
//   and R' = L (s P log b) S B^-1 every factor but log b cancels in the real part
//   (Re(x y x^-1) = Re y), which leaves s log|b_i|; the bottom formula
//   R' = T (-L (P / s) (log b)^-1 S)^-1 leaves -s log|b_j| in the same way.
//   k_ap_fast computes just that, one logarithm per cell and root. A cell whose
//   products could leave FP64's range (sum of e |log|b|| beyond kApRange, a cell
//   on a root) is left to k_ap_grads, which forms the products of the formulas
//   as they stand and redoes overflowed cells with a shared binary exponent per
//   quaternion (the reference redoes them in long double, :9011-9103); so is
//   every cell when some exponent is negative (QUATERNION::pow then drops the
//   imaginary part, and |b^e| is not |b|^e) or the exponents are so large that few
//   cells would be spared (ap_from_logs).
//   Sums are over fixed trees, so results do not depend on scheduling.
//
// k_adjoint: reverse mode through max_iter iterations of the map at points.
//   Each point is a group of 4 to 32 lanes, each lane taking a share of the
//   roots; the ordered product of the shares is a suffix scan of quaternion
//   products over the group, and each root's gradient is summed over the wave's
//   points by row swaps before one lane adds it to the block's LDS.
#include <float.h>

#include <string.h>

#include <algorithm>
#include <type_traits>

#include "qj_fp32.h"
#include "qj_geom.h"
#include "qj_internal.h"
#include "qj_math64.h"
#include "qj_quat.h"

namespace qj {

constexpr int kGBlock = 256;

// ------------------------------------------------------------ extended range

struct xq {
  q64 m;
  int e;
};
__device__ __forceinline__ xq xnorm(xq v) {
  const double mx = fmax(fmax(fabs(v.m.w), fabs(v.m.x)), fmax(fabs(v.m.y), fabs(v.m.z)));
  if (mx > 0.0 && isfinite(mx)) {
    int k;
    (void)frexp(mx, &k);
    v.m = q64{ldexp(v.m.w, -k), ldexp(v.m.x, -k), ldexp(v.m.y, -k), ldexp(v.m.z, -k)};
    v.e += k;
  }
  return v;
}
__device__ __forceinline__ xq xfrom(const q64& q) { return xnorm(xq{q, 0}); }
__device__ __forceinline__ xq mul(const xq& a, const xq& b) { return xnorm(xq{qmul(a.m, b.m), a.e + b.e}); }
__device__ __forceinline__ xq inv(const xq& a) {
  const q64 i = qinv(a.m);
  return xnorm(xq{i, -a.e});
}
__device__ __forceinline__ xq scaled(const xq& a, double s) { return xnorm(xq{qscale(a.m, s), a.e}); }
__device__ __forceinline__ double logmag(const xq& a) { return log(qmag(a.m)) + a.e * 0.6931471805599453; }
// <a,b> / <c,c> as a double
__device__ __forceinline__ double dotratio(const xq& a, const xq& b, const xq& c) {
  return qdot(a.m, b.m) / qdot(c.m, c.m) * ldexp(1.0, a.e + b.e - 2 * c.e);
}
__device__ __forceinline__ bool ok(const xq& a) {
  return isfinite(a.m.w) && isfinite(a.m.x) && isfinite(a.m.y) && isfinite(a.m.z);
}
// QUATERNION::pow with exps = exp(e log|q|) kept as mantissa * 2^k
__device__ __forceinline__ xq pw_x(const q64& q, double e) {
  const double partial = q.x * q.x + q.y * q.y + q.z * q.z;
  const double qMagnitude = sqrt(partial + q.w * q.w);
  const double vMagnitude = sqrt(partial);
  const double vMagnitudeInv = (vMagnitude > 0.0) ? 1.0 / vMagnitude : 0.0;
  const double scale = e * acos(q.w / qMagnitude) * vMagnitudeInv;
  const double magnitude = scale * vMagnitude;
  const double magnitudeInv = (magnitude > 0.0) ? 1.0 / magnitude : 0.0;
  const double lnE = e * log(qMagnitude);
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
  return xnorm(xq{{em * c, scale2 * q.x, scale2 * q.y, scale2 * q.z}, k});
}

// plain FP64 counterparts with the same interface
__device__ __forceinline__ q64 mul(const q64& a, const q64& b) { return qmul(a, b); }
__device__ __forceinline__ q64 inv(const q64& a) { return qinv(a); }
__device__ __forceinline__ q64 scaled(const q64& a, double s) { return qscale(a, s); }
__device__ __forceinline__ double logmag(const q64& a) { return log(qmag(a)); }
__device__ __forceinline__ double dotratio(const q64& a, const q64& b, const q64& c) {
  return (1.0 / qdot(c, c)) * qdot(a, b);  // (1.0 / R.dot(R)) * R.dot(Rd), OPTIMIZE_3D.cpp:8976
}
__device__ __forceinline__ bool ok(const q64& a) {
  return isfinite(a.w) && isfinite(a.x) && isfinite(a.y) && isfinite(a.z);
}
template <class Q>
__device__ __forceinline__ Q from64(const q64& q);
template <>
__device__ __forceinline__ q64 from64<q64>(const q64& q) { return q; }
template <>
__device__ __forceinline__ xq from64<xq>(const q64& q) { return xfrom(q); }
template <class Q>
__device__ __forceinline__ Q pw(const q64& b, double e);
template <>
__device__ __forceinline__ q64 pw<q64>(const q64& b, double e) { return qpow(b, e); }
template <>
__device__ __forceinline__ xq pw<xq>(const q64& b, double e) { return pw_x(b, e); }

// ------------------------------------------------------------ block reduction

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// acc[wave * K + k] += wave sum of v (lane 0 writes); K slots per wave
__device__ __forceinline__ void wave_acc(double* acc, int K, int k, double v) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) acc[(threadIdx.x >> 6) * K + k] += v;
}

// ------------------------------------------------------------ AP gradients

struct APArgs {
  MapArgs a;
  GridGeom wg;
  double alpha, thr;
  double log_c;          // log(exp_scaling)
  FastDiv div_x, div_xy;  // of the map's grid, for fewer than 2^32 cells
};

// slot layout of the partial sums
enum { SL_SCORE = 0, SL_GEXP = 1, SL_GTS = 2, SL_GBS = 3, SL_ROOTS = 4 };

// A term that came out non-finite in FP64 redone with explicit exponents from
// the same FP64 factors (the reference redoes it in long double,
// OPTIMIZE_3D.cpp:8986-8995, 9011-9103). Returns 0 if a factor itself is not finite.
__device__ __forceinline__ double top_term_x(const q64& left, const q64& power, double scalar, const q64& lg,
                                             const q64& right, const q64& T, const q64& B, double dSdF) {
  if (!(ok(left) && ok(power) && ok(right) && ok(T) && ok(B))) return 0.0;
  const xq R = mul(xfrom(T), inv(xfrom(B)));
  const xq mid = mul(scaled(xfrom(power), scalar), xfrom(lg));
  const xq Rd = mul(mul(mul(xfrom(left), mid), xfrom(right)), inv(xfrom(B)));
  const double v = dSdF * dotratio(R, Rd, R);
  return isfinite(v) ? v : 0.0;
}
__device__ __forceinline__ double bottom_term_x(const q64& left, const q64& power, double scalar, const q64& ilg,
                                                const q64& right, const q64& T, const q64& B, double dSdF) {
  if (!(ok(left) && ok(power) && ok(right) && ok(T) && ok(B) && ok(ilg))) return 0.0;
  const xq R = mul(xfrom(T), inv(xfrom(B)));
  const xq mid = mul(scaled(xfrom(power), scalar), xfrom(ilg));
  const xq bd = mul(mul(mul(xfrom(q64{-1, 0, 0, 0}), xfrom(left)), mid), xfrom(right));
  const double v = dSdF * dotratio(R, mul(xfrom(T), inv(bd)), R);
  return isfinite(v) ? v : 0.0;
}

// Accumulates one cell's root terms (top: per root and bulk; bottom: per root
// and bulk) into acc. Every lane of the wave calls this (the reductions are
// wave-wide); lanes with active == false add zeros.
template <class Q>
__device__ __forceinline__ void cell_terms(const APArgs& g, ConstRoots roots, const q64& q0,
                                           const Q& T, const Q& B, double w, bool active, double* acc, int K) {
  const MapArgs& a = g.a;
  Q R = T;
  double dSdF = 0.0;
  bool valid = false;
  if (active) {
    R = mul(T, inv(B));
    const double Rm = logmag(R);
    // |R| <= 0 or inf: the reference skips the cell (OPTIMIZE_3D.cpp:8956)
    valid = isfinite(Rm) && ok(R);
    const double F = Rm + log(a.exp_scaling);
    const double tanhTerm = tanh(g.alpha * (F - g.thr));
    dSdF = -g.alpha * w * (1 - tanhTerm * tanhTerm);
  }
  const Q one = from64<Q>(q64{1, 0, 0, 0});
  // top: backward sweep, S = suffix product, prefix = T * S^-1
  {
    Q S = one;
    for (int i = a.nt - 1; i >= 0; i--) {
      double vt = 0.0, vb = 0.0;
      if (valid) {
        const RootRec64 r = load_root64(roots + i);
        const q64 base = qsub(q0, q64{r.w, r.x, r.y, r.z});
        const Q power = pw<Q>(base, r.e);
        const Q right = S;  // S_{i+1}
        S = mul(power, S);  // S_i
        const Q left = (i > 0) ? mul(T, inv(S)) : one;
        const q64 lg = qlog(base);
        const Q iB = inv(B);
        vt = dSdF * dotratio(R, mul(mul(mul(left, mul(scaled(power, a.sc_top), from64<Q>(lg))), right), iB), R);
        vb = dSdF * dotratio(R, mul(mul(mul(left, mul(scaled(power, r.p), from64<Q>(lg))), right), iB), R);
        if constexpr (std::is_same<Q, q64>::value) {
          if (!isfinite(vt)) vt = top_term_x(left, power, a.sc_top, lg, right, T, B, dSdF);
          if (!isfinite(vb)) vb = top_term_x(left, power, r.p, lg, right, T, B, dSdF);
        } else {
          if (!isfinite(vt)) vt = 0.0;
          if (!isfinite(vb)) vb = 0.0;
        }
      }
      wave_acc(acc, K, SL_ROOTS + i, vt);
      wave_acc(acc, K, SL_GTS, vb);
    }
  }
  if (a.nb > 0) {
    const ConstRoots rb = roots + a.nt;
    Q S = one;
    for (int i = a.nb - 1; i >= 0; i--) {
      double vt = 0.0, vb = 0.0;
      if (valid) {
        const RootRec64 r = load_root64(rb + i);
        const q64 base = qsub(q0, q64{r.w, r.x, r.y, r.z});
        const Q power = pw<Q>(base, r.e);
        const Q right = S;
        S = mul(power, S);
        const Q left = (i > 0) ? mul(B, inv(S)) : one;
        const q64 ilg = qinv(qlog(base));
        const Q m1 = from64<Q>(q64{-1, 0, 0, 0});
        if (a.sc_bottom > 0.0) {  // OPTIMIZE_3D.cpp:10084
          const Q bd = mul(mul(mul(m1, left), mul(scaled(power, 1.0 / a.sc_bottom), from64<Q>(ilg))), right);
          vt = dSdF * dotratio(R, mul(T, inv(bd)), R);
          if constexpr (std::is_same<Q, q64>::value) {
            if (!isfinite(vt)) vt = bottom_term_x(left, power, 1.0 / a.sc_bottom, ilg, right, T, B, dSdF);
          } else if (!isfinite(vt)) {
            vt = 0.0;
          }
        }
        if (!(r.p < 1e-8)) {  // OPTIMIZE_3D.cpp:10404-10405
          const Q bd = mul(mul(mul(m1, left), mul(scaled(power, 1.0 / r.p), from64<Q>(ilg))), right);
          vb = dSdF * dotratio(R, mul(T, inv(bd)), R);
          if constexpr (std::is_same<Q, q64>::value) {
            if (!isfinite(vb)) vb = bottom_term_x(left, power, 1.0 / r.p, ilg, right, T, B, dSdF);
          } else if (!isfinite(vb)) {
            vb = 0.0;
          }
        }
      }
      wave_acc(acc, K, SL_ROOTS + a.nt + i, vt);
      wave_acc(acc, K, SL_GBS, vb);
    }
  }
}

template <class Q>
__device__ __forceinline__ Q poly_fwd(ConstRoots r, int n, const q64& q) {
  Q res = pw<Q>(qsub(q, q64{r[0].w, r[0].x, r[0].y, r[0].z}), r[0].e);
  for (int i = 1; i < n; i++) res = mul(res, pw<Q>(qsub(q, q64{r[i].w, r[i].x, r[i].y, r[i].z}), r[i].e));
  return res;
}

// One cell outside the iteration: the origin (field left as it is) and cells
// that start beyond the escape radius. Returns whether the cell iterates.
__device__ __forceinline__ bool ap_cell(const APArgs& g, const double* __restrict__ weight,
                                        double* __restrict__ field, int64_t idx, q64& q0, double& w, double& F) {
  const MapArgs& a = g.a;
  const int64_t X = a.res[0], XY = X * a.res[1];
  int x, y, z;
  if (XY * a.res[2] <= (int64_t)0xffffffffll) {
    const uint32_t p = (uint32_t)idx, r = p - fast_div(p, g.div_xy) * (uint32_t)XY;
    z = (int)fast_div(p, g.div_xy);
    y = (int)fast_div(r, g.div_x);
    x = (int)(r - (uint32_t)y * (uint32_t)X);
  } else {
    z = (int)(idx / XY), y = (int)((idx - z * XY) / X), x = (int)(idx - z * XY - (int64_t)y * X);
  }
  double c[3];
  cell_center(a, x, y, z, c);
  w = field_lookup(g.wg, weight, c);
  q0 = q64{c[0], c[1], c[2], a.slice};
  const double mag0 = qmag(q0);
  if (mag0 < 1e-8) {
    F = field[idx];  // unwritten cell: score terms read the existing value
    return false;
  }
  if (!(mag0 < a.escape) || a.max_iter < 1) {
    F = log(mag0);
    field[idx] = F;
    return false;
  }
  return true;
}

// log(|q - r|^2) for a point (x, y, z, .) with (q.z - r.z)^2 given
__device__ __forceinline__ double log_norm2(double x, double y, double z, const RootRec64& r, double dz2) {
  const double dw = x - r.w, dx = y - r.x, dy = z - r.y;
  return log64(__builtin_fma(dw, dw, __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz2))));
}
__device__ __forceinline__ double log_norm2(const q64& q, const RootRec64& r) {
  const double dz = q.z - r.z;
  return log_norm2(q.w, q.x, q.y, r, dz * dz);
}

// Bounds of the cells that k_ap_grads takes from logarithms: the sums of e |log|b||
// of each polynomial, and |log|R|| + |log c|. Then T, B, their prefixes and
// suffixes and R are within e^+-330, their squares within e^+-660, and a product of
// a top and a bottom factor within e^660 times scalar and logarithm: no step of the
// formulas leaves FP64's range but those that bottom_term_x takes up.
constexpr double kApEach = 330.0;

// One cell from logarithms, as k_ap_fast takes it, for the lanes of cell; clears
// those that are out of bounds.
__device__ __forceinline__ void log_cell(const APArgs& g, ConstRoots roots, const q64& q0, bool& cell, double& F) {
  const MapArgs& a = g.a;
  double f = 0.0, st = 0.0, sb = 0.0, lm = 0.0;
  for (int i = 0; i < a.nt + a.nb; i++) {
    const RootRec64 r = load_root64(roots + i);
    const double l = log_norm2(q0, r), h = 0.5 * r.e;
    f = __builtin_fma(i < a.nt ? h : -h, l, f);
    if (i < a.nt) st = __builtin_fma(h, fabs(l), st);
    else sb = __builtin_fma(h, fabs(l), sb);
    lm = fmax(lm, fabs(l));
  }
  cell = cell && lm < 600.0 && st < kApEach && sb < kApEach && fabs(f) + fabs(g.log_c) < kApEach;
  if (cell) F = f + g.log_c;
}
__device__ __forceinline__ void log_terms(const APArgs& g, ConstRoots roots, const q64& q0, double F, double w,
                                          bool cell, double* acc, int K) {
  const MapArgs& a = g.a;
  double d = 0.0, gts = 0.0, gbs = 0.0;
  if (cell) {
    const double t = tanh(g.alpha * (F - g.thr));
    d = -g.alpha * w * (1 - t * t);
    if (!isfinite(d)) d = 0.0;  // a non-finite weight leaves the root terms out
  }
  for (int i = 0; i < a.nt + a.nb; i++) {
    const RootRec64 r = load_root64(roots + i);
    const double v = d != 0.0 ? 0.5 * d * log_norm2(q0, r) : 0.0;
    const bool top = i < a.nt;
    const double s = top ? a.sc_top : (a.sc_bottom > 0.0 ? -a.sc_bottom : 0.0);  // OPTIMIZE_3D.cpp:10084
    if (top) gts = __builtin_fma(r.p, v, gts);
    else if (!(r.p < 1e-8)) gbs = __builtin_fma(-r.p, v, gbs);  // :10404-10405
    wave_acc(acc, K, SL_ROOTS + i, s * v);
  }
  wave_acc(acc, K, SL_GTS, gts);
  wave_acc(acc, K, SL_GBS, gbs);
}

// The formulas as they stand, for the cells of `left` (kLeft; one bit per cell, 64
// cells a word) or for every cell. Each block takes a
// contiguous run of groups of 256 cells and writes one row of partial sums. The
// cells of `left` whose polynomials are each in range (k_ap_fast tests their sum)
// are taken from logarithms here as well: 64^3 with 200+200 real exponents, 1 %
// of the cells left, 6.3 ms a call without that, 0.90 with it (4.6 by the formulas for
// every cell). Held to two blocks per CU (284 registers otherwise): 64^3 with a
// negative exponent 5.5 to 4.7 ms.
template <bool kLeft>
__global__ __launch_bounds__(kGBlock, 2) void k_ap_grads(APArgs g, const RootRec64* __restrict__ roots,
                                                      const double* __restrict__ weight, double* __restrict__ field,
                                                      const unsigned long long* __restrict__ left, int64_t per,
                                                      double* __restrict__ partials, int K,
                                                      unsigned long long* __restrict__ n_adaptive) {
  extern __shared__ double acc[];  // (kGBlock/64) x K
  const MapArgs& a = g.a;
  for (int i = threadIdx.x; i < (kGBlock / 64) * K; i += kGBlock) acc[i] = 0.0;
  __syncthreads();
  const int64_t N = (int64_t)a.res[0] * a.res[1] * a.res[2];
  int64_t g0 = blockIdx.x, g1 = g0 + 1;  // every cell: a group per block
  if constexpr (kLeft) {
    g0 = blockIdx.x * per;
    g1 = min(g0 + per, (N + kGBlock - 1) / kGBlock);
    // a run without a flagged cell is passed over with one load per thread
    const int64_t nw = (N + 63) / 64, w1 = min(g1 * (kGBlock / 64), nw);
    bool any = false;
    for (int64_t i = g0 * (kGBlock / 64) + threadIdx.x; i < w1; i += kGBlock) any |= left[i] != 0ull;
    if (!__syncthreads_or(any)) g0 = g1;
  }
  for (int64_t gi = g0; gi < g1; gi++) {
    const int64_t idx = gi * kGBlock + threadIdx.x;
    bool active = idx < N;
    if constexpr (kLeft) active = active && ((left[idx >> 6] >> (idx & 63)) & 1ull);
    if (!__ballot(active)) continue;
    double w = 0.0;
    q64 q0{0, 0, 0, 0};
    double Ffield = 0.0;
    bool iterate = false;
    if (active) iterate = ap_cell(g, weight, field, idx, q0, w, Ffield);
    bool logs = kLeft && iterate;
    if (kLeft && __ballot(logs)) {
      log_cell(g, (ConstRoots)roots, q0, logs, Ffield);
      if (__ballot(logs)) log_terms(g, (ConstRoots)roots, q0, Ffield, w, logs, acc, K);
    }
    // forward sweep (computeRationalMapAP with one iteration)
    const bool formulas = iterate && !logs;
    q64 T{1, 0, 0, 0}, B{1, 0, 0, 0};
    bool ovf = false;
    if (formulas) {
      T = poly_fwd<q64>((ConstRoots)roots, a.nt, q0);
      q64 qn;
      if (a.nb > 0) {
        B = poly_fwd<q64>((ConstRoots)roots + a.nt, a.nb, q0);
        qn = qdiv(T, B);
        const double m2 = B.w * B.w + B.x * B.x + B.y * B.y + B.z * B.z;
        ovf = !(ok(T) && ok(B) && isfinite(m2) && ok(qn));
      } else {
        qn = T;
        ovf = !ok(T);
      }
      qn = qscale(qn, a.exp_scaling);
      const double mag = qmag(qn);
      ovf |= !isfinite(mag);
      Ffield = log(mag);
    }
    // gradients in FP64 for the cells that stayed finite
    if (__ballot(formulas)) cell_terms<q64>(g, (ConstRoots)roots, q0, T, B, w, formulas && !ovf, acc, K);
    // overflowed cells: the whole cell with explicit binary exponents
    const bool redo = formulas && ovf;
    if (__ballot(redo)) {
      xq TX = xfrom(q64{1, 0, 0, 0}), BX = TX;
      if (redo) {
        TX = poly_fwd<xq>((ConstRoots)roots, a.nt, q0);
        if (a.nb > 0) BX = poly_fwd<xq>((ConstRoots)roots + a.nt, a.nb, q0);
        const xq R = scaled(mul(TX, inv(BX)), a.exp_scaling);
        const double l = logmag(R);
        Ffield = isnan(l) ? 0.0 : l;  // OPTIMIZE_3D.cpp:1557-1561
      }
      cell_terms<xq>(g, (ConstRoots)roots, q0, TX, BX, w, redo, acc, K);
    }
    if (iterate) field[idx] = Ffield;
    double sc = 0.0, ge = 0.0;
    if (active) {
      sc = -tanh(g.alpha * Ffield) * w;
      const double S = tanh(g.alpha * (Ffield - g.thr));
      ge = -g.alpha * w * (1.0 - S * S);
    }
    wave_acc(acc, K, SL_SCORE, sc);
    wave_acc(acc, K, SL_GEXP, ge);
    const unsigned long long nr = __popcll(__ballot(redo));
    if ((threadIdx.x & 63) == 0 && nr) atomicAdd(n_adaptive, nr);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < K; k += kGBlock) {
    double s = 0.0;
    for (int wv = 0; wv < kGBlock / 64; wv++) s += acc[wv * K + k];
    partials[(int64_t)blockIdx.x * K + k] = s;
  }
}

// Wave sum in lane 63: row shifts and broadcasts instead of LDS shuffles.
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, kRows, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, kRows, 0xf, false);
  return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);  // row_shr:2
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31
  return v;
}

// Sum of e |log|b|| over both polynomials and |log c| up to which every
// product, |B|^2, quotient and |q|^2 of a cell, prefixes included, stays well
// inside FP64's range (2 x 340 < 1022 ln 2).
constexpr double kApRange = 340.0;
constexpr int kApWaves = 8, kApBlock = 64 * kApWaves;
constexpr int kApFastRows = 2;  // score, grad_exp, then sum of dSdF log|b_i| per root

// The AP pass of the cells that stay in range: 64 M cells per block, lane l of
// every wave holding cells l, l + 64, ... Each of the eight waves takes an eighth
// of the roots for all of the block's cells: the logarithms and, through LDS,
// each cell's sum of e log|b|; then, with dSdF known, the sum of dSdF log|b_i|
// over the cells, one wave reduction per root and block. R > 0: a wave has at
// most R roots and keeps their M R logarithms in registers between the two
// steps (R roots unrolled, in groups of kGroup so that four logarithms are
// always in flight; a group past the wave's last root is skipped, a root past
// it inside a group weighs 0). R = 0: any number of roots, and the second step
// computes the logarithms again for the cells whose dSdF is not exactly 0
// (tanh saturates at |alpha F| > 19). FP64 VALU bound: 36 instructions per cell
// and root. Figures beside ap_grads.
template <int M, int R>
__global__ __launch_bounds__(kApBlock) void k_ap_fast(APArgs g, const RootRec64* __restrict__ roots,
                                                     const double* __restrict__ weight, double* __restrict__ field,
                                                     unsigned long long* __restrict__ left,
                                                     double* __restrict__ partials,
                                                     unsigned long long* __restrict__ n_adaptive) {
  constexpr int kCells = 64 * M, kWaves = kApWaves, kGroup = M >= 4 ? 1 : 4 / M;
  static_assert(R % kGroup == 0, "whole groups of roots");
  __shared__ double s_a[kWaves][kCells], s_b[kWaves][kCells];
  __shared__ double s_q[3][kCells];
  __shared__ double s_sum[2][kWaves];
  __shared__ int s_n[kWaves];
  const MapArgs& a = g.a;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t N = (int64_t)a.res[0] * a.res[1] * a.res[2];
  const int64_t idx = (int64_t)blockIdx.x * kCells + tid;
  if (blockIdx.x == 0 && tid == 0) *n_adaptive = 0ull;
  const bool owner = tid < kCells && idx < N;
  bool iterate = false;
  double w = 0.0, F = 0.0;
  q64 q0{1, 1, 1, 1};
  if (owner) iterate = ap_cell(g, weight, field, idx, q0, w, F);
  if (tid < kCells) {
    s_q[0][tid] = q0.w;
    s_q[1][tid] = q0.x;
    s_q[2][tid] = q0.y;
  }
  __syncthreads();
  const int nr = a.nt + a.nb, i0 = wave * nr / kWaves, i1 = (wave + 1) * nr / kWaves;
  // the roots in turn from top and bottom, what is left of the longer one last: the
  // running sums of logarithms stay small, and with them their roundings
  const int pairs = 2 * (a.nt < a.nb ? a.nt : a.nb);
  const int lo = (a.nt > a.nb ? 0 : a.nt) - (pairs >> 1);
  auto root_at = [&](int j) {
    const int two = (j >> 1) + (j & 1) * a.nt;
    return j < pairs ? two : j + lo;
  };
  double x[M], y[M], z[M], f[M] = {}, s[M] = {}, lm[M] = {}, l[R > 0 ? R : 1][M];
#pragma unroll
  for (int u = 0; u < M; u++) {
    x[u] = s_q[0][lane + 64 * u];
    y[u] = s_q[1][lane + 64 * u];
    z[u] = s_q[2][lane + 64 * u];
  }
  auto add = [&](const RootRec64& r, double h, bool top, double* lg) {
    const double dz = a.slice - r.z, dz2 = dz * dz, sg = top ? h : -h;
#pragma unroll
    for (int u = 0; u < M; u++) {
      lg[u] = log_norm2(x[u], y[u], z[u], r, dz2);
      f[u] = __builtin_fma(sg, lg[u], f[u]);
      s[u] = __builtin_fma(h, fabs(lg[u]), s[u]);
      lm[u] = fabs(lg[u]) > lm[u] ? fabs(lg[u]) : lm[u];
    }
  };
  if (R > 0) {
#pragma unroll
    for (int j = 0; j < R; j += kGroup) {
      if (i0 + j < i1) {
#pragma unroll
        for (int k = j; k < j + kGroup; k++) {
          const bool in = i0 + k < i1;
          const int i = root_at(in ? i0 + k : i1 - 1);
          const RootRec64 r = roots[i];
          add(r, in ? 0.5 * r.e : 0.0, i < a.nt, l[k]);
        }
      }
    }
  } else {
    for (int j = i0; j < i1; j++) {
      const int i = root_at(j);
      const RootRec64 r = roots[i];
      add(r, 0.5 * r.e, i < a.nt, l[0]);
    }
  }
#pragma unroll
  for (int u = 0; u < M; u++) {
    s_a[wave][lane + 64 * u] = f[u];
    // |b|^2 zero, denormal or beyond the range shows as |log| > 700
    s_b[wave][lane + 64 * u] = lm[u] < 600.0 ? s[u] : __builtin_inf();
  }
  __syncthreads();
  bool act = false, flagged = false;
  double d = 0.0, sc = 0.0, ge = 0.0;
  if (owner) {
    bool mine = true;
    if (iterate) {
      double fs = 0.0, ss = 0.0;
      for (int v = 0; v < kWaves; v++) {
        fs += s_a[v][tid];
        ss += s_b[v][tid];
      }
      const double lc = g.log_c;
      mine = ss + fabs(lc) < kApRange;
      flagged = !mine;
      if (mine) {
        F = fs + lc;
        field[idx] = F;
      }
    }
    if (mine) {
      const double t0 = tanh64(g.alpha * F);
      const double t1 = g.thr == 0.0 ? t0 : tanh64(g.alpha * (F - g.thr));
      sc = -t0 * w;
      ge = -g.alpha * w * (1.0 - t1 * t1);
      act = iterate && isfinite(ge) && ge != 0.0;  // a non-finite weight leaves the root terms out
      d = act ? ge : 0.0;
    }
  }
  const unsigned long long mf = __ballot(flagged), ma = __ballot(act);
  sc = wave_sum63(sc);
  ge = wave_sum63(ge);
  if (lane == 63) {
    s_sum[0][wave] = sc;
    s_sum[1][wave] = ge;
    s_n[wave] = (int)__popcll(ma);
    if (tid < kCells && (idx & ~63ll) < N) left[idx >> 6] = mf;
  }
  __syncthreads();  // s_a and s_b have been read by their owners
  const int K = kApFastRows + nr;
  double* row = partials + (int64_t)blockIdx.x * K;
  if (tid < 2) {
    double t = 0.0;
    for (int v = 0; v < kWaves; v++) t += s_sum[tid][v];
    row[tid] = t;
  }
  double dd[M];
  if (R > 0) {
    // (log64 is finite for every argument, so a weight of 0 leaves a cell out)
    if (tid < kCells) s_a[0][tid] = d;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < M; u++) dd[u] = s_a[0][lane + 64 * u];
#pragma unroll
    for (int k = 0; k < (R > 0 ? R : 1); k++) {
      if (i0 + k < i1) {
        double v = 0.0;
#pragma unroll
        for (int u = 0; u < M; u++) v = __builtin_fma(dd[u], l[k][u], v);
        v = wave_sum63(v);
        if (lane == 63) row[kApFastRows + root_at(i0 + k)] = 0.5 * v;
      }
    }
    return;
  }
  // R = 0: the cells with a dSdF, listed in cell order
  int at = (int)__popcll(ma & ((1ull << lane) - 1ull)), nact = 0;
  for (int v = 0; v < kWaves; v++) {
    if (v < wave) at += s_n[v];
    nact += s_n[v];
  }
  if (act) {
    s_a[0][at] = q0.w;
    s_a[1][at] = q0.x;
    s_a[2][at] = q0.y;
    s_a[3][at] = d;
  }
  __syncthreads();
  const int nu = (nact + 63) >> 6;  // the same for the whole block
#pragma unroll
  for (int u = 0; u < M; u++) {
    const int j = lane + 64 * u;
    const bool in = j < nact;
    x[u] = in ? s_a[0][j] : 0.0;
    y[u] = in ? s_a[1][j] : 0.0;
    z[u] = in ? s_a[2][j] : 0.0;
    dd[u] = in ? s_a[3][j] : 0.0;
  }
  for (int j = i0; j < i1; j++) {
    const int i = root_at(j);
    const RootRec64 r = roots[i];
    const double dz = a.slice - r.z, dz2 = dz * dz;
    double v = 0.0;
#pragma unroll
    for (int u = 0; u < M; u++)
      if (u < nu) v = __builtin_fma(dd[u], log_norm2(x[u], y[u], z[u], r, dz2), v);
    v = wave_sum63(v);
    if (lane == 63) row[kApFastRows + i] = 0.5 * v;
  }
}

// Sums partials[b][k] over b for the kCols columns from k0 on: 1024 / kCols
// threads per column take strided runs of rows in order, then a fixed tree over
// them (deterministic). A block reads runs of kCols columns of a row; one column
// per block read every line sixteen times. 640 columns of 2048 rows: 19 us that
// way, 6.6 / 7.6 / 9.5 with 16 / 8 / 4 columns; the AP pass's 70 columns of 3600
// rows, where few blocks are left, 6.6 and 10.1 / 7.9 / 6.6.
constexpr int kSumThreads = 1024, kAdjCols = 16, kApCols = 4;
template <int kCols>
__device__ __forceinline__ double column_sum(const double* __restrict__ partials, int64_t nb, int K, int k0) {
  __shared__ double s_v[kSumThreads];
  const int k = k0 + (int)(threadIdx.x & (kCols - 1));
  double v = 0.0;
  if (k < K) {
#pragma unroll 8
    for (int64_t b = threadIdx.x / kCols; b < nb; b += kSumThreads / kCols) v += partials[b * K + k];
  }
  s_v[threadIdx.x] = v;
  __syncthreads();
  for (int w = kSumThreads / 2; w >= kCols; w >>= 1) {
    if ((int)threadIdx.x < w) s_v[threadIdx.x] += s_v[threadIdx.x + w];
    __syncthreads();
  }
  return s_v[threadIdx.x & (kCols - 1)];
}
__global__ void k_zero_count(unsigned long long* p) {
  if (threadIdx.x == 0) *p = 0ull;
}

// Column sums over two arrays at once: blocks (., 0) sum the columns of the
// first, blocks (., 1) of the second, and both results and the cell count go to
// pinned host memory, which the caller reads after its one wait.
__global__ __launch_bounds__(kSumThreads) void k_ap_finish(const double* __restrict__ p0, int64_t n0, int K0,
                                                           const double* __restrict__ p1, int64_t n1, int K1,
                                                           const unsigned long long* __restrict__ n_adaptive,
                                                           double* __restrict__ h) {
  const int second = blockIdx.y, k0 = blockIdx.x * kApCols, k = k0 + (int)threadIdx.x;
  const int K = second ? K1 : K0;
  if (k0 >= K) return;
  const double v = column_sum<kApCols>(second ? p1 : p0, second ? n1 : n0, K, k0);
  if (threadIdx.x < kApCols && k < K) {
    h[1 + (second ? K0 : 0) + k] = v;
    if (k == 0 && second) h[0] = (double)*n_adaptive;  // exact below 2^53
  }
}

// Whether the cells are worth k_ap_fast. |b^e| = |b|^e needs exponents that are not
// negative. And where a polynomial's sum of e |log|b|| is out of bounds (kApEach) in
// many cells, most waves of k_ap_grads hold one and run the formulas after all.
// Roots 0.6 about the centre of a box of edge 3, calls in us by the formulas alone and
// with k_ap_fast, by that sum at the box's far corner (each logarithm at least 1): 8+8
// roots, 64^3, at 250 / 360 / 460 / 610 226 / 239 / 387 / 457 and 81 / 87 / 352 / 518;
// 32+32 roots, 97^3, at 325 / 450 / 610 2264 / 2408 / 3779 and 467 / 2102 / 5129, 16^3
// at 450 253 and 307; 200+200 roots, 64^3, at 380 4134 and 874. So up to 400.
static bool ap_from_logs(const MapArgs& a, const std::vector<RootRec64>& roots) {
  const double most = 400.0;
  double half = 0.0, away = 0.0, e[2] = {0.0, 0.0};
  for (int i = 0; i < 3; i++) half += 0.25 * a.dx[i] * a.dx[i] * (double)a.res[i] * (double)a.res[i];
  half = sqrt(half);
  auto distance2 = [&](const RootRec64& r) {
    const double d[4] = {r.w - a.center[0], r.x - a.center[1], r.y - a.center[2], r.z - a.slice};
    return d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + d[3] * d[3];
  };
  for (size_t i = 0; i < roots.size(); i++) {
    if (!(roots[i].e >= 0.0 && roots[i].e <= DBL_MAX)) return false;
    e[(int)i >= a.nt] += roots[i].e;
    away = fmax(away, distance2(roots[i]));
  }
  if (fmax(e[0], e[1]) * fmax(1.0, ::log(half + sqrt(away))) <= most) return true;
  double s[2] = {0.0, 0.0};
  for (size_t i = 0; i < roots.size(); i++)
    s[(int)i >= a.nt] += roots[i].e * fmax(1.0, ::log(half + sqrt(distance2(roots[i]))));
  return s[0] <= most && s[1] <= most;
}

// 256 cells a block keep four logarithms per lane in flight and share the block's
// set-up; below 128 such blocks (half the CUs) 64 cells a block spread the work
// further: 25^3 35.4 against 39.1 us a call, 40^3 43.5 against 39.8, 64^3 77.5
// against 59.3 (64- against 256-cell blocks, 32+32 real exponents). A wave keeps the
// logarithms of up to 8 or 16 roots in registers (128 and 192 VGPRs), of up to 32
// in 64-cell blocks; beyond 128 roots on grids of 256-cell blocks and 256 on
// smaller ones they are computed twice (97^3 with 32+32 roots: 149 us that way, 128
// kept). Against the product formulas for every cell: 97^3 2280 to 126 us a call,
// 25^3 257 to 36 us; the kernel takes 108 us of the 126, its FP64 issue about 80.
qj_status ap_grads(qj_workspace* ws, const MapArgs& a, const qj_rational* f, const qj_grid* wg, const double* d_weight,
                   double alpha, double thr, double* d_field, double* gt, double* gb, qj_ap_grads* out,
                   hipStream_t s) {
  const int64_t N = (int64_t)a.res[0] * a.res[1] * a.res[2];
  const int nr = a.nt + a.nb, K = SL_ROOTS + nr, KF = kApFastRows + nr;
  const size_t lds = sizeof(double) * (kGBlock / 64) * K;
  if (lds > 64 * 1024) {
    set_error("too many roots for the gradient kernel (%d)", nr);
    return QJ_ERR_CAPACITY;
  }
  const bool fast = ap_from_logs(a, f->h64);
  const int64_t groups = (N + kGBlock - 1) / kGBlock;
  const bool wide = groups >= 128;
  const int per_wave = (nr + kApWaves - 1) / kApWaves;  // roots of the busiest wave
  const int64_t cells = wide || per_wave > 32 ? 256 : 64;
  const int64_t rows_f = fast ? (N + cells - 1) / cells : 0;
  // rows of the general kernel: one per group when it does all the work
  const int64_t per = fast ? (groups + 511) / 512 : 1, rows_g = (groups + per - 1) / per;
  const int64_t nwords = (N + 63) / 64;
  qj_status st = ensure_partials(ws, rows_f * KF + rows_g * K + nwords + 1, s);
  if (st) return st;
  if ((st = ensure_pinned(ws, 1 + KF + K, s))) return st;
  APArgs g;
  g.a = a;
  make_geom(wg, &g.wg);
  g.alpha = alpha;
  g.thr = thr;
  g.log_c = ::log(a.exp_scaling);
  const uint64_t XY = (uint64_t)a.res[0] * (uint64_t)a.res[1];
  g.div_x = make_fastdiv((uint32_t)a.res[0]);
  g.div_xy = make_fastdiv(XY <= 0xffffffffull ? (uint32_t)XY : 1u);
  double* pf = ws->d_partials;
  double* pg = pf + rows_f * KF;
  unsigned long long* left = (unsigned long long*)(pg + rows_g * K);
  unsigned long long* nad = left + nwords;
  if (fast) {
    const auto k = cells == 64 ? (per_wave <= 8 ? k_ap_fast<1, 8> : k_ap_fast<1, 32>)
                               : (per_wave <= 8 ? k_ap_fast<4, 8> : per_wave <= 16 ? k_ap_fast<4, 16> : k_ap_fast<4, 0>);
    hipLaunchKernelGGL(k, dim3((unsigned)rows_f), dim3(kApBlock), 0, s, g, f->d64, d_weight, d_field, left, pf, nad);
  } else {
    hipLaunchKernelGGL(k_zero_count, dim3(1), dim3(64), 0, s, nad);
  }
  QJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(fast ? k_ap_grads<true> : k_ap_grads<false>, dim3((unsigned)rows_g), dim3(kGBlock), lds, s, g,
                     f->d64, d_weight, d_field, (const unsigned long long*)left, per, pg, K, nad);
  QJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_ap_finish, dim3((K + kApCols - 1) / kApCols, 2), dim3(kSumThreads), 0, s, (const double*)pf,
                     rows_f, KF, (const double*)pg, rows_g, K, (const unsigned long long*)nad, ws->h_pinned);
  QJ_HIP(hipGetLastError());
  QJ_HIP(hipStreamSynchronize(s));
  const double* hf = ws->h_pinned + 1;        // fast cells
  const double* hg = ws->h_pinned + 1 + KF;  // the others
  out->score = hf[0] + hg[SL_SCORE];
  out->grad_exp = hf[1] + hg[SL_GEXP];
  out->adaptive_cells = (int64_t)ws->h_pinned[0];
  double gts = hg[SL_GTS], gbs = hg[SL_GBS];
  for (int i = 0; i < a.nt; i++) {
    const double v = hf[kApFastRows + i];
    gt[i] = a.sc_top * v + hg[SL_ROOTS + i];
    gts += f->h64[i].p * v;
  }
  for (int i = a.nt; i < nr; i++) {
    const double v = hf[kApFastRows + i], p = f->h64[i].p;
    // OPTIMIZE_3D.cpp:10084 and :10404-10405
    gb[i - a.nt] = (a.sc_bottom > 0.0 ? -a.sc_bottom * v : 0.0) + hg[SL_ROOTS + i];
    if (!(p < 1e-8)) gbs -= p * v;
  }
  out->grad_top_scalar = gts;
  out->grad_bottom_scalar = gbs;
  return QJ_OK;
}

// ------------------------------------------------------------ adjoint at points

template <class T>
struct Q4 {
  T w, x, y, z;
};
template <class T>
__device__ __forceinline__ Q4<T> mul(const Q4<T>& l, const Q4<T>& r) {
  Q4<T> f;
  f.x = l.y * r.z - l.z * r.y + r.w * l.x + l.w * r.x;
  f.y = l.z * r.x - l.x * r.z + r.w * l.y + l.w * r.y;
  f.z = l.x * r.y - l.y * r.x + r.w * l.z + l.w * r.z;
  f.w = l.w * r.w - l.x * r.x - r.y * l.y - l.z * r.z;
  return f;
}
template <class T>
__device__ __forceinline__ Q4<T> conj(const Q4<T>& a) { return {a.w, -a.x, -a.y, -a.z}; }
template <class T>
__device__ __forceinline__ Q4<T> sc(const Q4<T>& a, T s) { return {a.w * s, a.x * s, a.y * s, a.z * s}; }
template <class T>
__device__ __forceinline__ T dot(const Q4<T>& a, const Q4<T>& b) { return a.w * b.w + a.x * b.x + a.y * b.y + a.z * b.z; }
template <class T>
__device__ __forceinline__ Q4<T> unit(const Q4<T>& a) {
  const T n = sqrt(dot(a, a));
  return n > T(0) ? sc(a, T(1) / n) : a;
}

// The elementary functions of the adjoint's backward sweep in its two precisions.
template <class T>
struct Fn;
template <>
struct Fn<double> {
  __device__ __forceinline__ static void root(double x, double& r, double& inv) { sqrt_rsqrt64(x, r, inv); }
  __device__ __forceinline__ static double recip(double x) { return div64(1.0, x); }
  __device__ __forceinline__ static double log(double x) { return log64<true>(x); }
  __device__ __forceinline__ static double exp(double x) { return exp64<true>(x); }
  __device__ __forceinline__ static double angle(double y, double w) { return angle64<true>(y, w); }
  __device__ __forceinline__ static void sincos(double m, double& s, double& c) { sincos64<true>(m, s, c); }
};
template <>
struct Fn<float> {
  __device__ __forceinline__ static void root(float x, float& r, float& inv) {
    const float y = __builtin_amdgcn_rsqf(x);
    inv = __builtin_fmaf(0.5f * y, __builtin_fmaf(-x * y, y, 1.0f), y);
    r = x * inv;
  }
  __device__ __forceinline__ static float recip(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
  }
  __device__ __forceinline__ static float log(float x) { return logf(x); }
  __device__ __forceinline__ static float exp(float x) { return expf(x); }
  __device__ __forceinline__ static float angle(float y, float w) { return angle_upper(y, w); }
  __device__ __forceinline__ static void sincos(float m, float& s, float& c) { sincosf(m, &s, &c); }
};

// One root; the block's copy of them is in LDS, where a lane's read takes about
// 100 cycles instead of the 500 of a scattered load.
struct AdjRoot {
  double w, x, y, z, e;
};

// One power term t = (q - r)^e (QUATERNION::pow, QUATERNION.cpp:375-393, for
// e > 0). Exponents 1 and 2 are p = b and b b, |p| = |b|^e; others (kGen) the
// unit polar p = (A, C v) with A = cos m, C = sin m / |v|, m = e angle(|v|, w).
// b is taken in FP64 also where the rest is FP32: q - r next to a root.
template <class T>
struct Term {
  Q4<T> b, p;
  T n2, part;  // |b|^2, |v|^2
  T e, A, C;
  bool two, gen;
};
template <class T, bool kGen>
__device__ __forceinline__ Term<T> make_term(const Q4<double>& q, const AdjRoot& rr) {
  Term<T> t;
  t.e = T(rr.e);
  t.two = rr.e == 2.0;
  t.gen = kGen && rr.e != 1.0 && !t.two;
  t.b = Q4<T>{T(q.w - rr.w), T(q.x - rr.x), T(q.y - rr.y), T(q.z - rr.z)};
  t.part = t.b.x * t.b.x + t.b.y * t.b.y + t.b.z * t.b.z;
  t.n2 = t.part + t.b.w * t.b.w;
  t.p = t.b;
  if (t.two) {
    const T w2 = T(2) * t.b.w;
    t.p = Q4<T>{t.b.w * t.b.w - t.part, w2 * t.b.x, w2 * t.b.y, w2 * t.b.z};
  }
  if (t.gen) {
    T rho, vi, s, c;
    Fn<T>::root(t.part, rho, vi);
    const bool v0 = !(t.part > T(0));
    Fn<T>::sincos(t.e * (v0 ? (t.b.w < T(0) ? T(3.141592653589793) : T(0)) : Fn<T>::angle(rho, t.b.w)), s, c);
    t.A = c;
    t.C = v0 ? t.e / t.b.w : s * vi;  // limit v -> 0 (w > 0)
    t.p = Q4<T>{t.A, t.C * t.b.x, t.C * t.b.y, t.C * t.b.z};
  }
  return t;
}
// b's adjoint from p = |t| / |Q| times the polar term's, in unit form
template <class T>
__device__ __forceinline__ Q4<T> polar_vjp(const Term<T>& t, const Q4<T>& p) {
  T r, ri;
  Fn<T>::root(t.n2, r, ri);
  const T w = t.b.w, e = t.e;
  const T gA = p.w;
  const T gC = p.x * t.b.x + p.y * t.b.y + p.z * t.b.z;
  const T Gr = (gA * e * t.A + gC * e * t.C) * ri;
  if (!(t.part > T(0))) {
    // purely real base: d/db of (w^e, e w^(e-1) v) / w^e
    return Q4<T>{Gr, t.C * p.x, t.C * p.y, t.C * p.z};
  }
  T rho, vi;
  Fn<T>::root(t.part, rho, vi);
  const T Gth = -gA * e * t.C * rho + gC * e * t.A * vi;
  const T ri2 = ri * ri;
  const T coef = Gr * ri + Gth * w * (ri2 * vi) - gC * t.C * (vi * vi);
  return Q4<T>{Gr * (w * ri) - Gth * (rho * ri2), coef * t.b.x + t.C * p.x, coef * t.b.y + t.C * p.y,
               coef * t.b.z + t.C * p.z};
}
// One step of the backward sweep: b's adjoint from W = R M conj(R) (see
// k_adjoint), and W turned past the term, u W conj(u) with u = p / |p|. The
// exponents 1 and 2 take 1 / |b|^2 and no square root.
template <class T>
__device__ __forceinline__ Q4<T> sweep_step(const Term<T>& t, Q4<T>& W) {
  if (t.gen) {
    const Q4<T> tb = mul(t.p, W);
    W = mul(tb, conj(t.p));
    return polar_vjp(t, tb);
  }
  const T s = Fn<T>::recip(t.n2);
  const Q4<T> tb = sc(mul(t.p, W), s);
  if (!t.two) {
    W = mul(tb, conj(t.b));
    return tb;
  }
  // t = b^2: (p conj(b) + conj(b) p) / |b|^2
  W = sc(mul(tb, conj(t.p)), s);
  const T f = T(2) * s;
  return Q4<T>{f * (tb.w * t.b.w + (tb.x * t.b.x + tb.y * t.b.y + tb.z * t.b.z)), f * (t.b.w * tb.x - tb.w * t.b.x),
               f * (t.b.w * tb.y - tb.w * t.b.y), f * (t.b.w * tb.z - tb.w * t.b.z)};
}

constexpr int kAdjBlock = 128;
constexpr int kMaxAdjIter = 16;
// iterations whose group products are kept for the backward sweep (private
// memory: 17 values each); later ones are formed again
constexpr int kAdjKeep = 3;

template <int kCtrl>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, false));
}
template <int kCtrl>
__device__ __forceinline__ double dpp_mov(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, 0xf, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, 0xf, 0xf, false);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
// v + the value 16 (32) lanes across: the row swaps of v with itself
template <int kRows>
__device__ __forceinline__ double swap_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
  if constexpr (kRows == 16) {
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) + __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
  } else {
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) + __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
  }
}
// sum over the groups of a wave, lane by lane (the lanes that hold the same roots)
template <int L>
__device__ __forceinline__ double across_groups(double v) {
  if constexpr (L <= 4) v += dpp_mov<0x124>(v);  // row_ror:4
  if constexpr (L <= 8) v += dpp_mov<0x128>(v);  // row_ror:8
  if constexpr (L <= 16) v = swap_add<16>(v);
  if constexpr (L <= 32) v = swap_add<32>(v);
  return v;
}
// the value d lanes up inside a group (lanes past its end: anything)
template <int L, int d, class T>
__device__ __forceinline__ Q4<T> lanes_up(const Q4<T>& a) {
  if constexpr (L <= 16) {
    constexpr int c = 0x100 + d;  // row_shl
    return {dpp_mov<c>(a.w), dpp_mov<c>(a.x), dpp_mov<c>(a.y), dpp_mov<c>(a.z)};
  } else {
    return {__shfl_down(a.w, d, L), __shfl_down(a.x, d, L), __shfl_down(a.y, d, L), __shfl_down(a.z, d, L)};
  }
}
template <int L, class T>
__device__ __forceinline__ T group_sum(T v) {
  for (int o = L / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
template <int L, class T>
__device__ __forceinline__ Q4<T> group_sum_q(const Q4<T>& a) {
  return {group_sum<L>(a.w), group_sum<L>(a.x), group_sum<L>(a.y), group_sum<L>(a.z)};
}

// Over a group: a polynomial's unit product, and the unit product of the roots
// after this lane's share.
template <class T>
struct Share {
  Q4<T> all, after;
};
template <int L, int d, class T>
__device__ __forceinline__ void suffix_step(Q4<T>& suf, int sub) {
  if constexpr (d < L) {
    const Q4<T> z = mul(suf, lanes_up<L, d>(suf));
    if (sub + d < L) suf = z;
    suffix_step<L, 2 * d>(suf, sub);
  }
}
// c: root steps of every lane (uniform); the lane's roots are [lo, hi). Always in
// FP64; ln: the polynomial's log magnitude.
template <int L, bool kGen>
__device__ __forceinline__ Share<double> group_product(const AdjRoot* roots, int lo, int hi, int c,
                                                       const Q4<double>& q, int sub, double& ln) {
  // exponents 1 and 2 as they are, brought to a norm in [0.7, 1.5) by a power
  // of two each (2^+-60 over a share of 100 roots)
  Q4<double> p{1, 0, 0, 0};
  double lg = 0;
  int E = 0;
  for (int j = 0; j < c; j++) {
    if (lo + j < hi) {
      const Term<double> t = make_term<double, kGen>(q, roots[lo + j]);
      if (kGen && t.gen) {
        p = mul(p, t.p);
        lg += t.e * log64<true>(t.n2);
      } else {
        // half the norm's exponent
        int k = ((int)(__builtin_bit_cast(uint64_t, t.n2) >> 52) - 1022) >> 1;
        if (t.two) k *= 2;
        E += k;
        p = mul(p, sc(t.p, __builtin_bit_cast(double, (uint64_t)(1023 - k) << 52)));
      }
    }
  }
  double n2 = dot(p, p), r, ri;
  sqrt_rsqrt64(n2, r, ri);
  p = sc(p, ri);
  ln = group_sum<L>(0.5 * (lg + log64<true>(n2)) + E * 0.6931471805599453);
  // ordered inclusive suffix products over the group (Hillis-Steele)
  suffix_step<L, 1>(p, sub);
  Share<double> s;
  s.all = unit(Q4<double>{__shfl(p.w, 0, L), __shfl(p.x, 0, L), __shfl(p.y, 0, L), __shfl(p.z, 0, L)});
  const Q4<double> nxt = lanes_up<L, 1>(p);
  s.after = sub + 1 < L ? unit(nxt) : Q4<double>{1, 0, 0, 0};
  return s;
}
template <class T>
__device__ __forceinline__ Q4<T> as(const Q4<double>& a) {
  return {T(a.w), T(a.x), T(a.y), T(a.z)};
}

// slot layout per root i (top then bottom): 5 i + {0..3} = d/d root component, 5 i + 4 = d/d e_i
//
// Reverse mode through max_iter iterations of the map. One group of L lanes
// per point; lane `sub` takes top roots [sub ct, sub ct + ct) and bottom roots
// [sub cb, sub cb + cb). Control flow is uniform over the wave (every group
// runs the same iterations and root steps, masked), so lane exchanges always
// see active partners. Forward, in FP64 for both precisions (an FP32 iterate is
// off by its rounding times the map's growth, 10 to 30 per iteration): the
// iterates up to the last one's start, with each iteration's group products.
// Backward, in T:
//   * a point's last iteration needs no product: F = log c + sum e log|b| over
//     the top roots - the same over the bottom ones, so b's adjoint is
//     +-g e b / |b|^2 and e's is +-g log|b|;
//   * before that, with q' = c T B^-1, M = |Q| conj(T) (Q' B) in unit parts and
//     R the product of the roots after root i, the term's adjoint is
//     u_i W_i, u_i its unit part and W_i = R M conj(R) (-M for the bottom
//     roots), which the sweep turns from one root to the next: W <- u W conj(u).
//     e's adjoint is W . log b.
// FP64 / FP32 VALU bound, long dependent chains. Figures beside points_adjoint.
template <class T, int L, bool kGen>
__global__ __launch_bounds__(kAdjBlock, 4) void k_adjoint(MapArgs a, const RootRec64* __restrict__ g_roots,
                                                       const double* __restrict__ pts, int64_t n,
                                                       const double* __restrict__ dJdF,
                                                       double* __restrict__ partials, int K) {
  extern __shared__ double acc[];  // (kAdjBlock/64) x K, then the roots
  AdjRoot* const roots = (AdjRoot*)(acc + (kAdjBlock / 64) * K);
  for (int i = threadIdx.x; i < (kAdjBlock / 64) * K; i += kAdjBlock) acc[i] = 0.0;
  for (int i = threadIdx.x; i < a.nt + a.nb; i += kAdjBlock)
    roots[i] = AdjRoot{g_roots[i].w, g_roots[i].x, g_roots[i].y, g_roots[i].z, g_roots[i].e};
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane & (L - 1);
  const int c[2] = {(a.nt + L - 1) / L, (a.nb + L - 1) / L};
  const int first[2] = {0, a.nt}, count[2] = {a.nt, a.nb};
  double* const mine = acc + wave * K;
  // one root's gradient, summed over the wave's points
  auto add = [&](int i, bool in, const Q4<T>& bb, T ge) {
    const double g0 = across_groups<L>(-(double)bb.w), g1 = across_groups<L>(-(double)bb.x),
                 g2 = across_groups<L>(-(double)bb.y), g3 = across_groups<L>(-(double)bb.z),
                 g4 = across_groups<L>((double)ge);
    if (lane < L && in) {
      // LDS adds without a return: the slots are this wave's own, so they land in program order
      double* r = mine + 5 * i;
      unsafeAtomicAdd(r, g0);
      unsafeAtomicAdd(r + 1, g1);
      unsafeAtomicAdd(r + 2, g2);
      unsafeAtomicAdd(r + 3, g3);
      unsafeAtomicAdd(r + 4, g4);
    }
  };
  constexpr int kPoints = kAdjBlock / L;
  for (int64_t base = (int64_t)blockIdx.x * kPoints; base < n; base += (int64_t)gridDim.x * kPoints) {
    const int64_t pid = base + threadIdx.x / L;
    const bool active = pid < n;
    Q4<double> qs[kMaxAdjIter];
    Share<T> kept[kAdjKeep][2];
    T kept_mag[kAdjKeep];
    qs[0] = active ? Q4<double>{pts[3 * pid], pts[3 * pid + 1], pts[3 * pid + 2], a.slice} : Q4<double>{1, 0, 0, 0};
    const T gF = active ? T(dJdF[pid]) : T(0);
    // one iteration's group products; Qmag = |q'|
    auto products = [&](const Q4<double>& q, Share<T>* s, Q4<double>& Qh, T& Qmag) {
      double lt, lb;
      const Share<double> t =
          group_product<L, kGen>(roots, sub * c[0], min(count[0], sub * c[0] + c[0]), c[0], q, sub, lt);
      Share<double> b{{1, 0, 0, 0}, {1, 0, 0, 0}};
      lb = 0.0;
      if (a.nb > 0)
        b = group_product<L, kGen>(roots + a.nt, sub * c[1], min(count[1], sub * c[1] + c[1]), c[1], q, sub, lb);
      const double m = a.exp_scaling * exp64<true>(lt - lb);
      s[0] = Share<T>{as<T>(t.all), as<T>(t.after)};
      s[1] = Share<T>{as<T>(b.all), as<T>(b.after)};
      Qh = sc(mul(t.all, conj(b.all)), m);
      Qmag = T(m);
    };
    // Kx: iterations the point runs; a point without a gradient runs none
    int Kx = 0;
    bool running = active && gF != T(0) && sqrt(dot(qs[0], qs[0])) < a.escape && a.max_iter > 0;
    for (int k = 0; __ballot(running); k++) {
      if (running) Kx = k + 1;
      if (k + 1 >= a.max_iter) break;
      const Q4<double> q = running ? qs[k] : Q4<double>{1, 0, 0, 0};
      Share<T> s[2];
      Q4<double> Qh;
      T Qmag;
      products(q, s, Qh, Qmag);
      if (k < kAdjKeep) {
        kept[k][0] = s[0];
        kept[k][1] = s[1];
        kept_mag[k] = Qmag;
      }
      if (running) {
        qs[k + 1] = Qh;
        const double mag = sqrt(dot(Qh, Qh));
        if (!(mag < a.escape) || ((a.flags & QJ_MAP_BLACK_HOLE) && mag < 10.0 * (double)FLT_MIN)) running = false;
      }
    }
    Q4<T> qbar{0, 0, 0, 0};
    for (int k = a.max_iter - 1; k >= 0; k--) {
      const bool last = k + 1 == Kx, inner = k + 1 < Kx;
      if (!__ballot(last || inner)) continue;
      const Q4<double> q = (last || inner) ? qs[k] : Q4<double>{1, 0, 0, 0};
      Q4<T> qnew{0, 0, 0, 0};
      if (__ballot(last)) {
        for (int p = 0; p < 2; p++) {
          const T g = p ? -gF : gF;
          const int lo = sub * c[p], hi = min(count[p], lo + c[p]);
          for (int j = 0; j < c[p]; j++) {
            const int i = first[p] + lo + j;
            Q4<T> bb{0, 0, 0, 0};
            T ge = 0;
            if (last && lo + j < hi) {
              const AdjRoot rr = roots[i];
              const Q4<T> b{T(q.w - rr.w), T(q.x - rr.x), T(q.y - rr.y), T(q.z - rr.z)};
              const T n2 = dot(b, b);
              bb = sc(b, g * T(rr.e) * Fn<T>::recip(n2));
              ge = g * T(0.5) * Fn<T>::log(n2);
              qnew = Q4<T>{qnew.w + bb.w, qnew.x + bb.x, qnew.y + bb.y, qnew.z + bb.z};
            }
            add(i, lo + j < hi, bb, ge);
          }
        }
      }
      if (__ballot(inner)) {
        Share<T> s[2];
        T Qmag;
        if (k < kAdjKeep) {
          s[0] = kept[k][0];
          s[1] = kept[k][1];
          Qmag = kept_mag[k];
        } else {
          Q4<double> Qh;
          products(q, s, Qh, Qmag);
        }
        const Q4<T> M = sc(mul(conj(s[0].all), mul(qbar, s[1].all)), Qmag);
        for (int p = 0; p < 2; p++) {
          const int lo = sub * c[p], hi = min(count[p], lo + c[p]);
          Q4<T> W = mul(mul(s[p].after, p ? sc(M, T(-1)) : M), conj(s[p].after));
          for (int j = c[p] - 1; j >= 0; j--) {
            const int i = first[p] + lo + j;
            Q4<T> bb{0, 0, 0, 0};
            T ge = 0;
            if (inner && lo + j < hi) {
              const Term<T> t = make_term<T, kGen>(q, roots[i]);
              // d t / d e = t log(b); log(b) = (log|b|, angle v / |v|)
              T rho, vi;
              Fn<T>::root(t.part, rho, vi);
              const T lv = t.part > T(0) ? Fn<T>::angle(rho, t.b.w) * vi : T(0);
              ge = W.w * (T(0.5) * Fn<T>::log(t.n2)) + lv * (W.x * t.b.x + W.y * t.b.y + W.z * t.b.z);
              bb = sweep_step(t, W);
              qnew = Q4<T>{qnew.w + bb.w, qnew.x + bb.x, qnew.y + bb.y, qnew.z + bb.z};
            }
            add(i, lo + j < hi, bb, ge);
          }
        }
      }
      qnew = group_sum_q<L>(qnew);
      if (last || inner) qbar = qnew;
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < K; k += kAdjBlock) {
    double s = 0.0;
    for (int wv = 0; wv < kAdjBlock / 64; wv++) s += acc[wv * K + k];
    partials[(int64_t)blockIdx.x * K + k] = s;
  }
}

// The sums of the slots' partials over the rows (rows = 0: no points), written to the root gradients (n x 4) or the powers' (dJ/dp = s dJ/de).
__global__ __launch_bounds__(kSumThreads) void k_adjoint_finish(const double* __restrict__ partials, int64_t rows,
                                                                int nt, int nr, double sc_top, double sc_bottom,
                                                                double* __restrict__ grad_roots,
                                                                double* __restrict__ grad_powers) {
  const int k = blockIdx.x * kAdjCols + (int)threadIdx.x;
  const double s = column_sum<kAdjCols>(partials, rows, 5 * nr, blockIdx.x * kAdjCols);
  if (threadIdx.x >= kAdjCols || k >= 5 * nr) return;
  const int i = k / 5, c = k - 5 * i;
  if (c < 4) grad_roots[4 * i + c] = s;
  else grad_powers[i] = s * (i < nt ? sc_top : sc_bottom);
}

// Blocks beyond kAdjRows loop over points, so at most that many rows are summed.
// Lanes per point by the roots a lane would have (gradient in us with 4 / 8 / 16 /
// 32 lanes, FP64): 40k points with 8+8 roots 42 / 57 / 96 / 184, with 64+64 200 /
// 186 / 186 / 245 (exponents 1) and 339 / 294 / 274 / 329 (real), 12k with 32+32
// 117 / 73 / 75 / 82; few points take twice the lanes to fill the chip: 3001 with
// 64+64 89 / 53 / 48 / 40, 300 with 16+16 31 / 22 / 20 / 20. FP32 has its minima at
// the same places (40k 64+64: 157 / 148 / 143 / 187). Against polar terms formed
// three times per iteration and every group product twice: 40k points with 64+64
// roots 917 to 186 us in FP64 and 354 to 143 in FP32, whose error against FP64 went
// from 3e-5 to 6e-8 with the FP64 iterates.
constexpr int64_t kAdjRows = 2048;
static int adj_lanes(const MapArgs& a, int64_t n) {
  const int m = a.nt > a.nb ? a.nt : a.nb;
  const int L = m <= 12 ? 4 : m < 32 ? 8 : 16;
  return n <= 8192 ? 2 * L : L;
}
template <class T, bool kGen>
static auto adjoint_kernel_of(int L) {
  return L == 4 ? k_adjoint<T, 4, kGen> : L == 8 ? k_adjoint<T, 8, kGen> : L == 16 ? k_adjoint<T, 16, kGen>
                                                                                 : k_adjoint<T, 32, kGen>;
}
static auto adjoint_kernel(qj_precision prec, int L, bool gen) {
  return prec == QJ_FP64 ? (gen ? adjoint_kernel_of<double, true>(L) : adjoint_kernel_of<double, false>(L))
                         : (gen ? adjoint_kernel_of<float, true>(L) : adjoint_kernel_of<float, false>(L));
}

qj_status points_adjoint(qj_workspace* ws, const MapArgs& a, const qj_rational* f, qj_precision prec,
                         const double* d_pts, int64_t n, const double* d_dJdF, double* d_gr, double* d_gp,
                         hipStream_t s) {
  const int nr = a.nt + a.nb;
  const int K = 5 * nr;
  if (a.max_iter > kMaxAdjIter) {
    set_error("the adjoint supports max_iter <= %d (got %d)", kMaxAdjIter, a.max_iter);
    return QJ_ERR_CAPACITY;
  }
  for (const RootRec64& r : f->h64)
    if (!(r.e > 0.0)) {
      set_error("the adjoint needs positive exponents (power_scalar * power > 0)");
      return QJ_ERR_INVALID;
    }
  if (sizeof(double) * (kAdjBlock / 64) * K > 64 * 1024) {
    set_error("too many roots for the adjoint kernel (%d)", nr);
    return QJ_ERR_CAPACITY;
  }
  // the sums and the roots: at most 64 + 32 KiB
  const size_t lds = sizeof(double) * (kAdjBlock / 64) * K + sizeof(AdjRoot) * (size_t)nr;
  const int L = adj_lanes(a, n);
  const int64_t per_block = kAdjBlock / L;  // points
  const int64_t rows = std::min<int64_t>((n + per_block - 1) / per_block, kAdjRows);
  qj_status st = ensure_partials(ws, rows * K, s);
  if (st) return st;
  if (n > 0) {
    hipLaunchKernelGGL(adjoint_kernel(prec, L, a.gen != 0), dim3((unsigned)rows), dim3(kAdjBlock), lds, s, a, f->d64,
                       d_pts, n, d_dJdF, ws->d_partials, K);
    QJ_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_adjoint_finish, dim3((K + kAdjCols - 1) / kAdjCols), dim3(kSumThreads), 0, s,
                     (const double*)ws->d_partials, rows, a.nt, nr,
                     a.sc_top, a.sc_bottom, d_gr, d_gp);
  QJ_HIP(hipGetLastError());
  return QJ_OK;
}

}  // namespace qj
