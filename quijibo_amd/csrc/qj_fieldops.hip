// FIELD_3D clean-up passes that the reference runs on a fractal before
// meshing it (toothOptimizer.cpp:250-254, OPTIMIZE_3D.cpp:4718):
//   clampInfsToMean  (FIELD_3D.cpp:5182-5207)  every infinite cell takes the
//                    mean of the non-infinite cells
//   clampNansToMean  (FIELD_3D.cpp:5212-5234)  every NaN cell takes the mean
//                    of the non-NaN cells
//   setBorders       (FIELD_3D.cpp:5357-5382)  the six faces take a constant
//
// The reference sums serially in x-fastest order, so a NaN cell makes the
// clampInfsToMean mean NaN and an infinite cell makes the clampNansToMean
// mean infinite (or NaN with both signs). Here the finite cells are summed in
// double-double arithmetic (error-free TwoSum per addition, a fixed tree over
// blocks, so the result does not depend on scheduling) and the non-finite
// ones separately in plain IEEE arithmetic, which gives the serial sum's
// non-finite outcomes exactly. The double-double sum is off the exact sum by
// at most about n u^2 sum|x_i| before its final rounding (u = 2^-53), so the
// mean is the correctly rounded sum over the count for any field that fits
// in memory; the reference's serial sum differs from that by up to
// (n - 1) u sum|x_i|. A finite sum beyond DBL_MAX gives NaN here (the
// serial sum gives inf).
//
// HBM-bound: the field is read twice (sum, then replace) and only replaced
// cells are written; the mean never leaves the device, so nothing waits on
// the host. Three launches: per-block partial sums, one block that combines
// them into the mean, and the replacement.
#include <math.h>

#include <algorithm>

#include "qj_geom.h"
#include "qj_internal.h"
#include "qj_math64.h"

namespace qj {

namespace {

constexpr int kOpsBlock = 256;
constexpr int kOpsGrid = 2048;  // 8 blocks per CU; a fixed count keeps the reduction tree fixed

struct DD {
  double hi, lo;
};

// Knuth's TwoSum: s + e == a + b exactly (no multiplications, so no contraction applies).
__device__ __forceinline__ DD two_sum(double a, double b) {
  const double s = a + b;
  const double bb = s - a;
  const double e = (a - (s - bb)) + (b - bb);
  return DD{s, e};
}
__device__ __forceinline__ DD fast_two_sum(double a, double b) {
  const double s = a + b;
  return DD{s, b - (s - a)};
}
__device__ __forceinline__ DD dd_add(DD a, DD b) {
  DD s = two_sum(a.hi, b.hi);
  s.lo += a.lo + b.lo;
  return fast_two_sum(s.hi, s.lo);
}
__device__ __forceinline__ DD dd_add1(DD a, double x) {
  DD s = two_sum(a.hi, x);
  s.lo += a.lo;
  return fast_two_sum(s.hi, s.lo);
}

// kNan false: cells summed are the non-infinite ones (clampInfsToMean);
// true: the non-NaN ones (clampNansToMean).
template <bool kNan>
__device__ __forceinline__ bool summed(double v) {
  return kNan ? !isnan(v) : !isinf(v);
}

struct Acc {
  DD s;
  double special;  // sum of the summed non-finite cells: 0, +-inf or NaN
  double count;    // exact below 2^53 cells
};

__device__ __forceinline__ Acc acc_add(Acc a, const Acc& b) {
  a.s = dd_add(a.s, b.s);
  a.special += b.special;
  a.count += b.count;
  return a;
}

// block reduction in a fixed order (tree over the 256 lanes through LDS)
__device__ Acc block_reduce(Acc a) {
  __shared__ double s_hi[kOpsBlock], s_lo[kOpsBlock], s_sp[kOpsBlock], s_ct[kOpsBlock];
  const int t = threadIdx.x;
  s_hi[t] = a.s.hi;
  s_lo[t] = a.s.lo;
  s_sp[t] = a.special;
  s_ct[t] = a.count;
  __syncthreads();
  for (int w = kOpsBlock / 2; w > 0; w >>= 1) {
    if (t < w) {
      Acc x{{s_hi[t], s_lo[t]}, s_sp[t], s_ct[t]};
      const Acc y{{s_hi[t + w], s_lo[t + w]}, s_sp[t + w], s_ct[t + w]};
      x = acc_add(x, y);
      s_hi[t] = x.s.hi;
      s_lo[t] = x.s.lo;
      s_sp[t] = x.special;
      s_ct[t] = x.count;
    }
    __syncthreads();
  }
  return Acc{{s_hi[0], s_lo[0]}, s_sp[0], s_ct[0]};
}

__device__ __forceinline__ void store_part(double* __restrict__ part, int64_t at, const Acc& a) {
  double* p = part + 4 * at;
  p[0] = a.s.hi;
  p[1] = a.s.lo;
  p[2] = a.special;
  p[3] = a.count;
}
// the partials of one sum combined by one block, in a fixed order
__device__ Acc combine(const double* __restrict__ part, int nparts) {
  Acc a{{0.0, 0.0}, 0.0, 0.0};
  for (int i = threadIdx.x; i < nparts; i += kOpsBlock) {
    const double* p = part + 4 * (int64_t)i;
    a = acc_add(a, Acc{{p[0], p[1]}, p[2], p[3]});
  }
  return block_reduce(a);
}
__device__ __forceinline__ double total_of(const Acc& a) {
  return isfinite(a.special) ? a.s.hi + a.s.lo : a.special;
}
__device__ __forceinline__ void acc_sum(Acc& a, double v) {
  if (isfinite(v)) a.s = dd_add1(a.s, v);
  else a.special += v;
}
__device__ __forceinline__ void acc_value(Acc& a, double v) {
  a.count += 1.0;
  acc_sum(a, v);
}

template <bool kNan>
__global__ __launch_bounds__(kOpsBlock) void k_mean_partials(const double* __restrict__ f, int64_t n,
                                                            double* __restrict__ part) {
  Acc a{{0.0, 0.0}, 0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double v = f[i];
    if (summed<kNan>(v)) acc_value(a, v);
  }
  a = block_reduce(a);
  if (threadIdx.x == 0) store_part(part, blockIdx.x, a);
}

// one block: combine the partials, write [mean, count] after them (and the
// mean to pinned host memory when the caller reads it)
__global__ __launch_bounds__(kOpsBlock) void k_mean_final(double* __restrict__ part, int nparts,
                                                          double* __restrict__ h_mean) {
  const Acc a = combine(part, nparts);
  if (threadIdx.x == 0) {
    // Real mean = sum / nonInfsSeen: 0 / 0 is NaN when no cell is summed
    const double mean = total_of(a) / a.count;
    part[4 * (int64_t)nparts] = mean;
    part[4 * (int64_t)nparts + 1] = a.count;
    if (h_mean) *h_mean = mean;
  }
}

// mean_at: [mean, count of summed cells]; when every cell was summed there is
// nothing to replace and the field is not read again
template <bool kNan>
__global__ __launch_bounds__(kOpsBlock) void k_replace(double* __restrict__ f, int64_t n,
                                                       const double* __restrict__ mean_at) {
  if (mean_at[1] == (double)n) return;  // the same for every thread of the grid
  const double mean = mean_at[0];
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double v = f[i];
    if (kNan ? isnan(v) : isinf(v)) f[i] = mean;
  }
}

// the six faces: z = 0, Z-1 (X*Y cells each), y = 0, Y-1 (X*Z), x = 0, X-1 (Y*Z)
__global__ __launch_bounds__(kOpsBlock) void k_set_borders(double* __restrict__ f, int64_t X, int64_t Y, int64_t Z,
                                                           double value) {
  const int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x;
  const int64_t nz = X * Y, ny = X * Z, nx = Y * Z;
  int64_t x, y, z;
  if (i < 2 * nz) {
    const int64_t r = i % nz;
    x = r % X;
    y = r / X;
    z = i < nz ? 0 : Z - 1;
  } else if (i < 2 * (nz + ny)) {
    const int64_t j = i - 2 * nz, r = j % ny;
    x = r % X;
    z = r / X;
    y = j < ny ? 0 : Y - 1;
  } else if (i < 2 * (nz + ny + nx)) {
    const int64_t j = i - 2 * (nz + ny), r = j % nx;
    y = r % Y;
    z = r / Y;
    x = j < nx ? 0 : X - 1;
  } else {
    return;
  }
  f[x + y * X + z * X * Y] = value;
}

// ---------------------------------------------------------------- scoring fields of the shape optimizer

// outerShell + innerShell (FIELD_3D.cpp:5070-5145): whether the cell has a
// 26-neighbour of the other sign (cells at 0 have none)
__device__ __forceinline__ bool shell_cell(const double* __restrict__ d, int64_t i, int64_t x, int64_t y, int64_t z,
                                           int64_t X, int64_t Y, int64_t Z) {
  const int64_t XY = X * Y;
  const double c = d[i];
  bool flip = false;
  for (int k = -1; k <= 1; k++)
    for (int j = -1; j <= 1; j++)
      for (int h = -1; h <= 1; h++) {
        if (h == 0 && j == 0 && k == 0) continue;
        const int64_t xn = x + h, yn = y + j, zn = z + k;
        if (xn < 0 || xn > X - 1 || yn < 0 || yn > Y - 1 || zn < 0 || zn > Z - 1) continue;
        if (d[xn + yn * X + zn * XY] * c < 0) flip = true;
      }
  return flip;
}

// The layer numbers of invertedDistance (FIELD_3D.cpp:5248-5283: shell cells 1,
// then sweep after sweep every unnumbered cell 1 + its smallest 6-neighbour)
// are 1 + the taxicab distance to the nearest shell cell, and that distance is
// separable: one pass per axis, each the minimum over the line of value +
// distance along it. (The sweeps took one launch, one counter read-back and
// one wait each, about half the grid's edge of them: 50^3 25 sweeps, 1.5 ms.)
// A block takes 16 lines of one axis (4 rows for the
// x pass, whose shells make most of the work: a cell per thread at 50^3); the minimum over a line of n cells by
// doubling, v[i] = min(v[i], v[i - d] + d, v[i + d] + d) for d = 1, 2, 4, ... < n,
// between two LDS copies. Lines of neighbouring x are taken together along y and
// z, so that loads stay in runs of 64 B. The x pass starts from the shells; the
// z pass writes the inverted, signed value (FIELD_3D.cpp:5286-5296: 1 / number,
// negated inside and quartered outside) and the partial sums of its absolute
// value; part's last entry counts the cells no shell reaches. Latency bound:
// 50^3: 10 us along x (625 blocks; 21.5 with 16 rows each), 7 along y and 9 along z
// (157 blocks).
constexpr int kMaxLine = 512;
constexpr int lines_of(int axis) { return axis == 0 ? 4 : 16; }
constexpr uint32_t kFar = 0x3fffffffu;  // no shell cell on the lines so far
enum LineAxis { kAxisX = 0, kAxisY = 1, kAxisZ = 2 };

__device__ __forceinline__ double inverted_value(uint32_t layers, double dist) {
  double x = 1.0 / ((double)layers + 1.0);
  if (dist < 0) x *= -1;
  else x *= 0.25;
  return x;
}

template <int kAxis>
__global__ __launch_bounds__(kOpsBlock) void k_layers(const double* __restrict__ d, int64_t X, int64_t Y, int64_t Z,
                                                      uint32_t* __restrict__ lay, double* __restrict__ out,
                                                      double* __restrict__ part) {
  constexpr int kLines = lines_of(kAxis);
  extern __shared__ uint32_t s_v[];  // 2 x n x kLines
  const int64_t XY = X * Y;
  const int n = (int)(kAxis == kAxisX ? X : kAxis == kAxisY ? Y : Z);
  // the block's lines: consecutive rows (x), consecutive x of one z (y), consecutive x + y X (z)
  const int64_t per = kAxis == kAxisX ? Y * Z : kAxis == kAxisY ? X : XY;
  const int64_t groups = (per + kLines - 1) / kLines;
  const int64_t outer = blockIdx.x / groups, l0 = (blockIdx.x - outer * groups) * kLines;
  const int lines = (int)(per - l0 < kLines ? per - l0 : kLines);
  uint32_t *cur = s_v, *nxt = s_v + n * kLines;
  const int total = n * kLines;
  // element e: line e / n of a row block (x: memory order), else position e / kLines of line e % kLines
  auto place = [&](int e, int& line, int& pos, int64_t& at) {
    if (kAxis == kAxisX) {
      line = e / n;
      pos = e - line * n;
      at = (l0 + line) * X + pos;
    } else {
      line = e % kLines;
      pos = e / kLines;
      at = kAxis == kAxisY ? outer * XY + pos * X + l0 + line : pos * XY + l0 + line;
    }
  };
  for (int e = threadIdx.x; e < total; e += kOpsBlock) {
    int line, pos;
    int64_t at;
    place(e, line, pos, at);
    uint32_t v = kFar;
    if (line < lines) {
      if (kAxis == kAxisX) {
        const int64_t row = l0 + line, z = row / Y;
        v = shell_cell(d, at, pos, row - z * Y, z, X, Y, Z) ? 0u : kFar;
      } else {
        v = lay[at];
      }
    }
    cur[pos * kLines + line] = v;
  }
  __syncthreads();
  for (int step = 1; step < n; step *= 2) {
    for (int e = threadIdx.x; e < total; e += kOpsBlock) {
      const int pos = e / kLines;
      uint32_t v = cur[e];
      if (pos >= step) v = min(v, cur[e - step * kLines] + step);
      if (pos + step < n) v = min(v, cur[e + step * kLines] + step);
      nxt[e] = v;
    }
    __syncthreads();
    uint32_t* t = cur;
    cur = nxt;
    nxt = t;
  }
  Acc a{{0.0, 0.0}, 0.0, 0.0};
  unsigned far = 0;
  for (int e = threadIdx.x; e < total; e += kOpsBlock) {
    int line, pos;
    int64_t at;
    place(e, line, pos, at);
    if (line >= lines) continue;
    const uint32_t v = cur[pos * kLines + line];
    if (kAxis != kAxisZ) {
      lay[at] = v < kFar ? v : kFar;
    } else {
      far += v >= kFar;
      const double x = inverted_value(v, d[at]);
      out[at] = x;
      acc_value(a, fabs(x));
    }
  }
  if (kAxis == kAxisZ) {
    a.count = (double)far;  // what the partial carries here: the cells without a number
    a = block_reduce(a);
    if (threadIdx.x == 0) store_part(part, blockIdx.x, a);
  }
}

// The same passes for lines beyond kMaxLine cells (their two LDS copies would
// not fit): one line per thread, forward and back.
template <int kAxis>
__global__ __launch_bounds__(kOpsBlock) void k_layers_long(const double* __restrict__ d, int64_t X, int64_t Y,
                                                           int64_t Z, uint32_t* __restrict__ lay,
                                                           double* __restrict__ out, double* __restrict__ part) {
  const int64_t XY = X * Y, n = kAxis == kAxisX ? X : kAxis == kAxisY ? Y : Z;
  const int64_t stride = kAxis == kAxisX ? 1 : kAxis == kAxisY ? X : XY;
  const int64_t count = XY * Z / n, l = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x;
  Acc a{{0.0, 0.0}, 0.0, 0.0};
  if (l < count) {
    const int64_t first = kAxis == kAxisX ? l * X : kAxis == kAxisY ? (l / X) * XY + l % X : l;
    uint32_t v = kFar;
    for (int64_t p = 0; p < n; p++) {
      const int64_t at = first + p * stride;
      const uint32_t own = kAxis == kAxisX ? (shell_cell(d, at, p, l % Y, l / Y, X, Y, Z) ? 0u : kFar) : lay[at];
      v = min(own, v < kFar ? v + 1 : kFar);
      lay[at] = v;
    }
    double far = 0.0;
    for (int64_t p = n - 1; p >= 0; p--) {
      const int64_t at = first + p * stride;
      v = min(lay[at], v < kFar ? v + 1 : kFar);
      if (kAxis != kAxisZ) {
        lay[at] = v;
      } else {
        far += v >= kFar;
        const double x = inverted_value(v, d[at]);
        out[at] = x;
        acc_value(a, fabs(x));
      }
    }
    a.count = far;
  }
  if (kAxis == kAxisZ) {
    a = block_reduce(a);
    if (threadIdx.x == 0) store_part(part, blockIdx.x, a);
  }
}

// invertedDistanceNormalized's passes (FIELD_3D.cpp:5316-5352), each with the
// sums the next one needs: kStage 0 scales by 1 / the absolute sum and sums the
// inside and the outside (two partials per block), 1 scales those to absolute
// sum 0.5 each and sums absolute values. scal: what k_fold_sums left.
template <int kStage>
__global__ __launch_bounds__(kOpsBlock) void k_normalize(double* __restrict__ v, const double* __restrict__ d,
                                                         int64_t n, const double* __restrict__ scal,
                                                         double* __restrict__ part) {
  Acc a{{0.0, 0.0}, 0.0, 0.0}, b = a;
  const double s_in = kStage == 0 ? 1.0 / scal[0] : 0.5 / fabs(scal[0]);
  const double s_out = kStage == 0 ? s_in : 0.5 / fabs(scal[1]);
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const bool inside = d[i] < 0;
    const double x = v[i] * (inside ? s_in : s_out);
    v[i] = x;
    if (kStage == 0) acc_value(inside ? a : b, x);
    else acc_value(a, fabs(x));
  }
  a = block_reduce(a);
  if (threadIdx.x == 0) store_part(part, blockIdx.x, a);
  if (kStage == 0) {
    __syncthreads();
    b = block_reduce(b);
    if (threadIdx.x == 0) store_part(part, (int64_t)gridDim.x + blockIdx.x, b);
  }
}

// Block b: the total of partials [b nparts, (b + 1) nparts) (nlast of them in the
// last block) to d_out[b] and, with h_out, to pinned host memory; count0: the first one's count there too.
__global__ __launch_bounds__(kOpsBlock) void k_fold_sums(const double* __restrict__ part, int nparts,
                                                         int nlast, double* __restrict__ d_out, double* __restrict__ h_out,
                                                         double* __restrict__ h_count) {
  const Acc a = combine(part + 4 * (int64_t)blockIdx.x * nparts,
                        blockIdx.x + 1 == gridDim.x ? nlast : nparts);
  if (threadIdx.x == 0) {
    const double t = total_of(a);
    if (d_out) d_out[blockIdx.x] = t;
    if (h_out) h_out[blockIdx.x] = t;
    if (h_count && blockIdx.x == 0) *h_count = a.count;
  }
}

// The weight at the centre of cell i (the trilinear lookup). small: fewer than 2^32 cells.
__device__ __forceinline__ double cell_weight(const GridGeom& g, const GridGeom& wg, const double* __restrict__ w,
                                              int64_t i, bool small) {
  const int64_t X = g.res[0], XY = X * g.res[1];
  int64_t x, y, z;
  if (small) {
    const uint32_t p = (uint32_t)i, zu = fast_div(p, g.div_xy), r = p - zu * (uint32_t)XY;
    const uint32_t yu = fast_div(r, g.div_x);
    z = zu;
    y = yu;
    x = r - yu * (uint32_t)X;
  } else {
    z = i / XY;
    const int64_t r = i - z * XY;
    y = r / X;
    x = r - y * X;
  }
  double c[3];
  cell_center(g, (int)x, (int)y, (int)z, c);
  return field_lookup(wg, w, c);
}

// The weight at every cell and the partial sums of its absolute value: once per
// call, where the score kernel repeated both for every threshold.
__global__ __launch_bounds__(kOpsBlock) void k_cell_weights(GridGeom g, GridGeom wg, const double* __restrict__ w,
                                                            double* __restrict__ out, double* __restrict__ part) {
  const int64_t n = (int64_t)g.res[0] * g.res[1] * g.res[2];
  const bool small = n <= (int64_t)0xffffffffll;
  Acc a{{0.0, 0.0}, 0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double wt = cell_weight(g, wg, w, i, small);
    out[i] = wt;
    acc_sum(a, fabs(wt));
  }
  a = block_reduce(a);
  if (threadIdx.x == 0) store_part(part, blockIdx.x, a);
}

// weightScore / inverseDistanceScore (OPTIMIZE_3D.cpp:4502-4563) for kScores
// thresholds from blockIdx.y kScores on: the partial sums of
// -tanh(alpha (F - threshold)) w(cell centre). FP64 VALU bound (the tanh); the
// field and the cells' weights are read once per kScores thresholds. 50^3, 100
// thresholds: 39 us; one threshold per block with the lookup and the library's
// tanh 169 us, this split with the library's tanh 67 us, with a tanh of 2.6
// instead of 0.81 ulp 34 us.
constexpr int kScores = 4;
__global__ __launch_bounds__(kOpsBlock) void k_weight_score(const double* __restrict__ f,
                                                            const double* __restrict__ cw, int64_t n,
                                                            const double* __restrict__ thresholds, int nthr,
                                                            double alpha, double* __restrict__ part) {
  const int t0 = blockIdx.y * kScores;
  Acc a[kScores];
  double thr[kScores];
#pragma unroll
  for (int k = 0; k < kScores; k++) {
    a[k] = Acc{{0.0, 0.0}, 0.0, 0.0};
    thr[k] = thresholds[t0 + k < nthr ? t0 + k : nthr - 1];
  }
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double F = f[i], w = cw[i];
#pragma unroll
    for (int k = 0; k < kScores; k++) acc_sum(a[k], -tanh64(alpha * (F - thr[k])) * w);
  }
#pragma unroll
  for (int k = 0; k < kScores; k++) {
    const Acc s = block_reduce(a[k]);
    if (threadIdx.x == 0 && t0 + k < nthr) store_part(part, (int64_t)(t0 + k) * gridDim.x + blockIdx.x, s);
    __syncthreads();
  }
}

// The same for at most kScores thresholds (kN of them) in one pass: lookup, scores and
// the weights' absolute sum (slot kN) together, with no array of cell weights between.
// Up to 1024 blocks. FP64 VALU bound. One threshold, 128^3, 256^3 and 300^3: 47, 156
// and 232 us; by the two kernels, which take four thresholds for one and 8 bytes a
// cell, 84, 388 and 962; a lookup per threshold and the library's tanh 76, 332 and 511.
struct FewThresholds {
  double t[kScores];
};
template <int kN>
__global__ __launch_bounds__(kOpsBlock) void k_few_scores(const double* __restrict__ f, GridGeom g, GridGeom wg,
                                                          const double* __restrict__ w, FewThresholds thr,
                                                          double alpha, double* __restrict__ part) {
  const int64_t n = (int64_t)g.res[0] * g.res[1] * g.res[2];
  const bool small = n <= (int64_t)0xffffffffll;
  Acc a[kN + 1];
#pragma unroll
  for (int k = 0; k <= kN; k++) a[k] = Acc{{0.0, 0.0}, 0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double wt = cell_weight(g, wg, w, i, small);
    if (kN) {
      const double F = f[i];
#pragma unroll
      for (int k = 0; k < kN; k++) acc_sum(a[k], -tanh64(alpha * (F - thr.t[k])) * wt);
    }
    acc_sum(a[kN], fabs(wt));
  }
#pragma unroll
  for (int k = 0; k <= kN; k++) {
    const Acc s = block_reduce(a[k]);
    if (threadIdx.x == 0) store_part(part, (int64_t)k * gridDim.x + blockIdx.x, s);
    __syncthreads();
  }
}

// fieldMin / fieldMax (FIELD_3D.cpp:2960-2971, 3021-3032): the serial scan
// keeps the first cell that compares smaller (larger), starting from cell 0,
// so NaN cells are skipped unless cell 0 is NaN, and of equal values (0 and
// -0) the first wins. Reduced as (value, index) pairs with the index breaking
// ties; NaN cells never win.
struct VI {
  double v;
  int64_t i;
};
__device__ __forceinline__ VI vi_min(VI a, VI b) {
  if (b.i < 0) return a;
  if (a.i < 0) return b;
  return (b.v < a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
__device__ __forceinline__ VI vi_max(VI a, VI b) {
  if (b.i < 0) return a;
  if (a.i < 0) return b;
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

// the block's extrema in thread 0's mn and mx
__device__ void extrema_reduce(VI& mn, VI& mx, double (*s_v)[kOpsBlock], int64_t (*s_i)[kOpsBlock]) {
  const int t = threadIdx.x;
  s_v[0][t] = mn.v;
  s_i[0][t] = mn.i;
  s_v[1][t] = mx.v;
  s_i[1][t] = mx.i;
  __syncthreads();
  for (int w = kOpsBlock / 2; w > 0; w >>= 1) {
    if (t < w) {
      const VI a = vi_min(VI{s_v[0][t], s_i[0][t]}, VI{s_v[0][t + w], s_i[0][t + w]});
      const VI b = vi_max(VI{s_v[1][t], s_i[1][t]}, VI{s_v[1][t + w], s_i[1][t + w]});
      s_v[0][t] = a.v;
      s_i[0][t] = a.i;
      s_v[1][t] = b.v;
      s_i[1][t] = b.i;
    }
    __syncthreads();
  }
  mn = VI{s_v[0][0], s_i[0][0]};
  mx = VI{s_v[1][0], s_i[1][0]};
}

__global__ __launch_bounds__(kOpsBlock) void k_min_max(const double* __restrict__ f, int64_t n,
                                                       double* __restrict__ part) {
  __shared__ double s_v[2][kOpsBlock];
  __shared__ int64_t s_i[2][kOpsBlock];
  VI mn{0.0, -1}, mx{0.0, -1};
  const int64_t stride = (int64_t)gridDim.x * kOpsBlock;
  for (int64_t i = (int64_t)blockIdx.x * kOpsBlock + threadIdx.x; i < n; i += stride) {
    const double v = f[i];
    if (isnan(v)) continue;
    mn = vi_min(mn, VI{v, i});
    mx = vi_max(mx, VI{v, i});
  }
  extrema_reduce(mn, mx, s_v, s_i);
  if (threadIdx.x == 0) {
    double* p = part + 4 * (int64_t)blockIdx.x;
    p[0] = mn.v;
    p[1] = (double)mn.i;  // exact: indexes stay below 2^53
    p[2] = mx.v;
    p[3] = (double)mx.i;
  }
}

// one block: the extrema of the blocks' extrema, to pinned host memory. A NaN
// in cell 0 makes both NaN (nothing compares against a NaN start).
__global__ __launch_bounds__(kOpsBlock) void k_min_max_final(const double* __restrict__ part, int nparts,
                                                             const double* __restrict__ f, double* __restrict__ h) {
  __shared__ double s_v[2][kOpsBlock];
  __shared__ int64_t s_i[2][kOpsBlock];
  VI mn{0.0, -1}, mx{0.0, -1};
  for (int i = threadIdx.x; i < nparts; i += kOpsBlock) {
    const double* p = part + 4 * (int64_t)i;
    mn = vi_min(mn, VI{p[0], (int64_t)p[1]});
    mx = vi_max(mx, VI{p[2], (int64_t)p[3]});
  }
  extrema_reduce(mn, mx, s_v, s_i);
  if (threadIdx.x == 0) {
    const bool nan = isnan(f[0]);
    h[0] = nan ? f[0] : mn.v;
    h[1] = nan ? f[0] : mx.v;
  }
}

}  // namespace

qj_status field_clamp_to_mean(qj_workspace* ws, double* d_field, int64_t n, bool nans, double* mean_out,
                              hipStream_t s) {
  if (n <= 0) {
    if (mean_out) *mean_out = NAN;  // 0 / 0: no cell is summed
    return QJ_OK;
  }
  qj_status st = ensure_partials(ws, 4 * (int64_t)kOpsGrid + 2, s);
  if (st) return st;
  const int64_t want = (n + kOpsBlock - 1) / kOpsBlock;
  const int grid = (int)(want < kOpsGrid ? want : kOpsGrid);
  if (nans) hipLaunchKernelGGL(k_mean_partials<true>, dim3(grid), dim3(kOpsBlock), 0, s, d_field, n, ws->d_partials);
  else hipLaunchKernelGGL(k_mean_partials<false>, dim3(grid), dim3(kOpsBlock), 0, s, d_field, n, ws->d_partials);
  QJ_HIP(hipGetLastError());
  if (mean_out && (st = ensure_pinned(ws, 1, s))) return st;
  hipLaunchKernelGGL(k_mean_final, dim3(1), dim3(kOpsBlock), 0, s, ws->d_partials, grid,
                     mean_out ? ws->h_pinned : (double*)nullptr);
  QJ_HIP(hipGetLastError());
  const double* mean_at = ws->d_partials + 4 * (int64_t)grid;
  if (nans) hipLaunchKernelGGL(k_replace<true>, dim3(grid), dim3(kOpsBlock), 0, s, d_field, n, mean_at);
  else hipLaunchKernelGGL(k_replace<false>, dim3(grid), dim3(kOpsBlock), 0, s, d_field, n, mean_at);
  QJ_HIP(hipGetLastError());
  if (mean_out) {
    QJ_HIP(hipStreamSynchronize(s));
    *mean_out = ws->h_pinned[0];
  }
  return QJ_OK;
}

qj_status field_set_borders(const int32_t* res, double value, double* d_field, hipStream_t s) {
  const int64_t X = res[0], Y = res[1], Z = res[2];
  const int64_t m = 2 * (X * Y + X * Z + Y * Z);
  const int64_t blocks = (m + kOpsBlock - 1) / kOpsBlock;
  if (blocks > INT32_MAX) return QJ_ERR_CAPACITY;
  hipLaunchKernelGGL(k_set_borders, dim3((unsigned)blocks), dim3(kOpsBlock), 0, s, d_field, X, Y, Z, value);
  QJ_HIP(hipGetLastError());
  return QJ_OK;
}

}  // namespace qj

namespace qj {

// Per-cell scratch of a call: kept in the workspace up to kKeepCells cells
// (128 MiB), a temporary of the call beyond, so that one call on a huge grid
// does not hold its memory.
constexpr int64_t kKeepCells = int64_t(1) << 24;
struct CellScratch {
  void* p = nullptr;
  bool own = false;
  ~CellScratch() {
    if (own) (void)hipFree(p);
  }
};

template <int kAxis>
static qj_status launch_layers(const double* d, int64_t X, int64_t Y, int64_t Z, uint32_t* lay, double* out,
                               double* part, int64_t* blocks, hipStream_t s) {
  const int64_t n = kAxis == kAxisX ? X : kAxis == kAxisY ? Y : Z, lines = X * Y * Z / n;
  if (n <= kMaxLine) {
    constexpr int kLines = lines_of(kAxis);
    const int64_t per = kAxis == kAxisY ? X : lines, outer = kAxis == kAxisY ? Z : 1;
    *blocks = outer * ((per + kLines - 1) / kLines);
    if (*blocks > INT32_MAX) return QJ_ERR_CAPACITY;
    hipLaunchKernelGGL(k_layers<kAxis>, dim3((unsigned)*blocks), dim3(kOpsBlock),
                       2 * sizeof(uint32_t) * kLines * (size_t)n, s, d, X, Y, Z, lay, out, part);
  } else {
    *blocks = (lines + kOpsBlock - 1) / kOpsBlock;
    if (*blocks > INT32_MAX) return QJ_ERR_CAPACITY;
    hipLaunchKernelGGL(k_layers_long<kAxis>, dim3((unsigned)*blocks), dim3(kOpsBlock), 0, s, d, X, Y, Z, lay, out,
                       part);
  }
  QJ_HIP(hipGetLastError());
  return QJ_OK;
}

// Three layer passes, then (normalized) two scaling passes, every sum folded on
// the device: one wait at the end.
qj_status field_inverted_distance(qj_workspace* ws, const double* d_dist, const qj_grid* grid, bool normalized,
                                  double* d_out, double* abs_sum, hipStream_t s) {
  const int64_t X = grid->res[0], Y = grid->res[1], Z = grid->res[2], n = X * Y * Z;
  if (n <= 0) return QJ_OK;
  const int64_t zlines = X * Y;
  const int64_t zblocks = Z <= kMaxLine ? (zlines + lines_of(kAxisZ) - 1) / lines_of(kAxisZ) : (zlines + kOpsBlock - 1) / kOpsBlock;
  const int64_t want = (n + kOpsBlock - 1) / kOpsBlock;
  const int grid_sum = (int)(want < kOpsGrid ? want : kOpsGrid);
  const int64_t nparts = std::max<int64_t>(zblocks, 2 * (int64_t)grid_sum);
  const bool keep = n <= kKeepCells;
  qj_status st = ensure_partials(ws, 4 * nparts + 2 + (keep ? (n + 1) / 2 : 0), s);
  if (st) return st;
  if ((st = ensure_pinned(ws, 2, s))) return st;
  double* part = ws->d_partials;
  double* scal = part + 4 * nparts;
  CellScratch cells;
  if (keep) cells.p = scal + 2;
  else QJ_HIP(hipMalloc(&cells.p, sizeof(uint32_t) * (size_t)n));
  cells.own = !keep;
  uint32_t* lay = (uint32_t*)cells.p;
  int64_t nb = 0;
  if ((st = launch_layers<kAxisX>(d_dist, X, Y, Z, lay, d_out, part, &nb, s)) ||
      (st = launch_layers<kAxisY>(d_dist, X, Y, Z, lay, d_out, part, &nb, s)) ||
      (st = launch_layers<kAxisZ>(d_dist, X, Y, Z, lay, d_out, part, &nb, s)))
    return st;
  // h_pinned: [0] the absolute sum of the result, [1] the cells without a number
  double* h = ws->h_pinned;
  hipLaunchKernelGGL(k_fold_sums, dim3(1), dim3(kOpsBlock), 0, s, (const double*)part, (int)nb, (int)nb, scal, h,
                     h + 1);
  QJ_HIP(hipGetLastError());
  if (normalized) {
    hipLaunchKernelGGL(k_normalize<0>, dim3(grid_sum), dim3(kOpsBlock), 0, s, d_out, d_dist, n, (const double*)scal,
                       part);
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_fold_sums, dim3(2), dim3(kOpsBlock), 0, s, (const double*)part, grid_sum, grid_sum, scal,
                       (double*)nullptr, (double*)nullptr);
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_normalize<1>, dim3(grid_sum), dim3(kOpsBlock), 0, s, d_out, d_dist, n, (const double*)scal,
                       part);
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_fold_sums, dim3(1), dim3(kOpsBlock), 0, s, (const double*)part, grid_sum, grid_sum,
                       (double*)nullptr, h, (double*)nullptr);
    QJ_HIP(hipGetLastError());
  }
  QJ_HIP(hipStreamSynchronize(s));
  if (h[1] > 0.0) {
    // a cell that no shell cell reaches: the reference's sweeps never end
    set_error("inverted distance: %.0f cells can never be numbered (no surface reaches them)", h[1]);
    return QJ_ERR_NUMERIC;
  }
  if (abs_sum) *abs_sum = h[0];
  return QJ_OK;
}

qj_status field_min_max(qj_workspace* ws, const double* d_field, int64_t n, double* mn, double* mx, hipStream_t s) {
  if (n <= 0) return QJ_ERR_INVALID;
  const int64_t want = (n + kOpsBlock - 1) / kOpsBlock;
  const int grid = (int)(want < kOpsGrid ? want : kOpsGrid);
  qj_status st = ensure_partials(ws, 4 * (int64_t)grid, s);
  if (st) return st;
  if ((st = ensure_pinned(ws, 2, s))) return st;
  hipLaunchKernelGGL(k_min_max, dim3(grid), dim3(kOpsBlock), 0, s, d_field, n, ws->d_partials);
  QJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_min_max_final, dim3(1), dim3(kOpsBlock), 0, s, (const double*)ws->d_partials, grid, d_field,
                     ws->h_pinned);
  QJ_HIP(hipGetLastError());
  QJ_HIP(hipStreamSynchronize(s));
  *mn = ws->h_pinned[0];
  *mx = ws->h_pinned[1];
  return QJ_OK;
}

qj_status weight_scores(qj_workspace* ws, const double* d_field, const qj_grid* grid, const qj_grid* wgrid,
                        const double* d_weight, double alpha, const double* thresholds, int nthr, double* scores,
                        double* max_score, hipStream_t s) {
  GridGeom g, wg;
  make_geom(grid, &g);
  make_geom(wgrid, &wg);
  const int64_t n = (int64_t)g.res[0] * g.res[1] * g.res[2];
  if (n <= 0 || nthr < 0) return QJ_ERR_INVALID;
  const int slots = nthr + 1;
  qj_status st;
  if (nthr <= kScores) {
    const int gx = (int)std::min<int64_t>((n + kOpsBlock - 1) / kOpsBlock, 1024);
    if ((st = ensure_partials(ws, 4 * (int64_t)gx * slots, s))) return st;
    if ((st = ensure_pinned(ws, slots, s))) return st;
    FewThresholds few{};
    for (int t = 0; t < nthr; t++) few.t[t] = thresholds[t];
    const auto k = nthr == 0   ? k_few_scores<0>
                   : nthr == 1 ? k_few_scores<1>
                   : nthr == 2 ? k_few_scores<2>
                   : nthr == 3 ? k_few_scores<3>
                               : k_few_scores<4>;
    hipLaunchKernelGGL(k, dim3(gx), dim3(kOpsBlock), 0, s, d_field, g, wg, d_weight, few, alpha, ws->d_partials);
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_fold_sums, dim3(slots), dim3(kOpsBlock), 0, s, (const double*)ws->d_partials, gx, gx,
                       (double*)nullptr, ws->h_pinned, (double*)nullptr);
    QJ_HIP(hipGetLastError());
    QJ_HIP(hipStreamSynchronize(s));
    for (int t = 0; t < nthr; t++) scores[t] = ws->h_pinned[t];
    if (max_score) *max_score = ws->h_pinned[nthr];
    return QJ_OK;
  }
  // up to 8 cells per thread where the thresholds fill the chip by themselves:
  // the four block sums cost as much as some 10 cells (50^3, 100 thresholds: 6400
  // blocks of 2 cells take a fifth longer than 1750)
  const int64_t want = (n + kOpsBlock - 1) / kOpsBlock, ny = (nthr + kScores - 1) / kScores;
  const int64_t per = std::min<int64_t>(8, std::max<int64_t>(1, want * ny / 1536));
  const int gx = (int)std::min<int64_t>((want + per - 1) / per, 256);
  const int gw = (int)std::min<int64_t>(want, 256);
  // the partials (the last slot's: the weights' absolute sum), the thresholds, the cells' weights
  const bool keep = n <= kKeepCells;
  if ((st = ensure_partials(ws, 4 * ((int64_t)gx * nthr + gw) + (int64_t)slots + (keep ? n : 0), s))) return st;
  if ((st = ensure_pinned(ws, 2 * (int64_t)slots, s))) return st;
  double* part = ws->d_partials;
  double* d_thr = part + 4 * ((int64_t)gx * nthr + gw);
  CellScratch cells;
  if (keep) cells.p = d_thr + slots;
  else QJ_HIP(hipMalloc(&cells.p, sizeof(double) * (size_t)n));
  cells.own = !keep;
  double* cw = (double*)cells.p;
  hipLaunchKernelGGL(k_cell_weights, dim3(gw), dim3(kOpsBlock), 0, s, g, wg, d_weight, cw,
                     part + 4 * (int64_t)gx * nthr);
  QJ_HIP(hipGetLastError());
  double* h_thr = ws->h_pinned + slots;
  for (int t = 0; t < nthr; t++) h_thr[t] = thresholds[t];
  QJ_HIP(hipMemcpyAsync(d_thr, h_thr, sizeof(double) * (size_t)nthr, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_weight_score, dim3(gx, (unsigned)ny), dim3(kOpsBlock), 0, s, d_field,
                     (const double*)cw, n, (const double*)d_thr, nthr, alpha, part);
  QJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_fold_sums, dim3(slots), dim3(kOpsBlock), 0, s, (const double*)part, gx, gw,
                     (double*)nullptr, ws->h_pinned, (double*)nullptr);
  QJ_HIP(hipGetLastError());
  QJ_HIP(hipStreamSynchronize(s));
  for (int t = 0; t < nthr; t++) scores[t] = ws->h_pinned[t];
  if (max_score) *max_score = ws->h_pinned[nthr];
  return QJ_OK;
}

}  // namespace qj
