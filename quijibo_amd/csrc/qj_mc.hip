// Marching cubes on a resident field (TRIANGLE_MESH(const FIELD_3D&) ->
// computeStagedMarchingCubes, TRIANGLE_MESH.cpp:989-1114), bit-exact with the
// CPU mesher: same flags, same vertex set and numbering, same vertex
// arithmetic, same triangle order, same degenerate filter.
//
// Pipeline per field (no host synchronisation between fields, see
// mc_run_tiles). The sign test is kept as one bit per grid point, so that the
// edges, cases and triangle counts of 64 points are a few operations on
// 64-bit words, and only vertices and triangles themselves take a lane each:
//   k_mc_signs      one bit per point: the float sign test
//   k_mc_edges      the +x, +y, +z edges that carry a vertex, and the vertices
//                   before every 8 points within a group (16384 points);
//                   its last block, or k_mc_scan: groups' vertex
//                   counts -> first vertex id per group (the reference numbers
//                   vertices by std::map<pair<int,int>> order = lower endpoint,
//                   then x<y<z)
//   k_mc_vertices   p0 + d0/(d0-d1) (p1-p0) at cell centres, no contraction,
//                   and a bit per edge whose vertex lies near an end (an FP32
//                   estimate)
//   k_mc_measure    the degenerate filter (edge < 1e-7 dropped) on the cells whose
//                   near vertices lie on edges that meet, where estimates do not
//                   decide it (kMeasureAll, kMeasureNear) and groups are few
//   k_mc_cells      triangle counts, and elsewhere the degenerate filter; its last
//                   block, or k_mc_scan: first triangle per group
//   k_mc_tris       each kept triangle written once, in cell then table order
#include <float.h>
#include <math.h>

#include <algorithm>
#include <vector>

#include "qj_eval.h"
#include "qj_geom.h"
#include "qj_internal.h"
#include "qj_mc_table.h"

namespace qj {

constexpr int kMcBlock = 256;

// edge id -> lower endpoint offset (dx,dy,dz) and axis
constexpr void edge_parts(int e, int& dx, int& dy, int& dz, int& axis) {
  if (e < 4) {
    axis = 0; dx = 0; dy = e & 1; dz = e >> 1;
  } else if (e < 8) {
    axis = 1; dx = e & 1; dy = 0; dz = (e >> 1) & 1;
  } else {
    axis = 2; dx = e & 1; dy = (e >> 1) & 1; dz = 0;
  }
}

struct McTables {
  signed char tri[256][16];
  unsigned char ntri[256];
  unsigned short emask[256];
  // per case row and triangle: the bit mask of its 3 edges, and its 3 edges in
  // table order, 4 bits each
  unsigned short tmask[256][5];
  unsigned short tedge[256][5];
  // the pairs of its edges that meet at a corner: bit 3 k + (xy, xz, yz) for
  // corner k = 4 dx + 2 dy + dz
  unsigned tpair[256][5];
};

constexpr McTables make_tables() {
  McTables t{QJ_MC_TRI_INIT, {}, {}, {}, {}, {}};
  for (int c = 0; c < 256; c++) {
    int n = 0;
    unsigned m = 0;
    for (int k = 0; k < 16 && t.tri[c][k] >= 0; k++) {
      n++;
      m |= 1u << t.tri[c][k];
    }
    t.ntri[c] = (unsigned char)(n / 3);
    t.emask[c] = (unsigned short)m;
    for (int q = 0; q < n / 3; q++) {
      unsigned tm = 0, tc = 0;
      for (int j = 0; j < 3; j++) {
        const int e = t.tri[c][3 * q + j];
        tm |= 1u << e;
        tc |= (unsigned)e << (4 * j);
      }
      t.tmask[c][q] = (unsigned short)tm;
      t.tedge[c][q] = (unsigned short)tc;
      for (int k = 0; k < 8; k++) {
        const int dx = k >> 2, dy = (k >> 1) & 1, dz = k & 1;
        const bool x = tm >> (dy + 2 * dz) & 1, y = tm >> (4 + dx + 2 * dz) & 1, z = tm >> (8 + dx + 2 * dy) & 1;
        t.tpair[c][q] |= (unsigned)((x && y) | (x && z) << 1 | (y && z) << 2) << (3 * k);
      }
    }
  }
  return t;
}

constexpr McTables kMcHost = make_tables();
__constant__ McTables kMc = make_tables();

// The triangle table staged in LDS for the kernels that look it up per lane: with
// divergent indices, reads of __constant__ memory are scattered vector loads;
// from LDS they are ds_reads.
static_assert(kMcBlock == 256, "one table entry per thread");

// s_tri: the 256 x 16 triangle table as 1024 words; s_ntri: triangles per case
__device__ __forceinline__ void stage_tri(uint32_t* s_tri, uint8_t* s_ntri) {
  const uint32_t* src = (const uint32_t*)&kMc.tri[0][0];
  for (int i = threadIdx.x; i < 1024; i += kMcBlock) s_tri[i] = src[i];
  s_ntri[threadIdx.x] = kMc.ntri[threadIdx.x];
  __syncthreads();
}

__device__ __forceinline__ int tri_edge(const uint32_t* s_tri, int flag, int k) {
  return ((const signed char*)s_tri)[flag * 16 + k];
}

__device__ __forceinline__ void edge_geom(int e, int& dx, int& dy, int& dz, int& axis) {
  edge_parts(e, dx, dy, dz, axis);
}

__device__ __forceinline__ double sq3(double e0, double e1, double e2) {
#pragma clang fp contract(off)
  return e0 * e0 + e1 * e1 + e2 * e2;
}

struct McState {
  int64_t cap_flags = 0, cap_toff = 0;
  int64_t cap_v = 0, cap_tp = 0, cap_keep = 0, cap_t = 0;
  uint8_t* flags = nullptr;
  // linear mesher: bit words of 64 points each (kMcArrays arrays of one
  // length), vertex ranks per 8 points, kept triangles of the cells that lost
  // some, first triangle per word, counts per group of 16384 points
  uint64_t* words = nullptr;
  uint2* ranks = nullptr;
  uint8_t* kmask = nullptr;
  uint32_t* tword = nullptr;
  uint32_t* groups = nullptr;
  int64_t cap_words = 0, cap_ranks = 0, cap_kmask = 0, cap_tword = 0, cap_groups = 0;
  uint32_t* tri_off = nullptr; // per active cell triangle count -> offset
  double* verts = nullptr;
  int32_t* tris_pre = nullptr;
  uint32_t* keep = nullptr;    // per pre-filter triangle keep -> offset
  int32_t* tris = nullptr;
  void* tmp = nullptr;
  size_t tmp_bytes = 0;
  uint32_t* totals = nullptr;  // [0] active [1] vertices [2] triangles pre-filter [3] triangles
  int64_t nv = 0, nt = 0;
  // non-linear mesher: two slabs of field values (chunk i's in slab[i % 2]; the
  // next chunk's is evaluated on stream s2 while this one is meshed), slice
  // offsets, error counter
  double* slab[2] = {nullptr, nullptr};
  int64_t cap_slab[2] = {0, 0};
  hipStream_t s2 = nullptr;
  hipEvent_t ev_start = nullptr, ev_field[2] = {nullptr, nullptr}, ev_free[2] = {nullptr, nullptr};
  uint32_t *aword = nullptr, *lost = nullptr;  // per word: active cells before it in its group; dropped triangles
  int64_t cap_aword = 0, cap_lost = 0;
  uint32_t* vpt = nullptr;  // vertices of a range of points: owning point, edge axis
  uint8_t* vax = nullptr;
  int64_t cap_vpt = 0, cap_vax = 0;
  unsigned int* d_bad = nullptr;
  // edge cache of the last non-linear mesh (TRIANGLE_MESH.cpp:431-586): per
  // vertex its edge (lower endpoint x, y, z, axis), per active cell (x, y, z, flag)
  int32_t* c_edges = nullptr;
  int32_t* c_cells = nullptr;
  int64_t cap_ce = 0, cap_cc = 0, ncells = 0;
  bool cache_valid = false;
  // linear mesher over several fields: the vertices and triangles before each
  uint64_t* d_base = nullptr;
  int64_t cap_base = 0;
  uint32_t* tickets = nullptr;  // blocks that have finished (see finish_scan)
};

// grid coordinates of a point index (the mesher runs on fields of < 2^32 points)
__device__ __forceinline__ void point_xyz(const GridGeom& g, int64_t p, int64_t& x, int64_t& y, int64_t& z) {
  const uint32_t pu = (uint32_t)p;
  const uint32_t zu = fast_div(pu, g.div_xy);
  const uint32_t r = pu - zu * (uint32_t)g.res[0] * (uint32_t)g.res[1];
  const uint32_t yu = fast_div(r, g.div_x);
  z = zu;
  y = yu;
  x = r - yu * (uint32_t)g.res[0];
}

// Workgroups go to the 8 XCDs round-robin (block b to XCD b % 8); the point
// kernels deal each XCD a contiguous run of point blocks instead, so the
// field rows a block shares with its neighbours are fetched into one L2.
__device__ __forceinline__ int64_t xcd_block(int64_t nb) {
  const int64_t b = blockIdx.x, x = b & 7, k = b >> 3, per = nb >> 3, rem = nb & 7;
  return x * per + (x < rem ? x : rem) + k;
}

// One vertex of computeEdgeInterpolations (TRIANGLE_MESH.cpp:2373-2425): the
// edge from point (x, y, z) along `axis`, p0 + d0/(d0-d1) (p1-p0) between the
// two cell centres, in the reference's operation order with no contraction.
// k_mc_vertices writes it; k_mc_cells measures triangles with it, so both
// see the same bits.
__device__ __forceinline__ void mc_vertex(const GridGeom& g, int x, int y, int z, int axis, double f0, double f1,
                                          double iso, double* v) {
#pragma clang fp contract(off)
  double a[3], b[3];
  cell_center(g, x, y, z, a);
  cell_center(g, x + (axis == 0), y + (axis == 1), z + (axis == 2), b);
  const double d0 = f0 - iso;
  const double off0 = b[0] - a[0], off1 = b[1] - a[1], off2 = b[2] - a[2];
  const double d1 = f1 - iso;
  const double interpolation = d0 / (d0 - d1);
  v[0] = a[0] + interpolation * off0;
  v[1] = a[1] + interpolation * off1;
  v[2] = a[2] + interpolation * off2;
}

__device__ __forceinline__ double edge_len(const double* a, const double* b) {
#pragma clang fp contract(off)
  const double e0 = a[0] - b[0], e1 = a[1] - b[1], e2 = a[2] - b[2];
  return sqrt(e0 * e0 + e1 * e1 + e2 * e2);  // norm(v0 - v1), VEC3.h:215-216
}

// The degenerate filter (TRIANGLE_MESH.cpp:1088-1102) drops triangles with a
// side shorter than 1e-7. Two vertices of one triangle lie on edges of one
// cell: parallel or skew edges are at least one grid spacing h apart, and on
// two edges meeting at a corner c the vertices satisfy |v1 - v2| >=
// max |vi - c| (the edges are perpendicular). So with h >= kPrefilterSpacing
// a triangle with at most one vertex within 2e-7 of an end of its edge has
// every side longer than 1e-7. k_mc_vertices marks a vertex "near" from an FP32
// estimate t' of its place t on the edge: near unless t' h > kNearLimit and
// (1 - t') h > kNearLimit. |t' - t| stays below 2.5e-7 (corner values
// rounded to float, one subtraction and the products), so with
// h <= kPrefilterMaxSpacing every vertex within 2e-7 of an end is marked
// (2e-7 + 2.5e-7 h < 1e-6); NaN or infinite corners mark it too. Triangles
// with two or three marked vertices are measured with the FP64 vertices.
constexpr float kNearLimit = 1e-6f;
constexpr double kPrefilterSpacing = 1e-6;
constexpr double kPrefilterMaxSpacing = 3.0;
// On two edges that meet at a corner the vertices are sqrt(d0^2 + d1^2) apart
// for distances d0, d1 from it. FP32 estimates of those (relative error below
// 1e-6) decide all but a band of 1 % around 1e-7, as long as rounding of the
// FP64 coordinates (1e-11 up to kSureExtent) stays far inside the band; the rest is
// measured. kMeasureNear: coordinates beyond that. kMeasureAll: no prefilter.
constexpr float kSureShort = 0.99e-7f * 0.99e-7f, kSureLong = 1.01e-7f * 1.01e-7f;
constexpr double kSureExtent = 1e4;
constexpr double kSureSpacing = 1e-4;
enum McPrefilter { kMeasureAll = 0, kMeasureNear = 1, kMeasureUnsure = 2 };

// Whether the vertex of an edge with end values v0, v1 and grid spacing h may
// lie within 2e-7 of an end: near unless |v0| h > 1e-6 |v0 - v1| and
// |v1| h > 1e-6 |v0 - v1| (a vertex at place t has t = |v0| / |v0 - v1| and
// 1 - t = |v1| / |v0 - v1|, so no division); NaN and infinite ends make it near.
// Strictly greater: between subnormal ends the right side can round to 0, and
// an end of 0 is near then too (products rounded to n and n + 1 units of the
// smallest float differ by their true values' order, so none is passed over).
__device__ __forceinline__ bool mc_near(float v0, float v1, float h) {
  const float lim = kNearLimit * fabsf(v0 - v1);
  return !(fabsf(v0) * h > lim && fabsf(v1) * h > lim);
}

// The 12-bit mask of a cell's near edges from its float corner values (corner
// k = 4 dx + 2 dy + dz). prefilter = 0: all 12.
__device__ __forceinline__ unsigned mc_near_edges(const float* v, const GridGeom& g, int prefilter) {
  if (!prefilter) return 0xfffu;
  unsigned near = 0;
#pragma unroll
  for (int e = 0; e < 12; e++) {
    int dx = 0, dy = 0, dz = 0, axis = 0;
    edge_parts(e, dx, dy, dz, axis);
    const int k0 = 4 * dx + 2 * dy + dz, k1 = k0 + (axis == 0 ? 4 : (axis == 1 ? 2 : 1));
    near |= mc_near(v[k0], v[k1], fabsf((float)g.dx[axis])) ? (1u << e) : 0u;
  }
  return near;
}

// The 8 corner values of the cell at point p as floats (CUBE corners are
// floats, TRIANGLE_MESH.h:283-288; sign test at TRIANGLE_MESH.cpp:1037-1039),
// and its case.
__device__ __forceinline__ int mc_corners(const double* __restrict__ field, int64_t p, int64_t X, int64_t XY,
                                          double iso, float* v) {
  int flag = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int dx = k >> 2, dy = (k >> 1) & 1, dz = k & 1;
    v[k] = (float)(field[p + dx + dy * X + dz * XY] - iso);
    flag |= (v[k] > 0.0f) << k;
  }
  return flag;
}

// ---- linear mesher: one bit per grid point, 64 points (one word) at a time

constexpr int kMcWaves = kMcBlock / 64;        // waves per workgroup
constexpr int kMcGroupWords = kMcBlock;        // words per group: the unit of the two scans, one word per thread
constexpr int kMcGroupPoints = 64 * kMcGroupWords;
constexpr int kSignPoints = 8;                 // points per thread of k_mc_signs
constexpr int kTriBlocks = 2;                  // blocks of 256 cells per wave of k_mc_tris, at most
constexpr int kTriWaves = 256 * 16;            // waves that fill the chip before one takes a second block
constexpr int kListWords = 4;                  // words per wave of k_nl_vlist
constexpr int kScanBlock = 1024;

// Words whose bit i is point (or cell with lowest corner) 64 w + i; each array
// is wmax words long: those of the field's points, then at least
// mc_pad_words(g) that reads of a word's shifted rows may reach. Their bits
// and those of points past the last one are read but masked.
struct McGrid {
  GridGeom g;
  double iso;
  int prefilter;
  int64_t N, XY, nw;  // points, points per slice, words
  int64_t cells;      // cells with a lowest corner below this
  int64_t owned;      // edges of points below this
  bool floor;         // slice 0 is the grid's (not a slab's inside it)
  uint64_t* sgn;      // field value above the isovalue
  uint64_t* edge[3];  // the point's +x, +y, +z edge carries a vertex
  uint64_t* near[3];  // ... that may lie near an end of the edge
  uint64_t* drop;     // some of the cell's triangles were dropped: kmask holds the kept ones
};
constexpr int kMcArrays = 8;

static int64_t mc_pad_words(const GridGeom& g) {
  return ((int64_t)g.res[0] * g.res[1] + g.res[0] + 1) / 64 + 16;
}

static McGrid make_mc_grid(const McState& m, const GridGeom& g, int64_t wmax, double iso, int prefilter) {
  McGrid a;
  a.g = g;
  a.iso = iso;
  a.prefilter = prefilter;
  a.XY = (int64_t)g.res[0] * g.res[1];
  a.N = a.XY * g.res[2];
  a.nw = (a.N + 63) / 64;
  a.cells = a.N - a.XY;
  a.owned = a.N;
  a.floor = true;
  uint64_t* p[kMcArrays];
  for (int i = 0; i < kMcArrays; i++) p[i] = m.words + i * wmax;
  a.sgn = p[0];
  for (int i = 0; i < 3; i++) {
    a.edge[i] = p[1 + i];
    a.near[i] = p[4 + i];
  }
  a.drop = p[7];
  return a;
}

// A case row's triangles use exactly the edges whose corners differ in sign,
// except row 158, which leaves out kRow158Missing: the x edge at corner (0,0,0)
// and the y and z edges at (1,0,0). k_mc_edges builds on this.
constexpr int kRow158 = 158;
constexpr unsigned kRow158Missing = 1u << 0 | 1u << 5 | 1u << 9;
constexpr bool rows_use_crossing_edges() {
  for (int c = 0; c < 256; c++) {
    unsigned m = 0;
    for (int e = 0; e < 12; e++) {
      int dx = 0, dy = 0, dz = 0, axis = 0;
      edge_parts(e, dx, dy, dz, axis);
      const int k0 = 4 * dx + 2 * dy + dz, k1 = k0 + (axis == 0 ? 4 : (axis == 1 ? 2 : 1));
      if (((c >> k0) ^ (c >> k1)) & 1) m |= 1u << e;
    }
    if (kMcHost.emask[c] != (c == kRow158 ? m & ~kRow158Missing : m)) return false;
  }
  return true;
}
static_assert(rows_use_crossing_edges(), "the edges of the case rows");

// Bit B of the triangle count of 64 cells from the words of their corners (k =
// 4 dx + 2 dy + dz): the count's decision diagram over corners K-1..0 for the
// cases that agree with BASE above; equal halves need no test, and the compiler
// merges equal subtrees.
template <int B, int K, int BASE>
struct CountBits {
  static constexpr bool halves_equal() {
    for (int i = 0; i < (1 << (K - 1)); i++)
      if (((kMcHost.ntri[BASE + i] ^ kMcHost.ntri[BASE + (1 << (K - 1)) + i]) >> B) & 1) return false;
    return true;
  }
  static __device__ __forceinline__ uint64_t eval(const uint64_t* c) {
    const uint64_t lo = CountBits<B, K - 1, BASE>::eval(c);
    if constexpr (halves_equal()) {
      return lo;
    } else {
      const uint64_t hi = CountBits<B, K - 1, BASE + (1 << (K - 1))>::eval(c);
      return (c[K - 1] & hi) | (~c[K - 1] & lo);
    }
  }
};
template <int B, int BASE>
struct CountBits<B, 0, BASE> {
  static __device__ __forceinline__ uint64_t eval(const uint64_t*) {
    return (kMcHost.ntri[BASE] >> B) & 1 ? ~0ull : 0ull;
  }
};

// bits b.. of a word (b any integer)
__device__ __forceinline__ uint64_t bits_from(int64_t b) { return b <= 0 ? ~0ull : (b >= 64 ? 0ull : ~0ull << b); }

// word w of the array shifted down by `off` bits
__device__ __forceinline__ uint64_t shifted_word(const uint64_t* __restrict__ a, int64_t w, int64_t off) {
  const int64_t i = w + (off >> 6);
  const int sh = (int)(off & 63);
  const uint64_t lo = a[i], hi = a[i + 1];
  return (lo >> sh) | ((hi << 1) << (63 - sh));
}

// the points of word w that are last along x, along y, along z (or past the field's last)
struct EndMasks {
  uint64_t x, y, z;
};
__device__ __forceinline__ EndMasks end_masks(const McGrid& a, int64_t w) {
  EndMasks m{0, 0, bits_from(a.N - a.XY - 64 * w)};
  const int64_t X = a.g.res[0];
  const uint32_t p0 = (uint32_t)(64 * w);
  const uint32_t r0 = p0 - fast_div(p0, a.g.div_xy) * (uint32_t)a.XY;
  const uint32_t x0 = r0 - fast_div(r0, a.g.div_x) * (uint32_t)X;
  for (int64_t b = X - 1 - (int64_t)x0; b < 64; b += X) m.x |= 1ull << b;
  for (int64_t b = a.XY - X - (int64_t)r0; b < 64; b += a.XY) m.y |= bits_from(b) & ~bits_from(b + X);
  return m;
}

// inclusive prefix sum over the wave's lanes (DPP row shifts and broadcasts)
__device__ __forceinline__ uint32_t wave_inclusive(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
  return v;
}
__device__ __forceinline__ uint32_t wave_last(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }

// exclusive prefix over the block's threads; *total: the block's sum. Every thread of the block takes part.
template <int kThreads>
__device__ __forceinline__ uint32_t block_prefix(uint32_t v, uint32_t* total) {
  __shared__ uint32_t s_w[kThreads / 64];
  const uint32_t incl = wave_inclusive(v);
  if ((threadIdx.x & 63) == 63) s_w[threadIdx.x >> 6] = incl;
  __syncthreads();
  uint32_t before = 0, sum = 0;
  for (int i = 0; i < kThreads / 64; i++) {
    const uint32_t c = s_w[i];
    before += i < (int)(threadIdx.x >> 6) ? c : 0u;
    sum += c;
  }
  __syncthreads();
  *total = sum;
  return before + incl - v;
}

// this workgroup's wave number, workgroups in contiguous runs per XCD
__device__ __forceinline__ int64_t wave_index() {
  return (int64_t)__builtin_amdgcn_readfirstlane((int)(xcd_block(gridDim.x) * kMcWaves + (threadIdx.x >> 6)));
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The float sign test of every point (CUBE corners are floats,
// TRIANGLE_MESH.h:283-288; test at TRIANGLE_MESH.cpp:1037-1039). HBM-bound: one
// read of the field; a wave takes 512 consecutive points, eight loads in
// flight per lane. 256^3: 29.6 us, 4.5 TB/s (the 8 corners read per cell and a
// case byte written per cell, before: 109 us).
__global__ __launch_bounds__(kMcBlock) void k_mc_signs(const double* __restrict__ field, int64_t N, double iso,
                                                       uint64_t* __restrict__ sgn) {
  const int lane = threadIdx.x & 63;
  const int64_t p0 = ((int64_t)blockIdx.x * kMcWaves + (threadIdx.x >> 6)) * 64 * kSignPoints;
  if (p0 >= N) return;
  double v[kSignPoints];
#pragma unroll
  for (int i = 0; i < kSignPoints; i++) {
    const int64_t p = p0 + 64 * i + lane;
    v[i] = field[p < N ? p : N - 1];
  }
  uint64_t mine = 0;
#pragma unroll
  for (int i = 0; i < kSignPoints; i++) {
    const uint64_t word = __ballot((float)(v[i] - iso) > 0.0f);
    mine = lane == i ? word : mine;
  }
  if (lane < kSignPoints && p0 + 64 * lane < N) sgn[p0 / 64 + lane] = mine;
}

// The groups' counts to exclusive offsets in place, by one block, and the running
// total after this tile: base[2 tile + which] is what came before it; also in
// h_base (pinned memory). kAtomic: the counts come from other blocks of the same
// launch.
template <int kThreads, bool kAtomic>
__device__ __forceinline__ void scan_groups(uint32_t* __restrict__ groups, int64_t n, uint64_t* __restrict__ base,
                                            uint64_t* __restrict__ h_base, int tile, int which) {
  const auto count = [&](int64_t i) { return kAtomic ? atomicAdd(&groups[i], 0u) : groups[i]; };
  const int64_t per = (n + kThreads - 1) / kThreads, b = (int64_t)threadIdx.x * per;
  constexpr int kHeld = 4;  // counts in registers, so that up to 1024 groups are read once
  uint32_t held[kHeld], v = 0;
#pragma unroll
  for (int k = 0; k < kHeld; k++) held[k] = k < per && b + k < n ? count(b + k) : 0u;
#pragma unroll
  for (int k = 0; k < kHeld; k++) v += held[k];
  for (int64_t i = b + kHeld; i < b + per && i < n; i++) v += count(i);
  uint32_t total;
  uint32_t run = block_prefix<kThreads>(v, &total);
  for (int64_t i = b; i < b + per && i < n; i++) {
    uint32_t c = 0;
    if (i - b < kHeld) {
#pragma unroll
      for (int k = 0; k < kHeld; k++) c = i - b == k ? held[k] : c;
    } else {
      c = count(i);
    }
    groups[i] = run;
    run += c;
  }
  if (threadIdx.x == 0) {
    if (tile == 0) base[which] = 0;
    const uint64_t sum = (tile == 0 ? 0 : base[2 * tile + which]) + total;
    base[2 * (tile + 1) + which] = sum;
    if (h_base) h_base[2 * (tile + 1) + which] = sum;
  }
}

__global__ __launch_bounds__(kScanBlock) void k_mc_scan(uint32_t* __restrict__ groups, int64_t n,
                                                        uint64_t* __restrict__ base, uint64_t* __restrict__ h_base,
                                                        int tile, int which) {
  scan_groups<kScanBlock, false>(groups, n, base, h_base, tile, which);
}

// Where a kernel's last block to finish scans the counts, in place of a launch of
// its own: counts, tickets and the scan's reads are read-modify-writes, which all
// XCDs see in one order, and a ticket is drawn once the write before it has
// returned. Beyond 64 blocks the tickets are drawn from kTickets lines first: on
// one line they come back one in 7 ns (1024 blocks 9.8 us, 2 to 3 this way; the
// launch 4.7 and the gap before it 2 to 5). Tickets are left at 0. Beyond
// kFoldGroups a thread would read its counts one after another, twice, and the
// launch is the better one (base null).
constexpr int kTickets = 16, kTicketLine = 32, kFoldGroups = 4 * kMcBlock;
struct ScanTail {
  uint64_t *base, *h_base;
  uint32_t* tickets;  // kTickets + 1 lines
  int tile;
};
__device__ __forceinline__ bool draws_last(uint32_t* ticket, uint32_t after, uint32_t of) {
  uint32_t one = 1;
  asm volatile("" : "+v"(one) : "v"(after));  // not before `after` has come back
  if (atomicAdd(ticket, one) != of - 1) return false;
  atomicExch(ticket, 0u);
  return true;
}
__device__ __forceinline__ void finish_scan(uint32_t* __restrict__ groups, uint32_t total, const ScanTail& t,
                                            int which) {
  __shared__ int s_last;
  if (!t.base) {
    if (threadIdx.x == 0) groups[blockIdx.x] = total;
    return;
  }
  if (threadIdx.x == 0) {
    const uint32_t blocks = gridDim.x, before = atomicExch(&groups[blockIdx.x], total);
    if (blocks <= 64) {
      s_last = draws_last(t.tickets, before, blocks);
    } else {
      const uint32_t sub = blockIdx.x % kTickets, of = (blocks - sub + kTickets - 1) / kTickets;
      s_last = draws_last(t.tickets + (1 + sub) * kTicketLine, before, of) && draws_last(t.tickets, of, kTickets);
    }
  }
  __syncthreads();
  if (!s_last) return;
  scan_groups<kMcBlock, true>(groups, gridDim.x, t.base, t.h_base, t.tile, which);
}

// every third bit of 24 from 8
__device__ __forceinline__ uint32_t spread8(uint32_t x) {
  x = (x | x << 8) & 0x00f00fu;
  x = (x | x << 4) & 0x0c30c3u;
  return (x | x << 2) & 0x249249u;
}

// The edges that carry a vertex, one word of points per thread: those with
// ends of different sign, except where the only cells around an edge are of
// case 158 and leave it out (on three border lines of the grid). ranks[8 w + j]
// serves the triangle kernel's lookups: for points 64 w + 8 j.. the vertices
// before them in the group and the 24 edge bits in id order (point, then axis),
// so that a vertex's id is one masked bit count away. groups[]: vertices per
// group. Latency-bound: 256^3, 1024 blocks, 13 us with the scan (from the case
// bytes of the 12 cells around a point: 54 us and 14 of scans).
__global__ __launch_bounds__(kMcBlock) void k_mc_edges(McGrid a, uint2* __restrict__ ranks,
                                                       uint32_t* __restrict__ groups, ScanTail tail) {
  const int64_t w = (int64_t)blockIdx.x * kMcGroupWords + threadIdx.x;
  const int64_t X = a.g.res[0];
  uint64_t e[3] = {0, 0, 0};
  if (w < a.nw) {
    const uint64_t s0 = a.sgn[w];
    const EndMasks end = end_masks(a, w);
    const uint64_t in = ~bits_from(a.owned - 64 * w);
    e[0] = (s0 ^ shifted_word(a.sgn, w, 1)) & ~end.x & in;
    e[1] = (s0 ^ shifted_word(a.sgn, w, X)) & ~end.y & in;
    e[2] = (s0 ^ shifted_word(a.sgn, w, a.XY)) & ~end.z & in;
    const uint64_t z0 = a.floor ? ~bits_from(a.XY - 64 * w) : 0;  // z = 0
    const uint32_t p0 = (uint32_t)(64 * w);
    uint64_t y0 = 0;  // y = 0
    for (int64_t b = (int64_t)fast_div(p0, a.g.div_xy) * a.XY - (int64_t)p0; b < 64; b += a.XY)
      y0 |= bits_from(b) & ~bits_from(b + X);
    const uint64_t line[3] = {y0 & z0, z0 & end.x, y0 & end.x};
#pragma unroll
    for (int axis = 0; axis < 3; axis++)
      for (uint64_t m = e[axis] & line[axis]; m; m &= m - 1) {
        const int b = __ffsll((unsigned long long)m) - 1;
        const int64_t c = 64 * w + b - (axis ? 1 : 0);  // the cell that may leave the edge out, alone around it
        int flag = 0;
        for (int k = 0; k < 8; k++) {
          const int64_t q = c + (k >> 2) + ((k >> 1) & 1) * X + (k & 1) * a.XY;
          flag |= (int)((a.sgn[q >> 6] >> (q & 63)) & 1u) << k;
        }
        if (flag == kRow158) e[axis] &= ~(1ull << b);
      }
    for (int axis = 0; axis < 3; axis++) a.edge[axis][w] = e[axis];
  }
  uint32_t total;
  uint32_t run = block_prefix<kMcBlock>((uint32_t)(__popcll(e[0]) + __popcll(e[1]) + __popcll(e[2])), &total);
#pragma unroll
  for (int j = 0; j < 8; j++) {
    if (w >= a.nw) break;
    const uint32_t bits = spread8((uint32_t)(e[0] >> (8 * j)) & 0xffu) | spread8((uint32_t)(e[1] >> (8 * j)) & 0xffu) << 1 |
                          spread8((uint32_t)(e[2] >> (8 * j)) & 0xffu) << 2;
    ranks[8 * w + j] = uint2{run, bits};
    run += (uint32_t)__popc(bits);
  }
  finish_scan(groups, total, tail, 0);
}

// computeEdgeInterpolations (TRIANGLE_MESH.cpp:2373-2425). A wave lists the
// vertices of its 512 points (at most 3 per point) in LDS in id order and
// computes them one per lane, so that the FP64 work is not spread over mostly
// idle lanes; the tile's vertices go to verts from base[0] on (several tiles
// share the buffer). Ids at or beyond cap are not written (the host sees the
// overflow in the totals). Also marks the vertices near an end of their edge.
// Bound by the field's second read and the vertices' writes: a 256^3 torus tile
// (4.5 million vertices, 109 MB) 69 us, 3.5 TB/s; neither two vertices per lane
// in flight, nor stores made contiguous through LDS, nor leaving out the rotation
// made it faster. Below 32 waves per CU a wave takes two words instead of eight
// (97 x 101 x 89: 7.2 us, with eight 10.3).
template <int kVertWords>
__global__ __launch_bounds__(kMcBlock) void k_mc_vertices(const double* __restrict__ field, McGrid a,
                                                          const uint2* __restrict__ ranks,
                                                          const uint32_t* __restrict__ groups,
                                                          const uint64_t* __restrict__ base, int64_t cap,
                                                          double* __restrict__ verts) {
  __shared__ uint16_t s_v[kMcWaves][3 * 64 * kVertWords];
  __shared__ uint32_t s_near[kMcWaves][3][2 * kVertWords];
  const int64_t X = a.g.res[0], w0 = wave_index() * kVertWords;
  if (w0 >= a.nw) return;
  const int lane = threadIdx.x & 63;
  uint16_t* const list = s_v[threadIdx.x >> 6];
  uint32_t(*near)[2 * kVertWords] = s_near[threadIdx.x >> 6];
  if (lane < 3 * 2 * kVertWords) (&near[0][0])[lane] = 0u;
  const uint64_t *const ex = a.edge[0], *const ey = a.edge[1], *const ez = a.edge[2];
  uint32_t total = 0;
#pragma unroll
  for (int i = 0; i < kVertWords; i++) {
    uint64_t e[3] = {0, 0, 0};
    if (w0 + i < a.nw) {
      e[0] = ex[w0 + i];
      e[1] = ey[w0 + i];
      e[2] = ez[w0 + i];
    }
    uint32_t k = total;
#pragma unroll
    for (int axis = 0; axis < 3; axis++)
      k = __builtin_amdgcn_mbcnt_hi((uint32_t)(e[axis] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)e[axis], k));
#pragma unroll
    for (int axis = 0; axis < 3; axis++)
      if (__builtin_amdgcn_inverse_ballot_w64(e[axis])) list[k++] = (uint16_t)(i * 64 + lane | axis << 10);
    total += (uint32_t)(__popcll(e[0]) + __popcll(e[1]) + __popcll(e[2]));
  }
  wave_sync();
  if (total) {
    const int64_t first = (int64_t)(base[0] + groups[w0 / kMcGroupWords] + ranks[8 * w0].x);
    for (uint32_t j = lane; j < total; j += 64) {
      const unsigned en = list[j];
      const int axis = (int)(en >> 10), pt = (int)(en & 1023u);
      const int64_t q = 64 * w0 + pt;
      int64_t x, y, z;
      point_xyz(a.g, q, x, y, z);
      const double f0 = field[q], f1 = field[q + (axis == 0 ? 1 : (axis == 1 ? X : a.XY))];
      const float h = fabsf((float)(axis == 0 ? a.g.dx[0] : (axis == 1 ? a.g.dx[1] : a.g.dx[2])));
      if (!a.prefilter || mc_near((float)(f0 - a.iso), (float)(f1 - a.iso), h))
        atomicOr(&near[axis][pt >> 5], 1u << (pt & 31));
      double v[3];
      mc_vertex(a.g, (int)x, (int)y, (int)z, axis, f0, f1, a.iso, v);
      const int64_t id = first + j;
      if (id < cap) {
        verts[3 * id + 0] = v[0];
        verts[3 * id + 1] = v[1];
        verts[3 * id + 2] = v[2];
      }
    }
  }
  wave_sync();
  const int i = lane & (kVertWords - 1), axis = lane / kVertWords;
  if (axis < 3 && w0 + i < a.nw)
    (axis == 0 ? a.near[0] : (axis == 1 ? a.near[1] : a.near[2]))[w0 + i] =
        (uint64_t)near[axis][2 * i + 1] << 32 | near[axis][2 * i];
}

// The degenerate filter (TRIANGLE_MESH.cpp:1088-1102) for one cell with two or
// more near vertices: its triangles with two or three are measured with the
// FP64 vertices (the function the vertex kernel uses, so both see the same
// bits). Only a side between two near vertices can be short: a vertex that is
// not near is at least 2e-7 from both ends of its edge, so at least that far
// from a vertex on an edge through either end, and a grid spacing from vertices
// on the other edges. Estimates come first (kSureShort): a border of one value
// puts every vertex along it near, 1e-9 to 1e-6 from its corner. Returns the
// dropped triangles' bits; *row: all of the row's.
__device__ __forceinline__ unsigned mc_measure_cell(const double* __restrict__ field, const McGrid& a, int64_t p,
                                                    unsigned* row) {
  const int64_t X = a.g.res[0], XY = a.XY;
  int64_t x, y, z;
  point_xyz(a.g, p, x, y, z);
  float v[8];
  const int flag = mc_corners(field, p, X, XY, a.iso, v);
  const int n = kMc.ntri[flag];
  // per corner and pair of its edges (xy, xz, yz), bit 3 k + pair: surely short; not surely long
  unsigned brief = 0, unsure = 0xffffffu;
  if (a.prefilter == kMeasureUnsure) {
    unsure = 0;
    float d2[8][3];  // per corner and axis: the squared distance of the edge's vertex
#pragma unroll
    for (int e = 0; e < 12; e++) {
      int dx = 0, dy = 0, dz = 0, axis = 0;
      edge_parts(e, dx, dy, dz, axis);
      const int k0 = 4 * dx + 2 * dy + dz, k1 = k0 + (axis == 0 ? 4 : (axis == 1 ? 2 : 1));
      const float d = fabsf(v[k0] - v[k1]);
      const float scale = d >= 1e-30f && d <= 1e30f ? fabsf((float)a.g.dx[axis]) * __builtin_amdgcn_rcpf(d)
                                                    : __builtin_nanf("");
      d2[k0][axis] = (v[k0] * scale) * (v[k0] * scale);
      d2[k1][axis] = (v[k1] * scale) * (v[k1] * scale);
    }
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const float d = d2[k][q == 2 ? 1 : 0] + d2[k][q == 0 ? 1 : 2];
        brief |= d < kSureShort ? 1u << (3 * k + q) : 0u;
        unsure |= d > kSureLong ? 0u : 1u << (3 * k + q);
      }
  }
  *row = (1u << n) - 1u;
  unsigned dropped = 0, measure = *row;
  if (a.prefilter) {
    measure = 0;
#pragma unroll
    for (int t = 0; t < 5; t++) {
      const unsigned pairs = kMc.tpair[flag][t];  // none beyond the row's triangles
      dropped |= pairs & brief ? 1u << t : 0u;
      measure |= !(pairs & brief) && (pairs & unsure) ? 1u << t : 0u;
    }
  }
  const unsigned near = measure ? mc_near_edges(v, a.g, a.prefilter) : 0u;
  while (measure) {
    const int t = __ffs(measure) - 1;
    measure &= measure - 1;
    const unsigned nm = near & kMc.tmask[flag][t];
    const int m = __popc(nm);
    if (m < 2) continue;
    double w[3][3] = {};
    unsigned r = nm;
#pragma unroll
    for (int j = 0; j < 3; j++) {
      if (j < m) {  // constant indices into w keep it in registers
        const int e = __ffs(r) - 1;
        r &= r - 1;
        int dx, dy, dz, axis;
        edge_geom(e, dx, dy, dz, axis);
        const int64_t q0 = p + dx + dy * X + dz * XY;
        const int64_t q1 = q0 + (axis == 0 ? 1 : (axis == 1 ? X : XY));
        mc_vertex(a.g, (int)x + dx, (int)y + dy, (int)z + dz, axis, field[q0], field[q1], a.iso, w[j]);
      }
    }
    const double eps = 1e-7;
    bool degenerate = edge_len(w[0], w[1]) < eps;
    if (m == 3) degenerate = degenerate || edge_len(w[0], w[2]) < eps || edge_len(w[1], w[2]) < eps;
    if (degenerate) dropped |= 1u << t;
  }
  return dropped;
}

// The cases of 8 cells from bit b on, one byte each: byte k of m holds corner
// k's bits, transposed in three exchanges of blocks.
__device__ __forceinline__ uint64_t cases8(const uint64_t* c, int b) {
  uint64_t m = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) m |= ((c[k] >> b) & 0xffull) << (8 * k);
  uint64_t t = (m ^ (m >> 7)) & 0x00aa00aa00aa00aaull;
  m ^= t ^ (t << 7);
  t = (m ^ (m >> 14)) & 0x0000cccc0000ccccull;
  m ^= t ^ (t << 14);
  t = (m ^ (m >> 28)) & 0x00000000f0f0f0f0ull;
  return m ^ t ^ (t << 28);
}

// Word w's cells: *count triangles, the cases of those that have any (else 0)
// to flags; returns those cells' bits.
__device__ __forceinline__ uint64_t word_cases(const McGrid& a, int64_t w, uint8_t* __restrict__ flags,
                                               uint32_t* count) {
  const EndMasks end = end_masks(a, w);
  const uint64_t valid = ~(end.x | end.y | end.z | bits_from(a.cells - 64 * w));
  uint64_t c[8];
#pragma unroll
  for (int k = 0; k < 8; k++)
    c[k] = shifted_word(a.sgn, w, (k >> 2) + ((k >> 1) & 1) * (int64_t)a.g.res[0] + (k & 1) * a.XY);
  const uint64_t n0 = CountBits<0, 8, 0>::eval(c) & valid, n1 = CountBits<1, 8, 0>::eval(c) & valid,
                 n2 = CountBits<2, 8, 0>::eval(c) & valid, act = n0 | n1 | n2;
#pragma unroll
  for (int k = 0; k < 8; k++) c[k] &= act;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint64_t f0 = cases8(c, 16 * j), f1 = cases8(c, 16 * j + 8);
    ((uint4*)flags)[4 * w + j] = uint4{(uint32_t)f0, (uint32_t)(f0 >> 32), (uint32_t)f1, (uint32_t)(f1 >> 32)};
  }
  *count = (uint32_t)(__popcll(n0) + 2 * __popcll(n1) + 4 * __popcll(n2));
  return act;
}

// The cells of word w that may hold a triangle with two near vertices on edges that
// meet at a corner, among those of act (a border set by setBorders puts near
// vertices in every cell along it, but on parallel edges).
__device__ __forceinline__ uint64_t meeting_near_edges(const McGrid& a, int64_t w, uint64_t act) {
  const int64_t X = a.g.res[0], XY = a.XY;
  uint64_t near[12], cells = 0;
#pragma unroll
  for (int e = 0; e < 12; e++) {
    int dx = 0, dy = 0, dz = 0, axis = 0;
    edge_parts(e, dx, dy, dz, axis);
    near[e] = shifted_word(a.near[axis], w, dx + dy * X + dz * XY);
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int dx = k >> 2, dy = (k >> 1) & 1, dz = k & 1;
    const uint64_t nx = near[dy + 2 * dz], ny = near[4 + dx + 2 * dz], nz = near[8 + dx + 2 * dy];
    cells |= (nx & (ny | nz)) | (ny & nz);
  }
  return cells & act;
}

// The degenerate filter where estimates do not decide it (kMeasureAll,
// kMeasureNear): the first wave finds the candidates of `words` words, one per
// thread, and lists them in LDS, where all four take them one per thread. drop: the
// cells that lost triangles, kmask what they keep, lost the triangles lost per
// word. k_mc_cells does the same for its groups of 16384 cells; where those are fewer
// than the CUs and noise or values of 0 and 1 make every second cell a candidate,
// its blocks take 400 us one after another, and this kernel's spread over the chip.
// FP64 VALU bound. Times beside measure_words.
constexpr int kMeasureWords = 64;
__global__ __launch_bounds__(kMcBlock) void k_mc_measure(const double* __restrict__ field, McGrid a, int words,
                                                         uint8_t* __restrict__ kmask, uint32_t* __restrict__ lost) {
  __shared__ uint16_t s_list[64 * kMeasureWords];
  __shared__ uint32_t s_drop[2 * kMeasureWords], s_lost[kMeasureWords], s_cells;
  const int tid = threadIdx.x;
  const int64_t w0 = xcd_block(gridDim.x) * words, w = w0 + tid;
  const bool own = tid < words && w < a.nw;
  if (tid < kMeasureWords) {
    uint64_t cells = 0;
    if (own) {
      const EndMasks end = end_masks(a, w);
      uint64_t any = 0, all = ~0ull;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint64_t c = shifted_word(a.sgn, w, (k >> 2) + ((k >> 1) & 1) * (int64_t)a.g.res[0] + (k & 1) * a.XY);
        any |= c;
        all &= c;
      }
      cells = any & ~all & ~(end.x | end.y | end.z | bits_from(a.cells - 64 * w));
      if (cells && a.prefilter) cells = meeting_near_edges(a, w, cells);
    }
    s_drop[2 * tid] = s_drop[2 * tid + 1] = 0u;
    s_lost[tid] = 0u;
    const uint32_t mine = (uint32_t)__popcll(cells), incl = wave_inclusive(mine);
    uint32_t k = incl - mine;
    for (uint64_t m = cells; m; m &= m - 1)
      s_list[k++] = (uint16_t)(tid << 6 | (__ffsll((unsigned long long)m) - 1));
    if (tid == 63) s_cells = incl;
  }
  __syncthreads();
  for (uint32_t j = tid; j < s_cells; j += kMcBlock) {
    const unsigned i = s_list[j];
    const int64_t p = 64 * w0 + i;
    unsigned row;
    const unsigned d = mc_measure_cell(field, a, p, &row);
    if (d) {
      kmask[p] = (uint8_t)(row & ~d);
      atomicOr(&s_drop[i >> 5], 1u << (i & 31u));
      atomicAdd(&s_lost[i >> 6], (uint32_t)__popc(d));
    }
  }
  __syncthreads();
  if (own) {
    a.drop[w] = (uint64_t)s_drop[2 * tid + 1] << 32 | s_drop[2 * tid];
    lost[w] = s_lost[tid];
  }
}

// Triangle counts, one word of cells per thread: the counts' three bits as
// word operations on the corners' words. The degenerate filter measures the
// cells with near vertices on two edges that meet at a corner, found the same
// way, listed in LDS and measured one per thread, unless lost says what
// k_mc_measure dropped.
// flags: the case of every cell that has
// triangles, else 0. Latency-bound: 256^3, 1024 blocks, 19.2 us with the
// scan, of which the measurement's longest chain is 6 (20 with every near pair
// measured). tword: the triangles before word w in its group; groups:
// per group.
__global__ __launch_bounds__(kMcBlock) void k_mc_cells(const double* __restrict__ field, McGrid a,
                                                       uint8_t* __restrict__ flags, uint8_t* __restrict__ kmask,
                                                       const uint32_t* __restrict__ lost,
                                                       uint32_t* __restrict__ tword,
                                                       uint32_t* __restrict__ groups, ScanTail tail) {
  __shared__ uint16_t s_list[kMcWaves][64 * 64];
  __shared__ uint32_t s_drop[2 * kMcGroupWords], s_lost[kMcGroupWords], s_cells[kMcWaves];
  const int64_t w = (int64_t)blockIdx.x * kMcGroupWords + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t candidates = 0;
  uint32_t count = 0;
  if (w < a.nw) {
    const uint64_t act = word_cases(a, w, flags, &count);
    if (lost) count -= lost[w];
    else if (act) candidates = a.prefilter ? meeting_near_edges(a, w, act) : act;
  }
  s_drop[2 * threadIdx.x] = s_drop[2 * threadIdx.x + 1] = 0u;
  s_lost[threadIdx.x] = 0u;
  const uint32_t mine = (uint32_t)__popcll(candidates), incl = wave_inclusive(mine);
  uint32_t k = incl - mine;
  for (uint64_t m = candidates; m; m &= m - 1)
    s_list[wave][k++] = (uint16_t)(lane << 6 | (__ffsll((unsigned long long)m) - 1));
  if (lane == 63) s_cells[wave] = incl;
  __syncthreads();
  // the four waves' lists one after another, over all threads
  uint32_t from[kMcWaves + 1] = {0};
#pragma unroll
  for (int i = 0; i < kMcWaves; i++) from[i + 1] = from[i] + s_cells[i];
  for (uint32_t j = threadIdx.x; j < from[kMcWaves]; j += kMcBlock) {
    int v = 0;
#pragma unroll
    for (int i = 1; i < kMcWaves; i++) v += j >= from[i] ? 1 : 0;
    const unsigned i = (unsigned)v << 12 | s_list[v][j - (v == 0 ? 0 : v == 1 ? from[1] : v == 2 ? from[2] : from[3])];
    const int64_t p = (int64_t)blockIdx.x * kMcGroupPoints + i;
    unsigned row;
    const unsigned d = mc_measure_cell(field, a, p, &row);
    if (d) {
      kmask[p] = (uint8_t)(row & ~d);
      atomicOr(&s_drop[i >> 5], 1u << (i & 31u));
      atomicAdd(&s_lost[i >> 6], (uint32_t)__popc(d));
    }
  }
  __syncthreads();
  count -= s_lost[threadIdx.x];
  uint32_t total;
  const uint32_t before = block_prefix<kMcBlock>(count, &total);
  if (w < a.nw) {
    if (!lost) a.drop[w] = (uint64_t)s_drop[2 * threadIdx.x + 1] << 32 | s_drop[2 * threadIdx.x];
    tword[w] = before;
  }
  finish_scan(groups, total, tail, 1);
}

// addVertexPairTriangle (TRIANGLE_MESH.cpp:2490-2503) in cell order then table
// order. A wave takes blocks of 256 cells, four consecutive ones per lane: it
// lists a block's kept triangles (5 case + triangle of the row; cell) in LDS and
// writes them one per lane, so that consecutive lanes write consecutive
// triangles. The owner of an edge of cell p is p + dx + dy X + dz XY: four rows
// of points, whose ranks are staged in LDS with the groups' offsets added, so
// that a corner's vertex id is one LDS read and a masked bit count; ids count
// from id0, triangles from base[1] (null: 0). Triangles at or beyond tcap are not
// written. Bound by LDS latency at 7 waves per SIMD: a 256^3 torus tile (9.1
// million triangles, 109 MB) 54 us; 64 with 32-bit list entries (5 waves), 76 with a
// 16-bit rank per point and case and kept bytes of every cell. `blocks` per wave:
// the tables' staging is shared by up to kTriBlocks of them once the chip is full
// (one, two, four: 70, 62, 64 us with 32-bit entries, two and four 54 and 57 now;
// 97 x 101 x 89 with one 6.5, with four 20.7).
constexpr int kRankRow = 34;  // 8-point ranks per row: 257 points from any phase
__global__ __launch_bounds__(kMcBlock) void k_mc_tris(McGrid a, int blocks, const uint8_t* __restrict__ flags,
                                                      const uint64_t* __restrict__ drop,
                                                      const uint8_t* __restrict__ kmask,
                                                      const uint2* __restrict__ ranks,
                                                      const uint32_t* __restrict__ vgroups,
                                                      const uint32_t* __restrict__ tword,
                                                      const uint32_t* __restrict__ tgroups,
                                                      const uint64_t* __restrict__ base, uint32_t id0, int64_t tcap,
                                                      int32_t* __restrict__ tris) {
  __shared__ uint32_t s_te32[256 * 5 / 2];
  __shared__ uint8_t s_n[256];
  __shared__ uint32_t s_edge[12];
  __shared__ uint16_t s_row[kMcWaves][5 * 256];
  __shared__ uint8_t s_cell[kMcWaves][5 * 256];
  __shared__ uint2 s_rank[kMcWaves][4 * kRankRow];
  const unsigned short* s_te = (const unsigned short*)s_te32;
  const int64_t X = a.g.res[0], XY = a.XY;
  for (int i = threadIdx.x; i < 640; i += kMcBlock) s_te32[i] = ((const uint32_t*)&kMc.tedge[0][0])[i];
  s_n[threadIdx.x] = kMc.ntri[threadIdx.x];
  if (threadIdx.x < 12) {
    // per edge: its owner's place from the cell's in the staged rows << 2 | axis
    int dx, dy, dz, axis;
    edge_geom((int)threadIdx.x, dx, dy, dz, axis);
    const int phase = (int)((dy * X + dz * XY) & 7);
    s_edge[threadIdx.x] = (uint32_t)((dx + phase + 8 * kRankRow * (dy + 2 * dz)) << 2 | axis);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint16_t* const list = s_row[wave];
  uint8_t* const cell = s_cell[wave];
  uint2* const rank = s_rank[wave];
  const int64_t last_group = (a.nw - 1) / kMcGroupWords;
  const int64_t B0 = wave_index() * blocks;
  // the next block's cases are fetched while this one is written; words past the field's last hold no cells
  uint32_t next = 4 * B0 + (lane >> 4) < a.nw ? ((const uint32_t*)flags)[64 * B0 + lane] : 0u;
  for (int it = 0; it < blocks; it++) {
    const int64_t w0 = 4 * (B0 + it);
    const bool in = w0 + (lane >> 4) < a.nw;
    const uint32_t f4 = next;
    if (it + 1 < blocks) next = w0 + 4 + (lane >> 4) < a.nw ? ((const uint32_t*)flags)[16 * (w0 + 4) + lane] : 0u;
    if (!__ballot(f4 != 0u)) continue;
    // the four rows' ranks
    uint2 rv[4];
    uint32_t gv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (lane >= kRankRow) continue;
      const int64_t q = 8 * w0 + (((r & 1) * X + (r >> 1) * XY) >> 3) + lane;
      const int64_t gr = q / (kMcGroupPoints / 8);
      rv[r] = ranks[q];
      gv[r] = vgroups[gr < last_group ? gr : last_group];
    }
    const uint64_t lost = in ? drop[w0 + (lane >> 4)] : 0;
    unsigned keep = 0, lost4 = (unsigned)(lost >> (4 * (lane & 15))) & 15u;  // keep: 5 bits per cell
    unsigned n[4];
#pragma unroll
    for (int i = 0; i < 4; i++) n[i] = s_n[(f4 >> (8 * i)) & 0xffu];
    const bool some_lost = __ballot(lost4 != 0u) != 0;
    if (some_lost) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        unsigned m = (1u << n[i]) - 1u;
        if (lost4 >> i & 1u) m = kmask[64 * w0 + 4 * lane + i];
        keep |= m << (5 * i);
        n[i] = (unsigned)__popc(m);
      }
    }
    const uint32_t mine = n[0] + n[1] + n[2] + n[3], incl = wave_inclusive(mine), total = wave_last(incl);
    uint32_t at = incl - mine;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t e0 = ((f4 >> (8 * i)) & 0xffu) * 5u, c = (uint32_t)(4 * lane + i);
      if (some_lost) {
        uint32_t k = at;
        for (unsigned m = keep >> (5 * i) & 31u; m; m &= m - 1) {
          cell[k] = (uint8_t)c;
          list[k++] = (uint16_t)(e0 + (uint32_t)(__ffs(m) - 1));
        }
      } else {
#pragma unroll
        for (uint32_t t = 0; t < 5; t++)
          if (t < n[i]) {
            list[at + t] = (uint16_t)(e0 + t);
            cell[at + t] = (uint8_t)c;
          }
      }
      at += n[i];
    }
    if (lane < kRankRow) {
#pragma unroll
      for (int r = 0; r < 4; r++) rank[kRankRow * r + lane] = uint2{rv[r].x + gv[r] + id0, rv[r].y};
    }
    wave_sync();
    const int64_t o = (int64_t)((base ? base[1] : 0) + tgroups[w0 / kMcGroupWords] + tword[w0]);
    for (uint32_t j = lane; j < total; j += 64) {
      const uint32_t te = s_te[list[j]], c = cell[j];
      int32_t id[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const uint32_t ed = s_edge[(te >> (4 * k)) & 15u], q = c + (ed >> 2);
        const uint2 rk = rank[q >> 3];
        id[k] = (int32_t)(rk.x + (uint32_t)__popc(rk.y & ((1u << (3u * (q & 7u) + (ed & 3u))) - 1u)));
      }
      if (o + j < tcap) {
        int32_t* const out = tris + 3 * (o + j);
        out[0] = id[0];
        out[1] = id[1];
        out[2] = id[2];
      }
    }
    wave_sync();
  }
}

// koff is the exclusive scan of the keep flags: triangle i is kept when its
// offset differs from the next one (or from the total for the last).
__global__ __launch_bounds__(kMcBlock) void k_mc_squeeze(const int32_t* __restrict__ tris_pre,
                                                         const uint32_t* __restrict__ koff, int64_t n,
                                                         const uint32_t* __restrict__ total,
                                                         int32_t* __restrict__ tris) {
  const int64_t i = (int64_t)blockIdx.x * kMcBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t o = koff[i];
  const uint32_t next = (i + 1 < n) ? koff[i + 1] : *total;
  if (next == o) return;
  tris[3 * (int64_t)o + 0] = tris_pre[3 * i + 0];
  tris[3 * (int64_t)o + 1] = tris_pre[3 * i + 1];
  tris[3 * (int64_t)o + 2] = tris_pre[3 * i + 2];
}

// ---------------------------------------------------------------- host side

template <class T>
static qj_status grow(T*& p, int64_t& cap, int64_t n, hipStream_t s) {
  if (n <= cap) return QJ_OK;
  if (p) {
    QJ_HIP(hipStreamSynchronize(s));
    QJ_HIP(hipFree(p));
    p = nullptr;
    cap = 0;
  }
  const int64_t want = n + n / 8 + 1024;
  QJ_HIP(hipMalloc(&p, sizeof(T) * (size_t)want));
  cap = want;
  return QJ_OK;
}

static unsigned nblocks(int64_t n) { return (unsigned)((n + kMcBlock - 1) / kMcBlock); }

// whether the cell-centre map is a rotation (edges meeting at a corner stay
// perpendicular) and every grid spacing lies in [lo, hi]
template <class G>
static bool is_turned_grid(const G& g, double lo, double hi) {
  bool ok = true;
  for (int i = 0; i < 3; i++) {
    ok &= fabs(g.dx[i]) >= lo && fabs(g.dx[i]) <= hi;
    for (int j = 0; j < 3; j++) {
      const double d = g.rot[i] * g.rot[j] + g.rot[3 + i] * g.rot[3 + j] + g.rot[6 + i] * g.rot[6 + j];
      ok &= fabs(d - (i == j ? 1.0 : 0.0)) < 1e-9;
    }
  }
  return ok;
}

// a bound on the coordinates' magnitudes
template <class G>
static double grid_extent(const G& g) {
  double e = 0.0;
  for (int i = 0; i < 3; i++) e += fabs(g.center[i]) + fabs(g.dx[i]) * g.res[i];
  return e;
}

static dim3 blocks_of(int64_t items, int64_t per) { return dim3((unsigned)((items + per - 1) / per)); }

static qj_status launch_tris(const McState& m, const McGrid& mg, const uint32_t* gv, const uint32_t* gt,
                             const uint64_t* base, uint32_t id0, int64_t tcap, int32_t* tris, hipStream_t s) {
  const int64_t nb = (mg.nw + 3) / 4;
  const int per = (int)std::min<int64_t>(kTriBlocks, std::max<int64_t>(1, nb / kTriWaves));
  hipLaunchKernelGGL(k_mc_tris, blocks_of(nb, per * kMcWaves), dim3(kMcBlock), 0, s, mg, per, (const uint8_t*)m.flags,
                     (const uint64_t*)mg.drop, (const uint8_t*)m.kmask, (const uint2*)m.ranks, gv,
                     (const uint32_t*)m.tword, gt, base, id0, tcap, tris);
  QJ_HIP(hipGetLastError());
  return QJ_OK;
}

// Words per block of k_mc_measure, or 0 where k_mc_cells measures: where estimates
// decide nearly all (kMeasureUnsure), and beyond two groups per CU. 256 cells a block,
// one per thread, until 2048 blocks fill the chip, then more. Calls in us, in
// k_mc_cells and in a kernel of its own (a case byte per cell and a kernel over all
// cells, before): kMeasureAll, noise, 24^3 409 / 66 (123), 64^3 545 / 87 (139), 97^3
// 578 / 147 (216), 160^3 601 / 439 (584), 168^3 858 / 503 (677), 200^3 957 / 824 (1057),
// 256^3 1811 / 1706 (2231); a sphere's surface 77 / 55 (110), 73 / 56 (114), 69 / 65
// (122), 87 / 90 (171), 87 / 90 (174), 100 / 105 (206), 142 / 160 (311).
static int measure_words(const McGrid& a, int64_t groups) {
  if (a.prefilter == kMeasureUnsure || groups > 512) return 0;
  return (int)std::min<int64_t>(kMeasureWords, std::max<int64_t>(4, (a.nw + 2047) / 2048));
}

// Meshes n fields one after another on the stream without waiting on the
// host: every count stays on the device (running vertex and triangle totals,
// per-tile counts) and is read back once at the end. The vertex and triangle
// buffers keep their size from earlier calls; a pass that outgrows them
// writes nothing beyond them, and the host then sizes them from the totals it
// read and runs the pass again.
// ext_v / ext_t (with their capacities in vertices and triangles): the
// caller's buffers, written directly in one pass; null = the workspace's.
qj_status mc_run_tiles(qj_workspace* ws, int n, const double* const* fields, const qj_grid* grids, double iso,
                       int64_t* nv_out, int64_t* nt_out, hipStream_t s, double* ext_v, int64_t ext_vcap,
                       int32_t* ext_t, int64_t ext_tcap) {
  const bool ext = ext_v != nullptr;
  if (!ws->mc) ws->mc = new McState();
  McState& m = *(McState*)ws->mc;
  m.nv = m.nt = 0;
  m.cache_valid = false;
  if (n <= 0) return QJ_OK;
  std::vector<GridGeom> geo((size_t)n);
  std::vector<int> prefilter((size_t)n);
  int64_t nmax = 0, total_pts = 0, pad_max = 0;
  bool measured = false;
  for (int k = 0; k < n; k++) {
    GridGeom& g = geo[(size_t)k];
    make_geom(&grids[k], &g);
    const int64_t N = (int64_t)g.res[0] * g.res[1] * g.res[2];
    const int64_t cells = (int64_t)(g.res[0] - 1) * (g.res[1] - 1) * (g.res[2] - 1);
    if (N > (int64_t)UINT32_MAX || 5 * cells > (int64_t)INT32_MAX) {
      set_error("marching cubes on %lld points exceeds 32-bit vertex/triangle ids; split the field in tiles",
                (long long)N);
      return QJ_ERR_CAPACITY;
    }
    nmax = N > nmax ? N : nmax;
    total_pts += N;
    pad_max = std::max(pad_max, mc_pad_words(g));
    prefilter[(size_t)k] = !is_turned_grid(g, kPrefilterSpacing, kPrefilterMaxSpacing) ? kMeasureAll
                           : grid_extent(g) <= kSureExtent                            ? kMeasureUnsure
                                                                                      : kMeasureNear;
    measured |= prefilter[(size_t)k] != kMeasureUnsure;
  }
  qj_status st;
  // words of 64 points, plus what the reads of a word's +y and +z rows run past the end
  const int64_t wmax = (nmax + 63) / 64 + pad_max;
  const int64_t gmax = (nmax + kMcGroupPoints - 1) / kMcGroupPoints;
  if ((st = grow(m.words, m.cap_words, kMcArrays * wmax, s)) || (st = grow(m.ranks, m.cap_ranks, 8 * wmax, s)) ||
      (st = grow(m.flags, m.cap_flags, 64 * ((nmax + 63) / 64), s)) || (st = grow(m.kmask, m.cap_kmask, nmax, s)) ||
      (st = grow(m.tword, m.cap_tword, wmax, s)) || (measured && (st = grow(m.lost, m.cap_lost, wmax, s))) ||
      (st = grow(m.groups, m.cap_groups, 2 * gmax, s)) || (st = grow(m.d_base, m.cap_base, 2 * ((int64_t)n + 1), s)))
    return st;
  if (!m.tickets) {
    // cleared before anything else can count on them: an error return below does not
    // wait for s, and the next call may come on another stream
    const size_t bytes = sizeof(uint32_t) * kTicketLine * (kTickets + 1);
    uint32_t* t = nullptr;
    QJ_HIP(hipMalloc(&t, bytes));
    hipError_t e = hipMemsetAsync(t, 0, bytes, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
      hipFree(t);
      return hip_fail(e, "clearing the tickets");
    }
    m.tickets = t;
  }
  // first sizes: a quarter of the points as vertices, half as triangles
  // (a 256^3 torus tile holds 0.42 and 0.73 of its points)
  if (!ext && m.cap_v == 0 && (st = grow(m.verts, m.cap_v, 3 * (total_pts / 4 + 1024), s))) return st;
  if (!ext && m.cap_t == 0 && (st = grow(m.tris, m.cap_t, 3 * (total_pts / 2 + 1024), s))) return st;
  if ((st = ensure_pinned(ws, 2 * ((int64_t)n + 1), s))) return st;
  uint64_t* const base = (uint64_t*)ws->h_pinned;
  base[0] = base[1] = 0;
  std::vector<int64_t> counts(2 * (size_t)n);
  uint64_t totals[2] = {0, 0};
  for (int pass = 0; pass < 2; pass++) {
    const int64_t vcap = ext ? ext_vcap : m.cap_v / 3, tcap = ext ? ext_tcap : m.cap_t / 3;
    double* const verts = ext ? ext_v : m.verts;
    int32_t* const tris = ext ? ext_t : m.tris;
    for (int k = 0; k < n; k++) {
      const GridGeom& g = geo[(size_t)k];
      const int64_t N = (int64_t)g.res[0] * g.res[1] * g.res[2];
      const int64_t cells = (int64_t)(g.res[0] - 1) * (g.res[1] - 1) * (g.res[2] - 1);
      const McGrid mg = make_mc_grid(m, g, wmax, iso, prefilter[(size_t)k]);
      const int64_t ng = cells > 0 ? (N + kMcGroupPoints - 1) / kMcGroupPoints : 0;
      uint32_t *gv = m.groups, *gt = m.groups + gmax;
      const ScanTail tail{ng <= kFoldGroups ? m.d_base : nullptr, base, m.tickets, k};
      const auto scan = [&](uint32_t* groups, int which) -> qj_status {
        if (ng > 0 && ng <= kFoldGroups) return QJ_OK;  // the kernel before it did
        hipLaunchKernelGGL(k_mc_scan, dim3(1), dim3(kScanBlock), 0, s, groups, ng, m.d_base, base, k, which);
        QJ_HIP(hipGetLastError());
        return QJ_OK;
      };
      if (ng) {
        hipLaunchKernelGGL(k_mc_signs, blocks_of(N, kSignPoints * kMcBlock), dim3(kMcBlock), 0, s, fields[k], N, iso,
                           mg.sgn);
        QJ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_mc_edges, dim3((unsigned)ng), dim3(kMcBlock), 0, s, mg, m.ranks, gv, tail);
        QJ_HIP(hipGetLastError());
      }
      if ((st = scan(gv, 0))) return st;
      if (ng) {
        const bool few = mg.nw < 2 * kTriWaves * 8;
        hipLaunchKernelGGL(few ? k_mc_vertices<2> : k_mc_vertices<8>, blocks_of(mg.nw, (few ? 2 : 8) * kMcWaves),
                           dim3(kMcBlock), 0, s, fields[k], mg,
                           (const uint2*)m.ranks, (const uint32_t*)gv, (const uint64_t*)(m.d_base + 2 * k), vcap,
                           verts);
        QJ_HIP(hipGetLastError());
        const uint32_t* lost = nullptr;
        if (const int words = measure_words(mg, ng)) {
          hipLaunchKernelGGL(k_mc_measure, blocks_of(mg.nw, words), dim3(kMcBlock), 0, s, fields[k], mg, words,
                             m.kmask, m.lost);
          QJ_HIP(hipGetLastError());
          lost = m.lost;
        }
        hipLaunchKernelGGL(k_mc_cells, dim3((unsigned)ng), dim3(kMcBlock), 0, s, fields[k], mg, m.flags, m.kmask, lost,
                           m.tword, gt, tail);
        QJ_HIP(hipGetLastError());
      }
      if ((st = scan(gt, 1))) return st;
      if (ng && (st = launch_tris(m, mg, gv, gt, (const uint64_t*)(m.d_base + 2 * k), 0, tcap, tris, s))) return st;
    }
    QJ_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < n; k++)
      for (int i = 0; i < 2; i++)
        counts[2 * (size_t)k + i] = (int64_t)(base[2 * ((size_t)k + 1) + i] - base[2 * (size_t)k + i]);
    totals[0] = base[2 * (size_t)n];
    totals[1] = base[2 * (size_t)n + 1];
    if ((int64_t)totals[0] <= vcap && (int64_t)totals[1] <= tcap) break;
    if (ext) {
      // the caller's buffers are too small: report the sizes needed
      for (int k = 0; k < n; k++) {
        if (nv_out) nv_out[k] = counts[2 * (size_t)k];
        if (nt_out) nt_out[k] = counts[2 * (size_t)k + 1];
      }
      set_error("marching cubes: the meshes need %llu vertices and %llu triangles (buffers for %lld and %lld)",
                (unsigned long long)totals[0], (unsigned long long)totals[1], (long long)vcap, (long long)tcap);
      return QJ_ERR_CAPACITY;
    }
    if (pass == 1) {
      set_error("marching cubes: counts changed between two passes over the same fields");
      return QJ_ERR_NUMERIC;
    }
    // outgrown: size the buffers from this pass's totals and mesh again
    if ((st = grow(m.verts, m.cap_v, 3 * (int64_t)totals[0], s)) ||
        (st = grow(m.tris, m.cap_t, 3 * (int64_t)totals[1], s)))
      return st;
  }
  m.nv = ext ? 0 : (int64_t)totals[0];
  m.nt = ext ? 0 : (int64_t)totals[1];
  for (int k = 0; k < n; k++) {
    if (nv_out) nv_out[k] = counts[2 * (size_t)k];
    if (nt_out) nt_out[k] = counts[2 * (size_t)k + 1];
  }
  return QJ_OK;
}

qj_status mc_run(qj_workspace* ws, const double* d_field, const qj_grid* grid, double iso, int64_t* nv_out,
                 int64_t* nt_out, hipStream_t s) {
  *nv_out = *nt_out = 0;
  return mc_run_tiles(ws, 1, &d_field, grid, iso, nv_out, nt_out, s);
}

qj_status mc_copy(qj_workspace* ws, double* v, int32_t* t, hipStream_t s) {
  McState* m = (McState*)ws->mc;
  if (!m) return QJ_ERR_INVALID;
  if (v && m->nv) QJ_HIP(hipMemcpyAsync(v, m->verts, sizeof(double) * 3 * m->nv, hipMemcpyDefault, s));
  if (t && m->nt) QJ_HIP(hipMemcpyAsync(t, m->tris, sizeof(int32_t) * 3 * m->nt, hipMemcpyDefault, s));
  QJ_HIP(hipStreamSynchronize(s));
  return QJ_OK;
}

qj_status mc_ptrs(qj_workspace* ws, const double** v, const int32_t** t) {
  McState* m = (McState*)ws->mc;
  if (!m) return QJ_ERR_INVALID;
  if (v) *v = m->verts;
  if (t) *t = m->tris;
  return QJ_OK;
}

void mc_free(qj_workspace* ws) {
  McState* m = (McState*)ws->mc;
  if (!m) return;
  hipFree(m->flags);
  hipFree(m->words);
  hipFree(m->ranks);
  hipFree(m->kmask);
  hipFree(m->tword);
  hipFree(m->groups);
  hipFree(m->tri_off);
  hipFree(m->verts);
  hipFree(m->tris_pre);
  hipFree(m->keep);
  hipFree(m->tris);
  hipFree(m->tmp);
  hipFree(m->totals);
  hipFree(m->slab[0]);
  hipFree(m->slab[1]);
  if (m->s2) {
    hipStreamSynchronize(m->s2);
    hipStreamDestroy(m->s2);
  }
  for (hipEvent_t e : {m->ev_start, m->ev_field[0], m->ev_field[1], m->ev_free[0], m->ev_free[1]})
    if (e) hipEventDestroy(e);
  hipFree(m->aword);
  hipFree(m->lost);
  hipFree(m->vpt);
  hipFree(m->vax);
  hipFree(m->d_bad);
  hipFree(m->c_edges);
  hipFree(m->c_cells);
  hipFree(m->d_base);
  hipFree(m->tickets);
  delete m;
  ws->mc = nullptr;
}


// ---------------------------------------------------------------- non-linear low-memory mesher

// TRIANGLE_MESH::computeNonlinearMarchingCubesLowMemoryHuge (TRIANGLE_MESH.cpp:681-768)
// streamed over z-chunks: for chunk [z0, z1) the map is evaluated on slices
// [z0, z1 + 1] (two above for the edges of the points at z1, whose ids belong to
// the next chunk, which takes over their values; none below: an edge's ends say
// whether it carries a vertex),
// cases come from the raw slab values log|q| (TRIANGLE_MESH.cpp:379) as sign
// words, as in the linear mesher, and every vertex is
// placed by bisection on re-evaluated values log|q| - iso (nonlinearValue
// :1755-1795, midpointSearch :2232-2271, at most 6 halvings, early exit at
// |value| < 1e-8). Vertex numbering, triangle order and the degenerate filter
// are those of the linear mesher. The re-evaluations take exponents 1 and 2
// as exact products (b and b b) and others in the polar form, as the FP64
// band does: the values differ from the polar form's in the last few ulps,
// the same order as the device math library against the host's.

// kPow: kExactOnly when every exponent is 1 or 2 (no polar code, far fewer
// registers), kExactInt otherwise; both give the same values for exponents 1
// and 2. kMap: the map in Lagrange order (QJ_MAP_LAGRANGE), in the extended
// range (QJ_MAP_EXTENDED_RANGE) or neither.
enum NlMap { kNlPlain = 0, kNlExt = 1, kNlLag = 2 };
template <int kPow, int kMap>
__device__ __forceinline__ double nonlinear_value(const MapArgs& a, const RootRec64* __restrict__ roots,
                                                  const double* p, double iso) {
  if (kMap == kNlLag) {
    // lagrangeNonlinearValue (TRIANGLE_MESH.cpp:1684-1730): an infinite |q|
    // restores the previous iterate and stops. Before the first iteration the
    // reference's previous magnitude is uninitialised; here it is |q0|.
    q64 q{p[0], p[1], p[2], a.slice};
    double magnitude = qmag(q), prev = magnitude;
    int it = 0;
    while (magnitude < a.escape && it < a.max_iter) {
      q = qscale(lagrange64<kPow>((ConstRoots)roots, a.nt, a.nb, q), a.exp_scaling);
      magnitude = qmag(q);
      if (isinf(magnitude)) {
        magnitude = prev;
        break;
      }
      prev = magnitude;
      it++;
      if (magnitude < kBlackHole) it = a.max_iter;
    }
    // an infinite value (|q| = 0) is reported as FLT_MAX (TRIANGLE_MESH.cpp:1733-1742)
    const double v = log(magnitude) - iso;
    return isinf(v) ? (double)FLT_MAX : v;
  }
  const q64 q0{p[0], p[1], p[2], a.slice};
  const Res64 r = kMap == kNlExt ? eval64e<kPow>(a, (ConstRoots)roots, q0) : eval64<kPow>(a, (ConstRoots)roots, q0);
  return r.F - iso;
}

// One vertex by bisection between grid points (x, y, z) and its +axis
// neighbour (computeNonlinearEdgeInterpolationsHuge :2034-2123 with
// midpointSearch :2232-2271). fa, fb: the field values at the two ends when the
// caller has them (the values minus iso are the end values), else null and they
// are evaluated. Counts edges whose end values do not straddle the surface in
// *bad (the reference exits there). Ends and midpoints go through one
// evaluation in one loop, so the map's code is there once (three inlined copies
// took 51 KB of instructions and 172 VGPRs for exponents 1 and 2).
template <int kPow, int kMap>
__device__ __forceinline__ void place_vertex(const MapArgs& a, const RootRec64* __restrict__ roots, double iso,
                                             int x, int y, int z, int axis, const double* fa, const double* fb,
                                             double* __restrict__ out, unsigned int* __restrict__ bad) {
#pragma clang fp contract(off)
  double pp[3], pn[3], m[3], vp = 0.0, vn = 0.0;
  cell_center(a, x, y, z, pp);
  cell_center(a, x + (axis == 0), y + (axis == 1), z + (axis == 2), pn);
  if (fa) {
    vp = *fa - iso;
    vn = *fb - iso;
  }
  // steps -2 and -1 evaluate the lower and the upper end, then up to 6 midpoints
  for (int step = fa ? 0 : -2;; step++) {
    if (step < 0) {
      m[0] = step == -2 ? pp[0] : pn[0];
      m[1] = step == -2 ? pp[1] : pn[1];
      m[2] = step == -2 ? pp[2] : pn[2];
    } else {
      if (step == 0) {
        // the positive end is the first (the lower endpoint) unless its value is negative
        if (vp * vn >= 0.0) atomicAdd(bad, 1u);  // the reference exits here (:2082-2097)
        if (vp < 0) {
          for (int i = 0; i < 3; i++) {
            const double t = pp[i];
            pp[i] = pn[i];
            pn[i] = t;
          }
          const double t = vp;
          vp = vn;
          vn = t;
        }
      }
      m[0] = pp[0] + pn[0];
      m[1] = pp[1] + pn[1];
      m[2] = pp[2] + pn[2];
      m[0] *= 0.5;
      m[1] *= 0.5;
      m[2] *= 0.5;
      if (vp * vn >= 0.0) {
        if (step > 0) atomicAdd(bad, 1u);
        break;
      }
      if (step >= 6) break;
    }
    const double v = nonlinear_value<kPow, kMap>(a, roots, m, iso);
    if (step == -2) {
      vp = v;
    } else if (step == -1) {
      vn = v;
    } else {
      if (fabs(v) < 1e-8) break;
      const bool neg = v < 0;
      for (int i = 0; i < 3; i++) {
        pn[i] = neg ? m[i] : pn[i];
        pp[i] = neg ? pp[i] : m[i];
      }
      vn = neg ? v : vn;
      vp = neg ? vp : v;
    }
  }
  out[0] = m[0];
  out[1] = m[1];
  out[2] = m[2];
}

// Triangles and active cells of a slab, one word of cells per thread, as
// k_mc_cells counts them. (One slab of 66 slices of 256^2: signs, edges and this
// 19, 11 and 15 us; case bytes and edges from them 62 and 78, and five scans.) tword, aword: before word w in its group; groups: per
// group, triangles from 0 on and active cells from `ngroups` on. kLost: the
// triangles less those that k_nl_filter dropped.
template <bool kLost>
__global__ __launch_bounds__(kMcBlock) void k_nl_count(McGrid a, uint8_t* __restrict__ flags,
                                                       const uint32_t* __restrict__ lost,
                                                       uint32_t* __restrict__ tword, uint32_t* __restrict__ aword,
                                                       uint32_t* __restrict__ groups, int64_t ngroups) {
  const int64_t w = (int64_t)blockIdx.x * kMcGroupWords + threadIdx.x;
  uint32_t count = 0, active = 0, total;
  if (w < a.nw) {
    active = (uint32_t)__popcll(word_cases(a, w, flags, &count));
    if (kLost) count -= lost[w];
    else a.drop[w] = 0;
  }
  const uint32_t t = block_prefix<kMcBlock>(count, &total);
  if (threadIdx.x == 0) groups[blockIdx.x] = total;
  const uint32_t c = block_prefix<kMcBlock>(active, &total);
  if (threadIdx.x == 0) groups[ngroups + blockIdx.x] = total;
  if (w >= a.nw) return;
  tword[w] = t;
  aword[w] = c;
}

// One block: groups holds n counts each of vertices, triangles and active
// cells; all to exclusive offsets in place, and to pinned memory: the vertices of
// points below p, all vertices, triangles, active cells. The block is small: one of
// 1024 threads waited 0.3 ms for a CU with room for its 16 waves while the next
// slab was evaluated on the other stream.
constexpr int kTotalsBlock = 256;
__global__ __launch_bounds__(kTotalsBlock) void k_nl_totals(uint32_t* __restrict__ groups, int64_t n,
                                                          const uint2* __restrict__ ranks, int64_t p, int64_t owned,
                                                          uint32_t* __restrict__ h_out) {
  const int64_t per = (n + kTotalsBlock - 1) / kTotalsBlock, b = (int64_t)threadIdx.x * per;
  uint32_t all = 0;
  for (int which = 0; which < 3; which++, groups += n) {
    uint32_t v = 0, total;
    for (int64_t i = b; i < b + per && i < n; i++) v += groups[i];
    uint32_t run = block_prefix<kTotalsBlock>(v, &total);
    for (int64_t i = b; i < b + per && i < n; i++) {
      const uint32_t c = groups[i];
      // the thread that holds p's group
      if (which == 0 && i == p / kMcGroupPoints && p < owned) {
        const uint2 rk = ranks[p >> 3];
        h_out[0] = run + rk.x + (uint32_t)__popc(rk.y & ((1u << (3 * (p & 7))) - 1u));
      }
      groups[i] = run;
      run += c;
    }
    if (which == 0) all = total;
    if (threadIdx.x == 0) h_out[1 + which] = total;
  }
  if (threadIdx.x == 0 && p >= owned) h_out[0] = all;
}

// The slab's vertices from local id `from` on, in id order: the owning point
// and the edge's axis. One wave per word of points.
__global__ __launch_bounds__(kMcBlock) void k_nl_vlist(McGrid a, const uint64_t* __restrict__ ex,
                                                       const uint64_t* __restrict__ ey,
                                                       const uint64_t* __restrict__ ez,
                                                       const uint2* __restrict__ ranks,
                                                       const uint32_t* __restrict__ groups, uint32_t from,
                                                       uint32_t* __restrict__ vpt, uint8_t* __restrict__ vax) {
  const int64_t w0 = ((int64_t)blockIdx.x * kMcWaves + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) *
                     kListWords;
  const int lane = threadIdx.x & 63;
#pragma unroll 1
  for (int i = 0; i < kListWords; i++) {
    const int64_t w = w0 + i;
    if (w >= a.nw) break;
    const uint64_t e[3] = {ex[w], ey[w], ez[w]};
    if (!(e[0] | e[1] | e[2])) continue;
    uint32_t k = groups[w / kMcGroupWords] + ranks[8 * w].x;
#pragma unroll
    for (int axis = 0; axis < 3; axis++)
      k = __builtin_amdgcn_mbcnt_hi((uint32_t)(e[axis] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)e[axis], k));
#pragma unroll
    for (int axis = 0; axis < 3; axis++)
      if (__builtin_amdgcn_inverse_ballot_w64(e[axis])) {
        if (k >= from) {
          vpt[k - from] = (uint32_t)(64 * w + lane);
          vax[k - from] = (uint8_t)axis;
        }
        k++;
      }
  }
}

// Vertices by bisection, one per thread over the list: both end values
// (evaluated, or read from the slab), then up to 6 midpoints (FP64 map
// evaluations on full waves; about one point in ten owns an edge, so a thread
// per point would leave most lanes idle). List entry t, a point of the slab
// that starts at slice z0, gets id base + t. ends: null, or the slab's values,
// when they are the end values' own (see slab_holds_end_values); the midpoints
// are always evaluated.
// FP64 VALU bound beside the next slab's FP32 evaluation. No bound on the
// registers (151 for exponents 1 and 2): held to five or four waves per SIMD
// (136 to 224 B spilled) meshes take -1 to 4 % longer.
template <int kPow, int kMap>
__global__ __launch_bounds__(kMcBlock) void k_nl_vertices(MapArgs a, const RootRec64* __restrict__ roots,
                                                          double iso, int64_t z0, const double* __restrict__ ends,
                                                          uint32_t n, const uint32_t* __restrict__ vpt,
                                                          const uint8_t* __restrict__ vax, uint32_t base,
                                                          double* __restrict__ verts, int32_t* __restrict__ edges,
                                                          unsigned int* __restrict__ bad) {
  const uint32_t t = blockIdx.x * kMcBlock + threadIdx.x;
  if (t >= n) return;
  const int64_t k = (int64_t)base + t;
  const int64_t X = a.res[0], XY = X * a.res[1];
  const int64_t q = vpt[t];
  const int axis = vax[t];
  const int64_t lz = q / XY, r = q - lz * XY;
  const int y = (int)(r / X), x = (int)(r - (int64_t)y * X), z = (int)(z0 + lz);
  const double* fa = ends ? ends + q : nullptr;
  const double* fb = ends ? ends + q + (axis == 0 ? 1 : axis == 1 ? X : XY) : nullptr;
  place_vertex<kPow, kMap>(a, roots, iso, x, y, z, axis, fa, fb, verts + 3 * k, bad);
  edges[4 * k + 0] = x;
  edges[4 * k + 1] = y;
  edges[4 * k + 2] = z;
  edges[4 * k + 3] = axis;
}

// Launch a mesher vertex kernel instantiated for the map's power mode and
// order (see nonlinear_value).
template <class... Args>
static void launch_nl_vertices(const MapArgs& a, dim3 grid, hipStream_t s, Args... args) {
  const int map = (a.flags & QJ_MAP_LAGRANGE) ? kNlLag : (a.flags & QJ_MAP_EXTENDED_RANGE) ? kNlExt : kNlPlain;
  const auto k = a.gen ? (map == kNlLag   ? k_nl_vertices<kExactInt, kNlLag>
                          : map == kNlExt ? k_nl_vertices<kExactInt, kNlExt>
                                          : k_nl_vertices<kExactInt, kNlPlain>)
                       : (map == kNlLag   ? k_nl_vertices<kExactOnly, kNlLag>
                          : map == kNlExt ? k_nl_vertices<kExactOnly, kNlExt>
                                          : k_nl_vertices<kExactOnly, kNlPlain>);
  hipLaunchKernelGGL(k, grid, dim3(kMcBlock), 0, s, a, args...);
}
// (x, y, z, flag) of the slab's active cells, in cell order; the slab starts at slice z0
__global__ __launch_bounds__(kMcBlock) void k_nl_cells(McGrid a, const uint8_t* __restrict__ flags,
                                                       const uint32_t* __restrict__ aword,
                                                       const uint32_t* __restrict__ groups, int64_t z0,
                                                       int32_t* __restrict__ cells) {
  const int64_t p = (int64_t)blockIdx.x * kMcBlock + threadIdx.x, w = p >> 6;
  const int lane = threadIdx.x & 63;
  const unsigned flag = p < a.cells ? flags[p] : 0u;
  const uint64_t act = __ballot(flag != 0u);
  if (!flag) return;
  const int64_t k = (int64_t)groups[w / kMcGroupWords] + aword[w] + __popcll(act & ((1ull << lane) - 1ull));
  int64_t x, y, z;
  point_xyz(a.g, p, x, y, z);
  ((int4*)cells)[k] = int4{(int32_t)x, (int32_t)y, (int32_t)(z0 + z), (int32_t)flag};
}

// The degenerate filter (TRIANGLE_MESH.cpp:1088-1102) on every triangle of a
// slab, one cell per thread: kmask holds what is left of a cell that lost any,
// drop their bits and lost the triangles per word. Only for grids whose spacing
// or map leaves the answer open (see nlmc_run).
__global__ __launch_bounds__(kMcBlock) void k_nl_filter(McGrid a, const uint8_t* __restrict__ flags,
                                                        const uint2* __restrict__ ranks,
                                                        const uint32_t* __restrict__ groups, uint32_t id0,
                                                        const double* __restrict__ verts, uint8_t* __restrict__ kmask,
                                                        uint32_t* __restrict__ lost) {
  __shared__ uint32_t s_tri[1024];
  __shared__ uint8_t s_ntri[256];
  stage_tri(s_tri, s_ntri);
  const int64_t p = (int64_t)blockIdx.x * kMcBlock + threadIdx.x, w = p >> 6;
  const int64_t X = a.g.res[0];
  const int flag = p < a.cells ? (int)flags[p] : 0;
  const int n = flag ? s_ntri[flag] : 0;
  unsigned dropped = 0;
  for (int t = 0; t < n; t++) {
    const double* v[3];
    for (int q = 0; q < 3; q++) {
      int dx, dy, dz, axis;
      edge_geom(tri_edge(s_tri, flag, 3 * t + q), dx, dy, dz, axis);
      const int64_t o = p + dx + dy * X + dz * a.XY;
      const uint2 rk = ranks[o >> 3];
      v[q] = verts + 3 * ((int64_t)id0 + groups[o / kMcGroupPoints] + rk.x +
                          __popc(rk.y & ((1u << (3 * (o & 7) + axis)) - 1u)));
    }
    const double eps = 1e-7;
    if (edge_len(v[0], v[1]) < eps || edge_len(v[0], v[2]) < eps || edge_len(v[1], v[2]) < eps) dropped |= 1u << t;
  }
  if (dropped) kmask[p] = (uint8_t)(((1u << n) - 1u) & ~dropped);
  const uint64_t m = __ballot(dropped != 0u);
  const uint32_t sum = wave_last(wave_inclusive((uint32_t)__popc(dropped)));
  if ((threadIdx.x & 63) == 0 && w < a.nw) {
    a.drop[w] = m;
    lost[w] = sum;
  }
}

template <class T>
static qj_status grow_keep(T*& p, int64_t& cap, int64_t n, int64_t used, hipStream_t s) {
  if (n <= cap) return QJ_OK;
  const int64_t want = n + n / 2 + 4096;
  T* q = nullptr;
  QJ_HIP(hipMalloc(&q, sizeof(T) * (size_t)want));
  if (p && used > 0) QJ_HIP(hipMemcpyAsync(q, p, sizeof(T) * (size_t)used, hipMemcpyDeviceToDevice, s));
  QJ_HIP(hipStreamSynchronize(s));
  if (p) QJ_HIP(hipFree(p));
  p = q;
  cap = want;
  return QJ_OK;
}

// Whether the slab's values can stand in for the bisection's end values
// (TRIANGLE_MESH.cpp:2063-2067 evaluates them again with nonlinearValue,
// whose values the reference's slices hold too: computeNonlinearSlice
// :330-378). In the FP32 + FP64 band field every cell with |F| < band holds
// the FP64 value of the evaluator nonlinear_value calls (k_list64 and
// k_band_sweep with the same power mode and range), and every other cell an
// FP32 value of the FP64 value's sign: with iso 0 the end values enter the
// bisection only through their signs (the orientation and the straddle
// tests; products of values of magnitude band or more do not underflow), so
// the vertices are those of the evaluated end values. Not for the caller's
// field (its values are not the map's), the Lagrange order (its value has
// its own infinite case), the plain FP64 slabs (the same values, but not worth
// a case of their own), the AP flags or a band of 0.
static bool slab_holds_end_values(const MapArgs& a, const double* src_field, double iso, qj_precision prec,
                                  double band) {
  return !src_field && prec == QJ_FP32_BAND && iso == 0.0 && band > 0.0 &&
         !(a.flags & (QJ_MAP_LAGRANGE | QJ_MAP_SKIP_ORIGIN | QJ_MAP_ADAPTIVE));
}

// what the word kernels need of a slab: its points' places in memory
static void slab_geom(const MapArgs& a, GridGeom* g) {
  *g = GridGeom{};
  for (int i = 0; i < 3; i++) g->res[i] = a.res[i];
  g->div_x = make_fastdiv((uint32_t)a.res[0]);
  g->div_xy = make_fastdiv((uint32_t)((int64_t)a.res[0] * a.res[1]));
}

qj_status nlmc_run(qj_workspace* ws, const MapArgs& a0, const qj_rational* f, double iso, qj_precision prec,
                   double band, int chunk, int64_t* nv_out, int64_t* nt_out, int64_t* n_bad, hipStream_t s,
                   const double* src_field) {
  if (!ws->mc) ws->mc = new McState();
  McState& m = *(McState*)ws->mc;
  m.nv = m.nt = 0;
  const int64_t X = a0.res[0], Y = a0.res[1], Z = a0.res[2], XY = X * Y;
  *nv_out = *nt_out = 0;
  *n_bad = 0;
  m.ncells = 0;
  m.cache_valid = false;
  if (X < 2 || Y < 2 || Z < 2) return QJ_OK;
  if (chunk < 1) chunk = 64;
  if (XY * (int64_t)(chunk + 3) > (int64_t)UINT32_MAX) {
    set_error("non-linear mesher: slab of %lld points exceeds 32-bit indices", (long long)(XY * (chunk + 3)));
    return QJ_ERR_CAPACITY;
  }
  const int64_t slab_pts = XY * (chunk + 2);
  qj_status st;
  // the slab stream is idle whenever the call returns, early error returns
  // included (its slab evaluations read the caller's roots)
  struct JoinOnExit {
    hipStream_t s = nullptr;
    ~JoinOnExit() {
      if (s) hipStreamSynchronize(s);
    }
  } join;
  if (!src_field) {
    if (m.s2) QJ_HIP(hipStreamSynchronize(m.s2));
    if ((st = grow(m.slab[0], m.cap_slab[0], slab_pts, s)) || (st = grow(m.slab[1], m.cap_slab[1], slab_pts, s)))
      return st;
    // the band lists at the largest slab's size, so no slab evaluation regrows them
    if ((st = ensure_list(ws, slab_pts, (a0.flags & QJ_MAP_ADAPTIVE) != 0, s))) return st;
    // created on the first mesh (what a failed creation left out, on the next)
    if (!m.s2) QJ_HIP(hipStreamCreateWithFlags(&m.s2, hipStreamNonBlocking));
    join.s = m.s2;
    for (hipEvent_t* e : {&m.ev_start, &m.ev_field[0], &m.ev_field[1], &m.ev_free[0], &m.ev_free[1]})
      if (!*e) QJ_HIP(hipEventCreateWithFlags(e, hipEventDisableTiming));
  }
  MapArgs a = a0;
  GridGeom geo;
  slab_geom(a, &geo);
  const int64_t wmax = (slab_pts + 63) / 64 + mc_pad_words(geo);
  const int64_t gmax = (slab_pts + kMcGroupPoints - 1) / kMcGroupPoints;
  // Bisection places a vertex at a multiple of 1/128 of its edge inside it (at
  // most six halvings after the first middle), so vertices on edges that meet are
  // at least sqrt(2) / 128 spacings apart, others a spacing: with spacings of
  // 1e-4 no side is below 1e-7 and the filter has nothing to drop.
  const bool sure = is_turned_grid(a, kSureSpacing, DBL_MAX) && grid_extent(a) <= kSureExtent;
  if ((st = grow(m.words, m.cap_words, kMcArrays * wmax, s)) || (st = grow(m.ranks, m.cap_ranks, 8 * wmax, s)) ||
      (st = grow(m.flags, m.cap_flags, 64 * ((slab_pts + 63) / 64), s)) ||
      (st = grow(m.tword, m.cap_tword, wmax, s)) || (st = grow(m.aword, m.cap_aword, wmax, s)) ||
      (st = grow(m.groups, m.cap_groups, 3 * gmax, s)) || (st = grow(m.d_base, m.cap_base, 4, s)) || (st = ensure_pinned(ws, 2, s)) ||
      (!sure && ((st = grow(m.kmask, m.cap_kmask, slab_pts, s)) || (st = grow(m.lost, m.cap_lost, wmax, s)))))
    return st;
  if (!m.d_bad) QJ_HIP(hipMalloc(&m.d_bad, sizeof(unsigned int)));
  QJ_HIP(hipMemsetAsync(m.d_bad, 0, sizeof(unsigned int), s));
  const bool reuse_ends = slab_holds_end_values(a, src_field, iso, prec, band);
  // slices of the slab of the chunk that starts at slice zc: the chunk's and up to two above
  auto slab_slices = [&](int64_t zc) { return std::min(zc + chunk + 2, Z) - zc; };
  // 1. slab of log|q| (or the caller's field, TRIANGLE_MESH.cpp:152-215): the
  // chunk at slice zc into slab[b] on stream s2 (the Lagrange order has no FP32
  // path: its slabs are FP64). Its first two slices are the other slab's last two,
  // evaluated on the same stream: they are copied (256^3 in chunks of 16 slices 4
  // to 6 % faster, of 64 1 to 2).
  auto eval_slab = [&](int64_t zc, int b) -> qj_status {
    const int64_t slices = slab_slices(zc), have = zc > 0 ? std::min<int64_t>(2, slices) : 0;
    if (have)
      QJ_HIP(hipMemcpyAsync(m.slab[b], m.slab[1 - b] + chunk * XY, sizeof(double) * (size_t)(have * XY),
                            hipMemcpyDeviceToDevice, m.s2));
    if (slices > have) {
      MapArgs sa = a;
      sa.res[2] = (int32_t)(slices - have);
      sa.zoff = (int32_t)(zc + have);
      qj_status e = launch_field(ws, sa, f, (a.flags & QJ_MAP_LAGRANGE) ? QJ_FP64 : prec, band, m.slab[b] + have * XY,
                                 m.s2);
      if (e) return e;
    }
    QJ_HIP(hipEventRecord(m.ev_field[b], m.s2));
    return QJ_OK;
  };
  if (!src_field) {
    // the first slab after the work the caller queued on s
    QJ_HIP(hipEventRecord(m.ev_start, s));
    QJ_HIP(hipStreamWaitEvent(m.s2, m.ev_start, 0));
    if ((st = eval_slab(0, 0))) return st;
  }
  uint64_t nv = 0, nt = 0, placed = 0;
  volatile uint32_t* const h = (volatile uint32_t*)ws->h_pinned;
  for (int64_t z0 = 0, ci = 0; z0 < Z; z0 += chunk, ci++) {
    const int64_t z1 = z0 + chunk < Z ? z0 + chunk : Z;
    const int b = (int)(ci & 1);
    const double* slab = src_field ? src_field + z0 * XY : m.slab[b];
    if (!src_field) {
      // the next chunk's slab goes into the other buffer once the previous
      // chunk's vertex kernel, its last reader, is done; this chunk's cases
      // wait for this chunk's slab
      if (z1 < Z) {
        if (ci > 0) QJ_HIP(hipStreamWaitEvent(m.s2, m.ev_free[1 - b], 0));
        if ((st = eval_slab(z1, 1 - b))) return st;
      }
      QJ_HIP(hipStreamWaitEvent(s, m.ev_field[b], 0));
    }
    // 2. signs, edges of the points in slices [z0, z1] and cells of [z0, z1)
    geo.res[2] = (int32_t)slab_slices(z0);
    McGrid mg = make_mc_grid(m, geo, wmax, 0.0, kMeasureAll);
    mg.cells = XY * (std::min(z1, Z - 1) - z0);
    mg.owned = XY * (std::min(z1 + 1, Z) - z0);
    mg.floor = z0 == 0;
    const int64_t ng = (mg.N + kMcGroupPoints - 1) / kMcGroupPoints;
    uint32_t *gv = m.groups, *gt = gv + ng, *ga = gt + ng;
    hipLaunchKernelGGL(k_mc_signs, blocks_of(mg.N, kSignPoints * kMcBlock), dim3(kMcBlock), 0, s, slab, mg.N, 0.0,
                       mg.sgn);
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_mc_edges, dim3((unsigned)ng), dim3(kMcBlock), 0, s, mg, m.ranks, gv, ScanTail{});
    QJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_nl_count<false>, dim3((unsigned)ng), dim3(kMcBlock), 0, s, mg, m.flags,
                       (const uint32_t*)nullptr, m.tword, m.aword, gt, ng);
    QJ_HIP(hipGetLastError());
    // 3. the counts: every buffer is sized from one read-back
    hipLaunchKernelGGL(k_nl_totals, dim3(1), dim3(kTotalsBlock), 0, s, gv, ng, (const uint2*)m.ranks, XY * (z1 - z0),
                       mg.owned, (uint32_t*)ws->h_pinned);
    QJ_HIP(hipGetLastError());
    QJ_HIP(hipStreamSynchronize(s));
    const uint64_t cnt_own = h[0], cnt_all = h[1], ntp = h[2], na = h[3];
    if (nv + cnt_all > (uint64_t)INT32_MAX) return QJ_ERR_CAPACITY;
    // 4. vertices: the chunk's triangles reach the first slice of the next
    // chunk, so that slice's are placed now (with the ids that the next chunk's
    // numbering gives them) and the chunk's own first slice was placed before
    if ((st = grow_keep(m.verts, m.cap_v, 3 * (int64_t)(nv + cnt_all), 3 * (int64_t)(nv + placed), s)) ||
        (st = grow_keep(m.c_edges, m.cap_ce, 4 * (int64_t)(nv + cnt_all), 4 * (int64_t)(nv + placed), s)) ||
        (st = grow_keep(m.c_cells, m.cap_cc, 4 * (m.ncells + (int64_t)na), 4 * m.ncells, s)) ||
        (st = grow_keep(m.tris, m.cap_t, 3 * (int64_t)(nt + ntp), 3 * (int64_t)nt, s)) ||
        (st = grow(m.vpt, m.cap_vpt, (int64_t)cnt_all, s)) || (st = grow(m.vax, m.cap_vax, (int64_t)cnt_all, s)))
      return st;
    if (cnt_all > placed) {
      hipLaunchKernelGGL(k_nl_vlist, blocks_of(mg.nw, kListWords * kMcWaves), dim3(kMcBlock), 0, s, mg,
                         (const uint64_t*)mg.edge[0], (const uint64_t*)mg.edge[1], (const uint64_t*)mg.edge[2],
                         (const uint2*)m.ranks, (const uint32_t*)gv, (uint32_t)placed, m.vpt, m.vax);
      QJ_HIP(hipGetLastError());
      launch_nl_vertices(a, dim3(nblocks((int64_t)(cnt_all - placed))), s, f->d64, iso, z0,
                         reuse_ends ? slab : (const double*)nullptr, (uint32_t)(cnt_all - placed),
                         (const uint32_t*)m.vpt, (const uint8_t*)m.vax, (uint32_t)(nv + placed), m.verts, m.c_edges,
                         m.d_bad);
      QJ_HIP(hipGetLastError());
    }
    if (!src_field) QJ_HIP(hipEventRecord(m.ev_free[b], s));  // the last reader of slab[b] is queued
    // 5. active cells and triangles, in cell order
    uint64_t kept = ntp;
    if (na > 0) {
      hipLaunchKernelGGL(k_nl_cells, dim3(nblocks(mg.cells)), dim3(kMcBlock), 0, s, mg, (const uint8_t*)m.flags,
                         (const uint32_t*)m.aword, (const uint32_t*)ga, z0, m.c_cells + 4 * m.ncells);
      QJ_HIP(hipGetLastError());
      m.ncells += (int64_t)na;
      if (!sure) {
        hipLaunchKernelGGL(k_nl_filter, blocks_of(64 * mg.nw, kMcBlock), dim3(kMcBlock), 0, s, mg,
                           (const uint8_t*)m.flags, (const uint2*)m.ranks, (const uint32_t*)gv, (uint32_t)nv,
                           (const double*)m.verts, m.kmask, m.lost);
        QJ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_nl_count<true>, dim3((unsigned)ng), dim3(kMcBlock), 0, s, mg, m.flags,
                           (const uint32_t*)m.lost, m.tword, m.aword, gt, ng);
        QJ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_mc_scan, dim3(1), dim3(kScanBlock), 0, s, gt, ng, m.d_base, (uint64_t*)nullptr, 0, 1);
        QJ_HIP(hipGetLastError());
        QJ_HIP(hipMemcpyAsync(&kept, m.d_base + 3, sizeof(kept), hipMemcpyDeviceToHost, s));
        QJ_HIP(hipStreamSynchronize(s));
      }
      if ((st = launch_tris(m, mg, gv, gt, nullptr, (uint32_t)nv, (int64_t)ntp, m.tris + 3 * nt, s))) return st;
    }
    nt += kept;
    nv += cnt_own;
    placed = cnt_all - cnt_own;
  }
  unsigned int bad = 0;
  QJ_HIP(hipMemcpyAsync(&bad, m.d_bad, sizeof(bad), hipMemcpyDeviceToHost, s));
  QJ_HIP(hipStreamSynchronize(s));
  m.nv = (int64_t)nv;
  m.nt = (int64_t)nt;
  m.cache_valid = true;
  *nv_out = m.nv;
  *nt_out = m.nt;
  *n_bad = bad;
  if (bad) {
    set_error("non-linear mesher: %u edges whose end values do not straddle the isosurface "
              "(the reference exits at TRIANGLE_MESH.cpp:2082-2097)", bad);
    return QJ_ERR_NUMERIC;
  }
  return QJ_OK;
}

// ---------------------------------------------------------------- edge cache

qj_status nlmc_cache(qj_workspace* ws, int64_t* n_edges, int32_t* edges, int64_t* n_cells, int32_t* cells,
                     hipStream_t s) {
  McState* m = (McState*)ws->mc;
  if (!m || !m->cache_valid) {
    set_error("qj_nlmc_cache: no non-linear mesh in this workspace");
    return QJ_ERR_INVALID;
  }
  if (n_edges) *n_edges = m->nv;
  if (n_cells) *n_cells = m->ncells;
  if (edges && m->nv) QJ_HIP(hipMemcpyAsync(edges, m->c_edges, sizeof(int32_t) * 4 * m->nv, hipMemcpyDefault, s));
  if (cells && m->ncells)
    QJ_HIP(hipMemcpyAsync(cells, m->c_cells, sizeof(int32_t) * 4 * m->ncells, hipMemcpyDefault, s));
  QJ_HIP(hipStreamSynchronize(s));
  return QJ_OK;
}

template <int kPow, int kMap>
__global__ __launch_bounds__(kMcBlock) void k_cache_vertices(MapArgs a, const RootRec64* __restrict__ roots,
                                                             double iso, const int32_t* __restrict__ edges, int64_t ne,
                                                             double* __restrict__ verts,
                                                             unsigned int* __restrict__ bad) {
  const int64_t i = (int64_t)blockIdx.x * kMcBlock + threadIdx.x;
  if (i >= ne) return;
  const int x = edges[4 * i], y = edges[4 * i + 1], z = edges[4 * i + 2], axis = edges[4 * i + 3];
  place_vertex<kPow, kMap>(a, roots, iso, x, y, z, axis, nullptr, nullptr, verts + 3 * i, bad);
}

template <class... Args>
static void launch_cache_vertices(const MapArgs& a, dim3 grid, hipStream_t s, Args... args) {
  const int map = (a.flags & QJ_MAP_LAGRANGE) ? kNlLag : (a.flags & QJ_MAP_EXTENDED_RANGE) ? kNlExt : kNlPlain;
  const auto k = a.gen ? (map == kNlLag   ? k_cache_vertices<kExactInt, kNlLag>
                          : map == kNlExt ? k_cache_vertices<kExactInt, kNlExt>
                                          : k_cache_vertices<kExactInt, kNlPlain>)
                       : (map == kNlLag   ? k_cache_vertices<kExactOnly, kNlLag>
                          : map == kNlExt ? k_cache_vertices<kExactOnly, kNlExt>
                                          : k_cache_vertices<kExactOnly, kNlPlain>);
  hipLaunchKernelGGL(k, grid, dim3(kMcBlock), 0, s, a, args...);
}

__global__ __launch_bounds__(kMcBlock) void k_cache_tricount(const int32_t* __restrict__ cells, int64_t nc,
                                                             uint32_t* __restrict__ tcount) {
  const int64_t i = (int64_t)blockIdx.x * kMcBlock + threadIdx.x;
  if (i < nc) tcount[i] = kMc.ntri[cells[4 * i + 3]];
}

// position of key in the ascending keys, or -1
__device__ __forceinline__ int64_t find_key(const int64_t* __restrict__ keys, int64_t n, int64_t key) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (keys[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return (lo < n && keys[lo] == key) ? lo : -1;
}

__global__ __launch_bounds__(kMcBlock) void k_cache_triangles(
    const int32_t* __restrict__ cells, int64_t nc, int64_t X, int64_t XY, const int64_t* __restrict__ keys,
    int64_t ne, const double* __restrict__ verts, const uint32_t* __restrict__ toff, int32_t* __restrict__ tris_pre,
    uint32_t* __restrict__ keep, unsigned int* __restrict__ missing) {
  const int64_t i = (int64_t)blockIdx.x * kMcBlock + threadIdx.x;
  if (i >= nc) return;
  const int64_t x = cells[4 * i], y = cells[4 * i + 1], z = cells[4 * i + 2];
  const int flag = cells[4 * i + 3];
  const int n = kMc.ntri[flag];
  uint32_t o = toff[i];
  for (int t = 0; t < n; t++) {
    int32_t v[3];
    bool ok = true;
    for (int q = 0; q < 3; q++) {
      int dx, dy, dz, axis;
      edge_geom(kMc.tri[flag][3 * t + q], dx, dy, dz, axis);
      const int64_t key = ((z + dz) * XY + (y + dy) * X + (x + dx)) * 3 + axis;
      const int64_t id = find_key(keys, ne, key);
      if (id < 0) ok = false;
      v[q] = id < 0 ? 0 : (int32_t)id;
    }
    bool degenerate = false;
    if (!ok) {
      atomicAdd(missing, 1u);
    } else {
      // vertex coordinates are read only for triangles whose three edges are listed
      const double eps = 1e-7;
      const double* p0 = verts + 3 * (int64_t)v[0];
      const double* p1 = verts + 3 * (int64_t)v[1];
      const double* p2 = verts + 3 * (int64_t)v[2];
      degenerate = edge_len(p0, p1) < eps || edge_len(p0, p2) < eps || edge_len(p1, p2) < eps;
    }
    tris_pre[3 * (int64_t)o + 0] = v[0];
    tris_pre[3 * (int64_t)o + 1] = v[1];
    tris_pre[3 * (int64_t)o + 2] = v[2];
    keep[o] = (degenerate || !ok) ? 0u : 1u;
    o++;
  }
}

qj_status nlmc_resume(qj_workspace* ws, const MapArgs& a, const qj_rational* f, double iso, int64_t ne,
                      const int32_t* h_edges, int64_t nc, const int32_t* h_cells, int64_t* nv_out, int64_t* nt_out,
                      hipStream_t s) {
  if (!ws->mc) ws->mc = new McState();
  McState& m = *(McState*)ws->mc;
  m.nv = m.nt = 0;
  m.cache_valid = false;
  *nv_out = *nt_out = 0;
  const int64_t X = a.res[0], Y = a.res[1], Z = a.res[2], XY = X * Y;
  if (ne < 0 || nc < 0 || (ne && !h_edges) || (nc && !h_cells) || ne > (int64_t)INT32_MAX ||
      nc > (int64_t)UINT32_MAX / 5) {
    set_error("qj_nlmc_resume: bad edge or cell arrays");
    return QJ_ERR_INVALID;
  }
  // every flag in 1..254 has at least one triangle, so active cells need edges
  if (nc > 0 && ne == 0) {
    set_error("qj_nlmc_resume: %lld active cells but no edges", (long long)nc);
    return QJ_ERR_INVALID;
  }
  // host checks: every edge inside the grid with its far end, keys strictly
  // ascending (the cache's vertex order); every cell inside the grid
  std::vector<int64_t> keys((size_t)ne);
  for (int64_t i = 0; i < ne; i++) {
    const int32_t x = h_edges[4 * i], y = h_edges[4 * i + 1], z = h_edges[4 * i + 2], ax = h_edges[4 * i + 3];
    if (x < 0 || y < 0 || z < 0 || ax < 0 || ax > 2 || x + (ax == 0) >= X || y + (ax == 1) >= Y ||
        z + (ax == 2) >= Z) {
      set_error("qj_nlmc_resume: edge %lld lies outside the grid", (long long)i);
      return QJ_ERR_INVALID;
    }
    keys[i] = ((int64_t)z * XY + (int64_t)y * X + x) * 3 + ax;
    if (i && keys[i] <= keys[i - 1]) {
      set_error("qj_nlmc_resume: edges must be in vertex order (lower endpoint, then axis)");
      return QJ_ERR_INVALID;
    }
  }
  for (int64_t i = 0; i < nc; i++) {
    const int32_t x = h_cells[4 * i], y = h_cells[4 * i + 1], z = h_cells[4 * i + 2], fl = h_cells[4 * i + 3];
    if (x < 0 || y < 0 || z < 0 || x >= X - 1 || y >= Y - 1 || z >= Z - 1 || fl < 1 || fl > 254) {
      set_error("qj_nlmc_resume: cell %lld lies outside the grid or has flag %d", (long long)i, (int)fl);
      return QJ_ERR_INVALID;
    }
  }
  qj_status st;
  if ((st = grow_keep(m.verts, m.cap_v, 3 * ne, 0, s)) || (st = grow_keep(m.c_edges, m.cap_ce, 4 * ne, 0, s)) ||
      (st = grow_keep(m.c_cells, m.cap_cc, 4 * nc, 0, s)) || (st = grow(m.tri_off, m.cap_toff, nc, s)))
    return st;
  if (!m.totals) QJ_HIP(hipMalloc(&m.totals, 4 * sizeof(uint32_t)));
  if (!m.d_bad) QJ_HIP(hipMalloc(&m.d_bad, sizeof(unsigned int)));
  int64_t* d_keys = nullptr;
  unsigned int* d_missing = nullptr;
  QJ_HIP(hipMalloc(&d_keys, sizeof(int64_t) * (size_t)(ne > 0 ? ne : 1)));
  QJ_HIP(hipMalloc(&d_missing, sizeof(unsigned int)));
  struct Free {
    void* a;
    void* b;
    ~Free() {
      (void)hipFree(a);
      (void)hipFree(b);
    }
  } guard{d_keys, d_missing};
  QJ_HIP(hipMemsetAsync(m.d_bad, 0, sizeof(unsigned int), s));
  QJ_HIP(hipMemsetAsync(d_missing, 0, sizeof(unsigned int), s));
  if (ne) {
    QJ_HIP(hipMemcpyAsync(d_keys, keys.data(), sizeof(int64_t) * ne, hipMemcpyHostToDevice, s));
    QJ_HIP(hipMemcpyAsync(m.c_edges, h_edges, sizeof(int32_t) * 4 * ne, hipMemcpyHostToDevice, s));
    launch_cache_vertices(a, dim3(nblocks(ne)), s, f->d64, iso, m.c_edges, ne, m.verts, m.d_bad);
    QJ_HIP(hipGetLastError());
  }
  int64_t nt = 0;
  if (nc) {
    QJ_HIP(hipMemcpyAsync(m.c_cells, h_cells, sizeof(int32_t) * 4 * nc, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_cache_tricount, dim3(nblocks(nc)), dim3(kMcBlock), 0, s, m.c_cells, nc, m.tri_off);
    QJ_HIP(hipGetLastError());
    const size_t need_tmp = scan_tmp_bytes(nc > 4096 ? nc : 4096);
    if (need_tmp > m.tmp_bytes) {
      if (m.tmp) {
        QJ_HIP(hipStreamSynchronize(s));
        QJ_HIP(hipFree(m.tmp));
      }
      m.tmp = nullptr;
      m.tmp_bytes = 0;
      QJ_HIP(hipMalloc(&m.tmp, need_tmp));
      m.tmp_bytes = need_tmp;
    }
    if ((st = scan_u32(m.tri_off, m.tri_off, nc, m.totals + 2, m.tmp, m.tmp_bytes, s))) return st;
    uint32_t h = 0;
    QJ_HIP(hipMemcpyAsync(&h, m.totals + 2, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    QJ_HIP(hipStreamSynchronize(s));
    const int64_t ntp = h;
    if ((st = grow(m.tris_pre, m.cap_tp, 3 * ntp, s)) || (st = grow(m.keep, m.cap_keep, ntp, s)) ||
        (st = grow(m.tris, m.cap_t, 3 * ntp, s)))
      return st;
    if (scan_tmp_bytes(ntp) > m.tmp_bytes) {
      QJ_HIP(hipStreamSynchronize(s));
      QJ_HIP(hipFree(m.tmp));
      m.tmp = nullptr;
      m.tmp_bytes = 0;
      QJ_HIP(hipMalloc(&m.tmp, scan_tmp_bytes(ntp)));
      m.tmp_bytes = scan_tmp_bytes(ntp);
    }
    if (ntp > 0) {
      hipLaunchKernelGGL(k_cache_triangles, dim3(nblocks(nc)), dim3(kMcBlock), 0, s, m.c_cells, nc, X, XY, d_keys,
                         ne, m.verts, m.tri_off, m.tris_pre, m.keep, d_missing);
      QJ_HIP(hipGetLastError());
      if ((st = scan_u32(m.keep, m.keep, ntp, m.totals + 3, m.tmp, m.tmp_bytes, s))) return st;
      QJ_HIP(hipMemcpyAsync(&h, m.totals + 3, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
      QJ_HIP(hipStreamSynchronize(s));
      nt = h;
      if (nt > 0) {
        hipLaunchKernelGGL(k_mc_squeeze, dim3(nblocks(ntp)), dim3(kMcBlock), 0, s, m.tris_pre, m.keep, ntp,
                           m.totals + 3, m.tris);
        QJ_HIP(hipGetLastError());
      }
    }
  }
  unsigned int bad = 0, missing = 0;
  QJ_HIP(hipMemcpyAsync(&bad, m.d_bad, sizeof(bad), hipMemcpyDeviceToHost, s));
  QJ_HIP(hipMemcpyAsync(&missing, d_missing, sizeof(missing), hipMemcpyDeviceToHost, s));
  QJ_HIP(hipStreamSynchronize(s));
  m.nv = ne;
  m.nt = nt;
  m.ncells = nc;
  m.cache_valid = true;
  *nv_out = m.nv;
  *nt_out = m.nt;
  if (missing) {
    set_error("qj_nlmc_resume: %u triangles reference edges the cache does not list", missing);
    return QJ_ERR_INVALID;
  }
  if (bad) {
    set_error("non-linear mesher: %u edges whose end values do not straddle the isosurface "
              "(the reference exits at TRIANGLE_MESH.cpp:2082-2097)", bad);
    return QJ_ERR_NUMERIC;
  }
  return QJ_OK;
}

}  // namespace qj
