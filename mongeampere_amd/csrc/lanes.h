// Groups of 16 lanes: one DPP row of the wave.  All lanes of a group run the
// same control flow (conditions come from ballots or row reductions), so a
// group works together on one cell or one bin; the four groups of a wave are
// independent.
#pragma once

#include <algorithm>

#include "geom_common.h"

namespace ma {

constexpr int kGroup = 16;
constexpr int kCellThreads = 256;                    // threads of the group kernels
constexpr int kCellGroups = kCellThreads / kGroup;   // groups (cells, bins) per workgroup
constexpr int kCellXcdRun = 64;                      // workgroups of an XCD's run (1024 cells)
// Pending nodes of a depth-first pyramid walk that expands a node into its 16
// grandchildren: 15 stay behind at each of the first kMaxLevels / 2 - 1 steps
// and 16 come from the next, 91 at most (the last step reaches bins).
constexpr int kWalkStack = 96;
static_assert((kMaxLevels / 2 - 1) * 15 + 16 <= kWalkStack, "stack of a pyramid walk");

constexpr int kDppShr = 0x110, kDppRor = 0x120, kDppBcast = 0x150;  // row_shr, row_ror, row_newbcast
template <int CTRL>
__device__ inline int dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ inline float dpp(float v) {
  return __int_as_float(dpp<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ inline double dpp(double v) {
  return __hiloint2double(dpp<CTRL>(__double2hiint(v)), dpp<CTRL>(__double2loint(v)));
}
template <class T>
__device__ inline T row_max(T v) {
  v = fmax(v, dpp<kDppRor + 8>(v));
  v = fmax(v, dpp<kDppRor + 4>(v));
  v = fmax(v, dpp<kDppRor + 2>(v));
  return fmax(v, dpp<kDppRor + 1>(v));
}
template <class T>
__device__ inline T row_min(T v) {
  return -row_max(-v);
}
__device__ inline unsigned row_min(unsigned v) {
  v = min(v, (unsigned)dpp<kDppRor + 8>((int)v));
  v = min(v, (unsigned)dpp<kDppRor + 4>((int)v));
  v = min(v, (unsigned)dpp<kDppRor + 2>((int)v));
  return min(v, (unsigned)dpp<kDppRor + 1>((int)v));
}
// largest of non-negative floats (their bit patterns order like integers)
__device__ inline float row_max_nonneg(float f) {
  int v = __float_as_int(f);
  v = max(v, dpp<kDppRor + 8>(v));
  v = max(v, dpp<kDppRor + 4>(v));
  v = max(v, dpp<kDppRor + 2>(v));
  return __int_as_float(max(v, dpp<kDppRor + 1>(v)));
}
template <class T>
__device__ inline T row_sum(T v) {
  v += dpp<kDppRor + 8>(v);
  v += dpp<kDppRor + 4>(v);
  v += dpp<kDppRor + 2>(v);
  return v + dpp<kDppRor + 1>(v);
}
// sum over aligned groups of 8 lanes (quad permutations, then the mirror
// image within 8)
__device__ inline double oct_sum(double v) {
  v += dpp<0xB1>(v);   // quad_perm 1,0,3,2
  v += dpp<0x4E>(v);   // quad_perm 2,3,0,1
  return v + dpp<0x141>(v);  // row_half_mirror
}
// inclusive prefix sum over the row
__device__ inline int row_scan(int v) {
  v += dpp<kDppShr + 1>(v);
  v += dpp<kDppShr + 2>(v);
  v += dpp<kDppShr + 4>(v);
  return v + dpp<kDppShr + 8>(v);
}
// values of lane `src` of the row; base4 = 4 x the row's first lane
__device__ inline int row_get(int v, int base4, int src) {
  return __builtin_amdgcn_ds_bpermute(base4 + 4 * src, v);
}
__device__ inline float row_get(float v, int base4, int src) {
  return __int_as_float(row_get(__float_as_int(v), base4, src));
}
__device__ inline double row_get(double v, int base4, int src) {
  return __hiloint2double(row_get(__double2hiint(v), base4, src),
                          row_get(__double2loint(v), base4, src));
}

// Ranges [lo, lo + cnt) of the group's lanes as one stream: f(q, b, valid) is
// called for 16 consecutive entries at a time, q the entry and b the lane
// whose range holds it; more() stops the stream.
template <class F, class M>
__device__ inline void for_ranges(int base, int l, int32_t lo, int cnt, M &&more, F &&f) {
  const int inc = row_scan(cnt);
  const int ex = inc - cnt, tot = dpp<kDppBcast + 15>(inc);
  for (int s0 = 0; s0 < tot && more(); s0 += kGroup) {
    const int s = s0 + l;
    int b = 0;  // the last lane whose range starts at or before s
#pragma unroll
    for (int step = 8; step > 0; step >>= 1)
      if (row_get(ex, 4 * base, b + step) <= s) b += step;
    const int32_t q = row_get(lo - ex, 4 * base, b) + s;
    f(q, b, s < tot);
  }
}

// ---------------------------------------------------------------------------
// Plane pyramid.  With coordinates about the grid's centre and v_j = |y_j|^2 -
// w_j, pi_j(x) = |x|^2 + v_j - 2 x.y_j.  A node keeps a gradient a and b = min
// over its Diracs of v_j - a.y_j (a lower bound of it above level 0), so that
//   min_j v_j - 2 x.y_j >= b + min over the node's box of (a - 2 x).y.
// Where the weights vary smoothly a is close to 2 x for the points x that the
// node's Diracs own, and the bound is tight to the square of the node's side.
// (The bound of the max-weight pyramid, dist^2(x, node) - max w, is loose by
// four times the distance from a Dirac to its cell times the node's side:
// with clustered Diracs a search for the owners of one bin then met about 500
// Diracs instead of 10.)
// a = 2 (centre of the node) - gw, gw the gradient of the weights by least
// squares over the 16 grandchildren of the node's even-level ancestor.
// ---------------------------------------------------------------------------
struct Plane {
  double ax, ay, b, pad;
};
// Diracs of an even-level node: number, sums of y and w.
struct NodeSums {
  double n, x, y, w;
};
struct NodeBox {
  double x0, y0, x1, y1;
};
__device__ inline NodeBox node_box(const Grid &g, uint32_t m, int lev) {
  const double side = g.h * (double)(1u << lev), half = 0.5 * g.h * (double)g.G;
  NodeBox q;
  q.x0 = compact1by1(m) * side - half;
  q.y0 = compact1by1(m >> 1) * side - half;
  q.x1 = q.x0 + side;
  q.y1 = q.y0 + side;
  return q;
}
// min of t.y over the box; mag gets the magnitude of its terms
__device__ inline double box_min(const NodeBox &q, double tx, double ty, double &mag) {
  const double px = tx > 0.0 ? q.x0 : q.x1, py = ty > 0.0 ? q.y0 : q.y1;
  mag = fabs(tx * px) + fabs(ty * py);
  return tx * px + ty * py;
}
// rounding allowance of a bound: its terms carry errors of a few 1e-16
constexpr double kPlaneEps = 1e-13;

// ---------------------------------------------------------------------------
// Sparse rows and sums of the conjugate gradient.  A row is read by a group
// of kRowLanes consecutive lanes, lane l taking entries l, l + kRowLanes, ...,
// so that a wave reads consecutive entries of consecutive rows.  The kernels
// that leave partial sums run cg_grid(n) workgroups of kCgThreads threads: at
// most all of the chip's wave slots at once, and few enough partial sums that
// every workgroup of the next kernel can add all of them up itself (in the
// same order: the scalars agree everywhere and from run to run).  4096
// workgroups of 256 threads took a launch of their own to fold the sums.
// Several rows of a group at once (2 or 4) made the kernels slower: 150k rows
// 10.2 -> 10.9 -> 14.9 us, 1k rows 4.0 -> 5.4 -> 6.6.
// ---------------------------------------------------------------------------
constexpr int kRowLanes = 8;
constexpr int kCgGrid = 512, kCgThreads = 1024;
constexpr int kCgGroups = kCgThreads / kRowLanes;  // rows of a workgroup at a time
static inline int cg_grid(int64_t n) {
  return (int)std::min<int64_t>(kCgGrid, (n + kCgGroups / 8 - 1) / (kCgGroups / 8));
}
// Workgroup b's share of nb when every XCD takes a run of consecutive ones:
// neighbouring rows, and the same rows in kernel after kernel, meet in one L2.
__device__ inline int64_t xcd_share(int64_t b, int64_t nb) {
  const int64_t x = b % kXcds, q = nb / kXcds, r = nb % kXcds;
  return x * q + min(x, r) + b / kXcds;
}
// the workgroup's rows [first, last) of n
__device__ inline void cg_rows(int64_t n, int64_t &first, int64_t &last) {
  const int64_t nb = gridDim.x, b = xcd_share(blockIdx.x, nb);
  first = n * b / nb;
  last = n * (b + 1) / nb;
}
// A row's first entries, loaded ahead of what decides whether they are needed
// (the done flag, the scalars of the iteration).
template <class T>
struct RowHead {
  int32_t q, e, c;
  T v;
  __device__ inline void load(const int32_t *__restrict__ ptr, const int32_t *__restrict__ col,
                              const T *__restrict__ val, int64_t i, bool valid, int lane) {
    q = e = c = 0;
    v = (T)0;
    if (!valid) return;
    q = ptr[i] + lane;
    e = ptr[i + 1];
    if (q < e) {  // (the matrix may hold no entry at all)
      c = col[q];
      v = val[q];
    }
  }
  // the row times x(j), FP64 accumulation, on every lane of the group
  template <class X>
  __device__ inline double dot(const int32_t *__restrict__ col, const T *__restrict__ val,
                               X &&x) const {
    double s = q < e ? (double)v * x(c) : 0.0;
    for (int32_t k = q + kRowLanes; k < e; k += kRowLanes) s += (double)val[k] * x(col[k]);
    return oct_sum(s);
  }
};
// sums over the workgroup (kCgThreads threads), on every thread; s holds N
// values per wave
template <int N>
__device__ inline void cg_block_sums(double (&v)[N], double *s) {
  constexpr int kWaves = kCgThreads / 64;
#pragma unroll
  for (int k = 0; k < N; k++) {
    v[k] = row_sum(v[k]);
    v[k] += __shfl_xor(v[k], 16);
    v[k] += __shfl_xor(v[k], 32);
    if (threadIdx.x % 64 == 0) s[k * kWaves + threadIdx.x / 64] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = row_sum(s[k * kWaves + threadIdx.x % kWaves]);
  __syncthreads();
}
static_assert(kCgThreads / 64 == kGroup, "one row of lanes adds up the waves");
__device__ inline double cg_block_sum(double v, double *s) {
  double a[1] = {v};
  cg_block_sums(a, s);
  return a[0];
}

}  // namespace ma
