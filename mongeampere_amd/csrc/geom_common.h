// Device helpers shared by the geometry translation units.
#pragma once

#include <cmath>
#include <cstdint>

#include "engine.h"

namespace ma {

constexpr int kBlock = 128;
constexpr double kInf = HUGE_VAL;
// relative tolerance under which a point counts as lying on a triangle edge
constexpr double kSnap = 1e-13;

__host__ __device__ inline uint32_t part1by1(uint32_t x) {
  x &= 0x0000ffffu;
  x = (x | (x << 8)) & 0x00ff00ffu;
  x = (x | (x << 4)) & 0x0f0f0f0fu;
  x = (x | (x << 2)) & 0x33333333u;
  x = (x | (x << 1)) & 0x55555555u;
  return x;
}
__host__ __device__ inline uint32_t compact1by1(uint32_t x) {
  x &= 0x55555555u;
  x = (x | (x >> 1)) & 0x33333333u;
  x = (x | (x >> 2)) & 0x0f0f0f0fu;
  x = (x | (x >> 4)) & 0x00ff00ffu;
  x = (x | (x >> 8)) & 0x0000ffffu;
  return x;
}
__host__ __device__ inline uint32_t morton2(uint32_t x, uint32_t y) {
  return part1by1(x) | (part1by1(y) << 1);
}
__device__ inline int bin_coord(double v, double o, double h, int G) {
  double f = floor((v - o) / h);
  return (f < 0.0) ? 0 : (f > (double)(G - 1) ? G - 1 : (int)f);
}
static inline unsigned nblocks(int64_t n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

// Workgroups are dispatched to the 8 XCDs in turn (workgroup b to XCD b % 8),
// each XCD with its own L2.  Kernels over Morton-ordered work, whose
// neighbouring workgroups read the same Diracs and triangles, renumber their
// workgroups so that every XCD takes runs of kXcdRun consecutive ones (runs
// dealt to the XCDs in turn, so that work that varies over the domain stays
// balanced between them); the blocks past the last whole round keep their
// number.  A bijection of [0, nb).
constexpr int kXcds = 8, kXcdRun = 16;
template <int RUN = kXcdRun>
__device__ inline int64_t xcd_block(int64_t b, int64_t nb) {
  const int64_t full = nb / (kXcds * RUN) * (kXcds * RUN);
  if (b >= full) return b;
  const int64_t x = b % kXcds, i = b / kXcds;
  return ((i / RUN) * kXcds + x) * RUN + i % RUN;
}

// w_k - w_j for weights carried in two words (w = hi + lo, |lo| <= ulp(hi) / 2,
// so that weight differences below the FP64 resolution of the weights still
// move the bisectors).  The difference of the high words is split into its
// FP64 value and its exact rounding error (Knuth's TwoSum); the low words join
// the error term.  lo == nullptr: plain FP64 weights.
__device__ inline double wdiff(const double *lo, double hk, int64_t k, double hj, int64_t j) {
#pragma clang fp contract(off)
  const double s = hk - hj;
  if (!lo) return s;
  const double bb = s - hk;
  const double err = (hk - (s - bb)) + (-hj - bb);
  return s + (err + (lo[k] - lo[j]));
}

__device__ inline void tri_bbox(const TriData &t, double &x0, double &y0, double &x1,
                                double &y1) {
  x0 = fmin(t.x[0], fmin(t.x[1], t.x[2]));
  x1 = fmax(t.x[0], fmax(t.x[1], t.x[2]));
  y0 = fmin(t.y[0], fmin(t.y[1], t.y[2]));
  y1 = fmax(t.y[0], fmax(t.y[1], t.y[2]));
}

// Offsets of the levels of the max-weight pyramid (level 0 = bins).
struct PyrOff {
  int64_t o[16];
};

// Albrecht-Collatz 6-point rule points (include/MA/quadrature.hpp:23-42):
// weights 1/30 for points 0..2, 9/30 for points 3..5, times the area.
template <class R>
struct AC6T {
  R px[6], py[6];
};
using AC6 = AC6T<double>;
template <class R>
__device__ inline void ac6_points(R ax, R ay, R bx, R by, R cx, R cy, AC6T<R> &q) {
  const R ux = bx - ax, uy = by - ay, vx = cx - ax, vy = cy - ay;
  const R h = R(0.5), s6 = R(1.0 / 6.0), t3 = R(2.0 / 3.0);
  q.px[0] = ax + h * ux + h * vx;
  q.py[0] = ay + h * uy + h * vy;
  q.px[1] = ax + h * ux;
  q.py[1] = ay + h * uy;
  q.px[2] = ax + h * vx;
  q.py[2] = ay + h * vy;
  q.px[3] = ax + s6 * ux + t3 * vx;
  q.py[3] = ay + s6 * uy + t3 * vy;
  q.px[4] = ax + s6 * vx + t3 * ux;
  q.py[4] = ay + s6 * vy + t3 * uy;
  q.px[5] = ax + s6 * ux + s6 * vx;
  q.py[5] = ay + s6 * uy + s6 * vy;
}

// Entries of the triangle bins: the triangle, and whether this bin is in the
// first column / row of bins its box meets (tbin entries sort by triangle).
constexpr int kTriShift = 2, kTriFirstX = 1, kTriFirstY = 2;

// Fragment output (FragOut): one record per fragment of positive area.
// frag_reserve: plain atomics, for kernels whose lanes are not converged.
__device__ inline void frag_reserve(const FragOut &o, int m, unsigned long long &f,
                                    unsigned long long &v) {
  f = atomicAdd(&o.count[0], 1ull);
  v = atomicAdd(&o.count[1], (unsigned long long)m);
}
// frag_reserve_block: every thread of a workgroup of 4 waves calls it (m = 0:
// no fragment); one atomic per counter per workgroup, slots in thread order.
// (All workgroups count at the same two addresses, about 8 ns an atomic: with
// one per wave 560k fragments took k_frag<1> 340 us, now 126.)
__device__ inline void frag_reserve_block(const FragOut &o, int m, unsigned long long &f,
                                          unsigned long long &v) {
  __shared__ int nf[4], nv[4];
  __shared__ unsigned long long bf, bv;
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  const int one = m > 0 ? 1 : 0;
  int cf = one, cv = m;  // inclusive prefix sums over the wave
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int tf = __shfl_up(cf, d, 64);
    const int tv = __shfl_up(cv, d, 64);
    if (lane >= d) {
      cf += tf;
      cv += tv;
    }
  }
  if (lane == 63) {
    nf[wave] = cf;
    nv[wave] = cv;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int tf = nf[0] + nf[1] + nf[2] + nf[3], tv = nv[0] + nv[1] + nv[2] + nv[3];
    if (tf > 0) {
      bf = atomicAdd(&o.count[0], (unsigned long long)tf);
      bv = atomicAdd(&o.count[1], (unsigned long long)tv);
    }
  }
  __syncthreads();
  for (int q = 0; q < wave; q++) {
    cf += nf[q];
    cv += nv[q];
  }
  f = bf + (unsigned long long)(cf - one);
  v = bv + (unsigned long long)(cv - m);
}
// Repeated vertices are left out of the output: a vertex within eps of the
// one kept before it, and a last vertex within eps of the first (zero-length
// edges, e.g. where a cell edge and a triangle edge both lie on the domain
// boundary: the two copies of the corner are rounded separately).  The
// polygons of the reference's traversal carry no such repeats, and a repeat
// would bias anything averaged over the vertices.  eps: 1e-12 of the
// fragment's extent (frag_eps).
struct DistinctRun {
  int cnt = 0;
  double eps = 0.0;
  double fx = 0.0, fy = 0.0, lx = 0.0, ly = 0.0;  // first and last kept vertex
  __device__ explicit DistinctRun(double e) : eps(e) {}
  __device__ bool same(double x, double y, double u, double v) const {
    return fabs(x - u) <= eps && fabs(y - v) <= eps;
  }
  // true if (x, y) is kept
  __device__ bool take(double x, double y) {
    if (cnt > 0 && same(x, y, lx, ly)) return false;
    if (cnt == 0) {
      fx = x;
      fy = y;
    }
    lx = x;
    ly = y;
    cnt++;
    return true;
  }
  __device__ int count() const { return (cnt > 1 && same(lx, ly, fx, fy)) ? cnt - 1 : cnt; }
};
__device__ inline double frag_eps(double xlo, double xhi, double ylo, double yhi) {
  return 1e-12 * fmax(xhi - xlo, yhi - ylo);
}
template <class LX, class LY>
__device__ inline double frag_eps_of(int n, LX lx, LY ly) {
  double xlo = INFINITY, xhi = -INFINITY, ylo = INFINITY, yhi = -INFINITY;
  for (int i = 0; i < n; i++) {
    const double x = (double)lx(i), y = (double)ly(i);
    xlo = fmin(xlo, x);
    xhi = fmax(xhi, x);
    ylo = fmin(ylo, y);
    yhi = fmax(yhi, y);
  }
  return frag_eps(xlo, xhi, ylo, yhi);
}
template <class LX, class LY>
__device__ inline int frag_distinct(int n, double eps, LX lx, LY ly) {
  DistinctRun d(eps);
  for (int i = 0; i < n; i++) d.take((double)lx(i), (double)ly(i));
  return d.count();
}
// Writes the record at slots (f, v) if both fit: the m distinct vertices
// (frag_distinct) of the n vertices (lx(i) + ox, ly(i) + oy).
template <class LX, class LY>
__device__ inline void frag_write(const FragOut &o, unsigned long long f, unsigned long long v,
                                  int m, int32_t cell, int32_t tri, double ox, double oy, int n,
                                  double eps, LX lx, LY ly) {
  if (f >= (unsigned long long)o.cap_frag || v + m > (unsigned long long)o.cap_vert) return;
  o.cell[f] = cell;
  o.tri[f] = tri;
  o.nv[f] = m;
  o.start[f] = (int64_t)v;
  DistinctRun d(eps);
  for (int i = 0; i < n; i++) {
    const double x = (double)lx(i), y = (double)ly(i);
    const int at = d.cnt;
    if (d.take(x, y) && at < m) {
      o.xy[2 * (v + at)] = x + ox;
      o.xy[2 * (v + at) + 1] = y + oy;
    }
  }
}

}  // namespace ma
