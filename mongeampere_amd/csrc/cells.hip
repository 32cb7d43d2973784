// Register-resident evaluation kernels:
//   k_cell_local  16 lanes per Dirac: power cell clipped in place, one vertex
//                 per lane (at most kMaxFast), by the Diracs of the
//                 surrounding bins, certified ring by ring or through the
//                 pyramids, written once to HBM;
//   k_pairs       (cell, triangle) pairs whose bounding boxes meet;
//   k_frag        one thread per pair: the cell polygon, in LDS, clipped in
//                 place by the triangle's three edges and integrated exactly
//                 in closed form; fragments that outgrow its slots stream
//                 through three clip stages in registers (k_frag_wide);
//   k_row_count, k_row_fill  Hessian rows from the edge integrals, straight
//                 into the CSR arrays.
// Cells that overflow kMaxFast vertices are flagged and evaluated by the
// general FP64 kernel (k_cells_general).
//
// The geometry kernels are templated on the arithmetic type R.  R = double is
// the FP64 mode.  R = float is the FP32 part of the mixed mode: coordinates
// local to the Dirac are formed in FP64 and rounded once to FP32; clip
// decisions whose FP32 value lies within the FP32 error bound of zero are
// re-decided in FP64 (and counted); fragment masses and cost integrals are
// accumulated with Kahan compensation and added to FP64 totals.
//
// Reference behaviour (paths relative to the MongeAmpere++ tree):
//   strict tie rule, edge labels   include/MA/voronoi_triangulation_intersection.hpp:125-198
//   per-fragment integrals         include/MA/kantorovich.hpp:109-135, include/MA/lloyd.hpp:45-60
//   quadrature                     include/MA/quadrature.hpp:23-42,69-85,122-143
#include <climits>
#include <type_traits>

#include "geom_common.h"
#include "lanes.h"

namespace ma {

constexpr int kNodeDiracs = 8;    // pyramid nodes with at most this many Diracs are taken whole
// Starting box half-width, in bins: wide enough for the large cells of sparse
// regions at converged weights (targets spread over a lognormal range, 1/20 of
// the mean density: such cells span ~10 bins; with 8 the few hundred of them
// sent every evaluation through the per-bin candidate build, a third of its
// time), narrow enough for FP32 local coordinates (errors ~1e-6 of a bin).
// Narrow when the last FP64 evaluation found many cells far from their
// Diracs (clustered Diracs over a spread density): those end on the bin path
// whatever the box, and a wide one only lengthens their search first.
constexpr double kBoxWide = 16.0, kBoxNarrow = 8.0;
// pyramid nodes a cell may visit in the far-cell regime (C4: solve 4.5 -> 3.5 s)
constexpr int kFarWalkBudget = 32;
constexpr int kBoxLabel = -3;     // edge label of that box's cut

// Tolerances per arithmetic type (all relative to the local scale):
//   snap  side of a triangle edge treated as zero (vertex on the edge line);
//   area  fragments below this area are degenerate (zero in exact arithmetic);
//   redo  cell-clip values below this are re-decided in FP64 (FP32 only);
//   pad   relative enlargement of the polygon radius in the pruning test,
//         covering the rounding of the stored vertices.
template <class R>
struct Tol;
template <>
struct Tol<double> {
  static constexpr double snap = 1e-13, area = 1e-13, redo = 0.0, pad = 0.0;
};
template <>
struct Tol<float> {
  // a few float ulps (2^-24 = 6e-8) of the local scale
  static constexpr float snap = 2.5e-7f, area = 5e-7f, redo = 1e-6f;
  static constexpr double pad = 1e-5;
};

struct CellArgs {
  Grid g;
  int64_t n;
  const double *pos, *w;
  const double *wlo;  // low words of two-word weights (nullptr: FP64 weights)
  const int32_t *perm, *rect;
  const int32_t *cand_start, *cand;  // per-bin candidate owners (CSR)
  const int32_t *tbin_start, *tbin_items, *bin_start;
  double dom[4];     // domain bounding box
  const TriData *tri;
  const float4 *tbox;  // FP32 outward-rounded triangle bounding boxes
  double *px, *py;   // FP64 cell vertices (local to the Dirac), [k * kMaxFast + v]
  float *pxf, *pyf;  // FP32 cell vertices (mixed mode)
  int32_t *plab;     // neighbour across edge v -> v+1 (-1: domain edge)
  int32_t *pn;       // vertex count, -1 = handled by the general kernel
  double *bbox;      // absolute bounding box of the cell (4 per Dirac)
  int32_t *tcount;   // candidate triangles per cell
  double *mass, *intg, *mom;  // mom: local first moments, interleaved (x, y)
  double *mom2;      // local second moments (xx, yy, xy) per Dirac (mode 3)
  int32_t *ovf, *novf;  // pairs left to k_frag_wide, and their count
  // edge integrals int rho ds, [k * kMaxFast + v]; -0.0 until an edge is seen
  // (FP64 in both modes: 128 B a cell, so that two cells' atomics do not meet in
  // a line; k_frag<float> at 10.4M pairs 0.60 ms with FP32 sums, 0.50 with these)
  double *eacc;
  const int32_t *triv;  // triangle vertex ids (counter-clockwise, as in tri)
  double *dval;      // adjoint w.r.t. vertex density values (mode 2)
  int32_t *flags;
  unsigned long long *counters;
  int force_general;  // route every cell to the general kernel (testing)
  int walk_budget;    // pyramid nodes a cell may visit before the bin path
  unsigned long long *stripes;  // striped event counters (EvalBuffers::stripes)
  int32_t *ptri;      // first kPadTri candidate triangles of each cell, [k * kPadTri + c]
  FragOut fo;         // fragment polygons (mode 1, when fo.count is set)
  // per Dirac: 1 if its cell took the bin path (far from its Dirac) in the
  // last evaluation of the same Diracs; with use_far such cells go to the
  // bin path at once instead of exhausting the site-centric search first
  unsigned char *far;
  int use_far;
  double box_half;  // half-width of the site-centric starting box (kBoxWide or kBoxNarrow bins)
};

template <class R>
struct CellBuf;
template <>
struct CellBuf<double> {
  __device__ static double *px(const CellArgs &a) { return a.px; }
  __device__ static double *py(const CellArgs &a) { return a.py; }
};
template <>
struct CellBuf<float> {
  __device__ static float *px(const CellArgs &a) { return a.pxf; }
  __device__ static float *py(const CellArgs &a) { return a.pyf; }
};

// ---------------------------------------------------------------------------
// Groups of 16 lanes (one DPP row of the wave) build one cell together: lane
// l holds polygon vertex l in registers, tests one candidate, one bin or one
// pyramid node at a time, and all control flow is uniform in the group.
// Candidates, bins and nodes are loaded 16 at a time, reductions and
// broadcasts are DPP moves, and no LDS limits the waves in flight; what bounds
// k_cell_local is VALU issue (75 - 80 % busy, 61 % of the lanes active).  One
// thread per cell with its polygon in LDS waited instead on dependent gathers
// and its wave's slowest lane (24 % of the lanes active, 1.4 - 1.8 waves per
// SIMD).  Measured, before and now: 1M Diracs at w = 0 in FP32 2.49 and
// 1.80 ms, 1M in FP64 at weights up to 1.6 bins off 8.5 and 3.35 ms, 2M on an
// annulus in FP64 13.0 and 2.94 ms, 1000 Diracs (too few threads before) 278
// and 27 us.
// ---------------------------------------------------------------------------
static_assert(kMaxFast == kGroup, "one polygon vertex per lane");

// a / b: a reciprocal and one correction (within an ulp; not near the ends of
// the range, which the reciprocal does not cover), FP64 as the compiler does it
__device__ inline float ratio(float a, float b) {
  if (!(fabsf(b) > 1e-30f && fabsf(b) < 1e30f)) return a / b;
  const float r = __builtin_amdgcn_rcpf(b), q = a * r;
  return fmaf(fmaf(-b, q, a), r, q);
}
__device__ inline double ratio(double a, double b) { return a / b; }

// The polygon of one group.  Lanes past the last vertex hold vertex 0.
// Half-plane of competitor j seen from Dirac k, in coordinates local to y_k:
// X stays in the cell of k iff kk - 2 X.Y > 0 (strict: ties are outside),
// Y = y_j - y_k, kk = |Y|^2 + w_k - w_j.
template <class R>
struct Cell {
  int l;       // lane in the group
  int base;    // first lane of the group in its wave
  double ih, h2;  // 1 / bin side, its square's inverse
  R x = R(0), y = R(0);  // vertex l
  int lab = -1;          // edge vertex l -> l + 1
  int n = 0;             // vertices (uniform in the group)
  float rb = 0.0f;       // radius of the polygon about the Dirac, squared, in bins (upper bound)
  bool cut = false;      // the starting box cut the domain box
  int nredo = 0;         // FP32 values re-decided in FP64 (this lane)

  __device__ explicit Cell(const Grid &g)
      : l((int)threadIdx.x & (kGroup - 1)), base((int)threadIdx.x & 48), ih(1.0 / g.h),
        h2(g.h * g.h) {}
  // lanes of the group with p set
  __device__ unsigned mask(bool p) const { return (unsigned)(__ballot(p) >> base) & 0xffffu; }
  template <class T>
  __device__ T get(T v, int src) const { return row_get(v, 4 * base, src); }
  __device__ double rho2() const { return (double)rb * h2; }

  __device__ void update_radius() {
    const float xb = (float)(x * (R)ih), yb = (float)(y * (R)ih);
    rb = row_max_nonneg(xb * xb + yb * yb) * (1.0f + 1e-6f + (float)Tol<R>::pad);
  }
  // Box [X0,X1] x [Y0,Y1] (local coordinates) with the labels of its bottom,
  // right, top and left edges, cut to a few bins around the Dirac (edges
  // labelled kBoxLabel): every vertex then stays within a few bins of the
  // Dirac, where FP32 local coordinates are accurate (a vertex on a box edge
  // at distance ~1 would carry an absolute error of ~1e-7, i.e. ~1e-4 of a
  // cell), and the search radius starts bounded.  A finished cell that still
  // touches the cut is handed to the general kernels.  Returns false if
  // nothing is left.
  __device__ bool init(double X0, double Y0, double X1, double Y1, double half) {
    int lb = -1, lr = -1, lt = -1, ll = -1;
    if (X0 < -half) { X0 = -half; ll = kBoxLabel; }
    if (X1 > half) { X1 = half; lr = kBoxLabel; }
    if (Y0 < -half) { Y0 = -half; lb = kBoxLabel; }
    if (Y1 > half) { Y1 = half; lt = kBoxLabel; }
    cut = (lb == kBoxLabel) || (lr == kBoxLabel) || (lt == kBoxLabel) || (ll == kBoxLabel);
    n = 4;
    x = (R)((l == 1 || l == 2) ? X1 : X0);
    y = (R)((l == 2 || l == 3) ? Y1 : Y0);
    lab = l == 1 ? lr : l == 2 ? lt : l == 3 ? ll : lb;
    update_radius();
    return X0 < X1 && Y0 < Y1;
  }
  // true if the finished cell may extend beyond the cut of init(): it still
  // touches the cut, or it came out empty although the box was cut (a cell
  // displaced from its Dirac by more than the box is not seen from inside it)
  __device__ bool touches_cut() const {
    if (n == 0) return cut;
    return mask(l < n && lab == kBoxLabel) != 0u;
  }
  // Clips by the half-plane that lane c brings: (Yx, Yy, kk), edge label
  // `label`.  The surviving vertices form one cyclic run; they move to the
  // front in order, followed by the exit point (label = the new neighbour) and
  // the entry point (label of the edge it lies on).  FP32: a value within
  // lane c's error bound thr of zero is replaced by the FP64 value at the same
  // (stored) point.  Returns whether the polygon changed; sets fail when it
  // outgrows the lanes or rounding breaks the single-run structure.
  __device__ bool clip(int c, double lYx, double lYy, double lkk, int label, float thr,
                       bool &fail) {
    const R Yx = get((R)lYx, c), Yy = get((R)lYy, c), kk = get((R)lkk, c);
    const int nlab = get(label, c);
    R s = kk - R(2) * (x * Yx + y * Yy);
    if (Tol<R>::redo > R(0)) {
      const bool redo = fabs(s) <= (R)get(thr, c);
      if (mask(redo)) {
        const double Y0 = get(lYx, c), Y1 = get(lYy, c), k0 = get(lkk, c);
        if (redo) {
          s = (R)(k0 - 2.0 * ((double)x * Y0 + (double)y * Y1));
          nredo += l < n;
        }
      }
    }
    const unsigned full = (1u << n) - 1u;
    unsigned in = mask(s > R(0)) & full;
    int kept, s0;  // survivors and the first of their run
    auto run = [&]() {
      kept = __popc(in);
      const int out = 32 - __clz((int)(~in & full));  // one past the last vertex cut off
      s0 = (in & 1u) ? (out == n ? 0 : out) : __ffs((int)in) - 1;
      const unsigned t = ((1u << kept) - 1u) << s0;
      return ((t | (t >> n)) & full) == in;
    };
    if (in == full) return false;
    if (in == 0u) {
      n = 0;
      return true;
    }
    bool single = run();
    if (sizeof(R) == sizeof(float) && !single) {
      // FP32 rounding broke the single run: classify every stored vertex in FP64
      const double Y0 = get(lYx, c), Y1 = get(lYy, c), k0 = get(lkk, c);
      in = mask(k0 - 2.0 * ((double)x * Y0 + (double)y * Y1) > 0.0) & full;
      nredo += l < n;
      if (in == full) return false;
      if (in == 0u) {
        n = 0;
        return true;
      }
      single = run();
    }
    if (!single || kept + 2 > kGroup) {
      fail = true;
      return false;
    }
    // slot l takes survivor s0 + l; slot kept the crossing of the edge out of
    // the last survivor, slot kept + 1 that of the edge into the first
    const bool ex = l == kept, en = l == kept + 1;
    int ia = s0 + (l < kept ? l : ex ? kept - 1 : en ? n - 1 : 0);
    int ib = s0 + (ex ? kept : 0);
    ia -= ia >= n ? n : 0;
    ib -= ib >= n ? n : 0;
    const R ax = get(x, ia), ay = get(y, ia), bx = get(x, ib), by = get(y, ib);
    const int al = get(lab, ia);
    R sa, sb;
    if (sizeof(R) == sizeof(float)) {
      sa = get(s, ia);
      sb = get(s, ib);
    } else {
      sa = kk - R(2) * (ax * Yx + ay * Yy);
      sb = kk - R(2) * (bx * Yx + by * Yy);
    }
    const R tt = (ex || en) ? ratio(sa, sa - sb) : R(0);
    x = ax + tt * (bx - ax);
    y = ay + tt * (by - ay);
    lab = ex ? nlab : al;
    n = kept + 2;
    return true;
  }
};

// Clips the polygon C of Dirac k (position (yx, yy), weight wk) by up to 16
// Diracs, lane l bringing Dirac j (-1: none).  A candidate that cannot reach
// the disc about the Dirac holding the polygon is discarded at once (pi_j -
// pi_k >= kk - 2 r |Y|); the others take their half-plane's smallest value
// over the polygon's vertices, and the deepest cut clips first: every clip
// then cuts, and 8.5 of them build a cell of 6 edges (taking the nearest
// bisector first and testing against the disc only: 7.8 clips and 9.4 that
// cut nothing, at 130 instructions each against 30 for the test).  The test
// runs in T: float in units of bins with its rounding bounded (near the
// Dirac), or double (far from it, where that bound would pass everything).
// SEEN: j may be an edge of the polygon already.
template <class T, bool SEEN, class R>
__device__ inline void clip_batch(const CellArgs &a, int64_t k, double yx, double yy, double wk,
                                  int32_t j, Cell<R> &C, bool &fail) {
  bool has = j >= 0 && j != (int32_t)k, hide = false;
  double Yx = 0.0, Yy = 0.0, kk = 1.0, d2 = 1.0;
  if (has) {
    const double2 pj = reinterpret_cast<const double2 *>(a.pos)[j];
    const double wj = a.w[j];
    Yx = pj.x - yx;
    Yy = pj.y - yy;
    d2 = Yx * Yx + Yy * Yy;
    const double dw = wdiff(a.wlo, wk, k, wj, j);  // w_k - w_j
    kk = d2 + dw;
    const double ct = kk - 1e-12 * (d2 + fabs(wk) + fabs(wj));
    if (d2 == 0.0) {
      // coincident Diracs: the larger weight (then the smaller caller index)
      // hides the other
      hide = dw < 0.0 || (dw == 0.0 && a.perm[j] < a.perm[k]);
      has = false;
    } else if (ct > 0.0 && ct * ct > 4.0 * C.rho2() * d2) {
      has = false;
    }
  }
  if (C.mask(hide)) {
    C.n = 0;
    return;
  }
  // the half-plane in T (float: in bins) and the bound of a value's rounding
  const double sc = sizeof(T) == sizeof(float) ? C.ih : 1.0;
  const T Tx = (T)(Yx * sc), Ty = (T)(Yy * sc), Tk = (T)(kk * (sc * sc));
  const float len = fabsf((float)(Yx * C.ih)) + fabsf((float)(Yy * C.ih));
  const float err = 1e-6f * (fabsf((float)(kk * (C.ih * C.ih))) +
                             2.0f * __builtin_amdgcn_sqrtf(C.rb) * len);
  const float thr = err * (float)C.h2;  // for the FP32 polygon's own values
  const float inv = __builtin_amdgcn_rcpf(len);
  // order of the candidates: depth of the cut over |Y|, the lane in the low
  // bits; kNone for those that do not cut
  constexpr unsigned kNone = ~0u;
  auto order = [&]() -> unsigned {
    const T vx = (T)((double)C.x * sc), vy = (T)((double)C.y * sc);
    T m = T(-kInf);
#define MA_VERTEX(v) m = fmax(m, dpp<kDppBcast + v>(vx) * Tx + dpp<kDppBcast + v>(vy) * Ty);
    MA_VERTEX(0) MA_VERTEX(1) MA_VERTEX(2) MA_VERTEX(3) MA_VERTEX(4) MA_VERTEX(5)
    if (C.n > 6) {
      MA_VERTEX(6) MA_VERTEX(7) MA_VERTEX(8)
      if (C.n > 9) {
        MA_VERTEX(9) MA_VERTEX(10) MA_VERTEX(11) MA_VERTEX(12) MA_VERTEX(13) MA_VERTEX(14)
        MA_VERTEX(15)
      }
    }
#undef MA_VERTEX
    const T d = Tk - T(2) * m;
    const bool reach = sizeof(T) == sizeof(float) ? !(d > (T)err) : !(d > T(0));
    const float key = sizeof(T) == sizeof(float) ? (float)d * inv
                                                 : (float)((double)d * (C.ih * C.ih)) * inv;
    const int u = __float_as_int(key);
    const unsigned o = (unsigned)(u ^ ((u >> 31) | (int)0x80000000)) & ~15u;
    return has && reach ? (o | (unsigned)C.l) : kNone;
  };
  if (!C.mask(has)) return;
  bool any = false;
  unsigned key = order();
  while (true) {
    const unsigned best = row_min(key);
    if (best == kNone) break;
    const int c = (int)(best & 15u);
    if (C.l == c) {
      has = false;
      key = kNone;
    }
    if (SEEN) {
      const int cand = C.get((int)j, c);
      if (C.mask(C.l < C.n && C.lab == cand)) continue;
    }
    const bool changed = C.clip(c, Yx, Yy, kk, (int)j, thr, fail);
    if (fail || C.n == 0) return;
    if (changed) {
      any = true;
      key = order();
    }
  }
  if (any) C.update_radius();
}

// Clips by the Diracs of the lanes' ranges (of `list`, or Diracs themselves).
template <class T, bool SEEN, class R>
__device__ inline void clip_ranges(const CellArgs &a, int64_t k, double yx, double yy, double wk,
                                   int32_t lo, int cnt, const int32_t *list, Cell<R> &C,
                                   bool &fail) {
  for_ranges(C.base, C.l, lo, cnt, [&]() { return C.n > 0 && !fail; },
             [&](int32_t q, int, bool valid) {
               const int32_t j = valid ? (list ? list[q] : q) : -1;
               clip_batch<T, SEEN>(a, k, yx, yy, wk, j, C, fail);
             });
}

// The triangles whose bounding box meets [px0,px1]x[py0,py1], once each, by
// the 16 lanes of a group: f(ti, i) for the i-th of them.  A triangle listed
// in several bins is taken in the bin of the lower-left corner of the overlap
// of the two boxes, which its bin entries mark (kTriFirstX, kTriFirstY).
// Returns their number.
template <class F>
__device__ inline int group_triangles(const CellArgs &a, int base, int l, double px0, double py0,
                                      double px1, double py1, F &&f) {
  const Grid &g = a.g;
  // lanes 0..3 locate one side each
  const double side = l == 0 ? px0 : l == 1 ? py0 : l == 2 ? px1 : py1;
  const int bc = bin_coord(side, (l & 1) ? g.y0 : g.x0, g.h, g.G);
  const int qx0 = dpp<kDppBcast + 0>(bc), qy0 = dpp<kDppBcast + 1>(bc);
  const int qx1 = dpp<kDppBcast + 2>(bc), qy1 = dpp<kDppBcast + 3>(bc);
  const int W = qx1 - qx0 + 1, nb = W * (qy1 - qy0 + 1);
  const float invW = 1.0f / (float)W;
  int count = 0;
  for (int t0 = 0; t0 < nb; t0 += kGroup) {
    const int t = t0 + l;
    int ty = (int)((float)t * invW);  // t / W, off by one at most
    ty += (t >= (ty + 1) * W) - (t < ty * W);
    const int by = qy0 + ty, bx = qx0 + t - ty * W;
    int32_t lo = 0;
    int cnt = 0;
    if (t < nb) {
      const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
      lo = a.tbin_start[b];
      cnt = a.tbin_start[b + 1] - lo;
    }
    const int first = (bx == qx0 ? kTriFirstX : 0) | (by == qy0 ? kTriFirstY : 0);
    for_ranges(base, l, lo, cnt, []() { return true; }, [&](int32_t q, int b, bool valid) {
      const int fb = row_get(first, 4 * base, b);
      bool hit = false;
      int32_t ti = 0;
      if (valid) {
        const int32_t it = a.tbin_items[q];
        ti = it >> kTriShift;
        if (((it | fb) & (kTriFirstX | kTriFirstY)) == (kTriFirstX | kTriFirstY)) {
          const float4 tb = a.tbox[ti];
          hit = !((double)tb.z < px0 || (double)tb.x > px1 || (double)tb.w < py0 ||
                  (double)tb.y > py1);
        }
      }
      const unsigned m = (unsigned)(__ballot(hit) >> base) & 0xffffu;
      if (hit) f(ti, count + __popc(m & ((1u << l) - 1u)));
      count += __popc(m);
    });
  }
  return count;
}

// FP32 polygons: the vertices of a finished cell between two neighbours are
// taken again as the crossing of the two bisectors, in FP64, and rounded once
// (the clips' own vertices carry the rounding of the far ends of the edges
// they cut; without this the masses at 1M Diracs are 9.5e-7 off in the 2-norm
// instead of 6.4e-8).  A vertex that moves by more than 1e-3 of a bin (bisectors
// nearly parallel) stays.
__device__ inline void polish(const CellArgs &a, int64_t k, double yx, double yy, double wk,
                              Cell<float> &C) {
  const int l = C.l, n = C.n;
  const int lp = l == 0 ? n - 1 : l - 1;
  const bool own = l < n && C.lab >= 0;
  double Yx = 0.0, Yy = 0.0, kk = 0.0;
  if (own) {
    const double2 pj = reinterpret_cast<const double2 *>(a.pos)[C.lab];
    Yx = pj.x - yx;
    Yy = pj.y - yy;
    kk = Yx * Yx + Yy * Yy + wdiff(a.wlo, wk, k, a.w[C.lab], C.lab);
  }
  const double Px = C.get(Yx, lp & (kGroup - 1)), Py = C.get(Yy, lp & (kGroup - 1));
  const double kp = C.get(kk, lp & (kGroup - 1));
  const double det = Px * Yy - Py * Yx;  // zero without two neighbours
  if (own && det != 0.0) {
    const double s = 0.5 / det;
    const double X = (kp * Yy - kk * Py) * s, Y = (Px * kk - Yx * kp) * s;
    if (fabs(X - (double)C.x) + fabs(Y - (double)C.y) <= 1e-3 * a.g.h) {
      C.x = (float)X;
      C.y = (float)Y;
    }
  }
  const float x0 = C.get(C.x, 0), y0 = C.get(C.y, 0);
  C.x = l < n ? C.x : x0;
  C.y = l < n ? C.y : y0;
}
__device__ inline void polish(const CellArgs &, int64_t, double, double, double, Cell<double> &) {}

// Writes a finished cell: polygon, bounding box, candidate triangles (counted,
// and the first kPadTri kept for k_pairs).
template <class R>
__device__ inline void write_cell(const CellArgs &a, int64_t k, double yx, double yy,
                                  const Cell<R> &C) {
  const int l = C.l, n = C.n;
  if (l == 0) a.pn[k] = n;
  if (n == 0) {
    if (l == 0) a.tcount[k] = 0;
    return;
  }
  if (l < n) {
    const int64_t at = k * kMaxFast + l;
    CellBuf<R>::px(a)[at] = C.x;
    CellBuf<R>::py(a)[at] = C.y;
    a.plab[at] = C.lab;
    a.eacc[at] = -0.0;  // "not seen": any contribution (>= 0) clears the sign
  }
  const double bx0 = (double)row_min(C.x) + yx, by0 = (double)row_min(C.y) + yy;
  const double bx1 = (double)row_max(C.x) + yx, by1 = (double)row_max(C.y) + yy;
  if (l < 4) a.bbox[4 * k + l] = l == 0 ? bx0 : l == 1 ? by0 : l == 2 ? bx1 : by1;
  const int cnt = group_triangles(a, C.base, l, bx0, by0, bx1, by1, [&](int32_t ti, int i) {
    if (i < kPadTri) a.ptri[k * kPadTri + i] = ti;
  });
  if (l == 0) a.tcount[k] = cnt;
}

__device__ inline void zero_cell_outputs(const CellArgs &a, int64_t k) {
  a.mass[k] = 0.0;
  a.intg[k] = 0.0;
  a.mom[2 * k] = 0.0;
  a.mom[2 * k + 1] = 0.0;
  if (a.mom2) {
    a.mom2[3 * k] = 0.0;
    a.mom2[3 * k + 1] = 0.0;
    a.mom2[3 * k + 2] = 0.0;
  }
}

// Lower bound of pi_j - pi_k over the polygon (squared radius rho2 about y_k)
// for every Dirac j at squared distance >= D2 from y_k with weight <= W: the
// polygon is safe from such j when D > rho and D^2 - 2 rho D - (W - w_k) > 0,
// decided on squares (no square roots).
__device__ inline bool far_enough(double D2, double rho2, double W, double wk) {
  const double t = D2 - (W - wk) - 1e-12 * (D2 + fabs(W) + fabs(wk));
  return D2 > rho2 && t > 0.0 && t * t > 4.0 * rho2 * D2;
}

// From ring kWalkFrom on, a cell whose bound needs kWalkAhead more rings and
// more than kWalkWeight radii (2 at equal weights: a wide polygon alone is
// better served by the next ring) walks the pyramid instead.  Cell kernel at 1M
// Diracs displaced by up to 1, 2 and 3 bins: 3.34, 3.64, 3.86 ms, against 3.35,
// 4.63, 5.24 ms after all 8 rings and 3.26, 3.77, 4.06 ms after 4; at w = 0 and
// up to half a bin those who walk early lose (2.57 against 2.16 ms after 4).
constexpr int kWalkFrom = 3;
constexpr float kWalkAhead = 4.0f, kWalkWeight = 2.5f;

// Multi-level certificate for the polygon (squared radius rho2 about y_k) once
// the bins within Chebyshev distance r of the Dirac's bin have been visited.
// At level l the 3 x 3 block of level-l nodes around the Dirac's node contains
// the bins within 2^l of its bin; the Diracs of that block not yet covered
// lie at least as far as the boundary of the covered region (the block one
// level down, or the visited square) and weigh at most the block's maximum
// (pyr3).  Blocks are nested and the top one is the whole grid, so every
// unvisited Dirac is bounded once.  Lane l takes level l.  When some level
// fails, `need` gets the distance (bins) at which its bound would hold.
template <class R>
__device__ inline bool certify_levels(const Grid &g, const double *pyr3, const PyrOff &off, int sbx,
                                      int sby, int r, double yx, double yy, const Cell<R> &C,
                                      double wk, float &need) {
  static_assert(kMaxLevels < kGroup, "one lane per level");
  const int G = g.G, l = C.l;
  const int vx0 = max(sbx - r, 0), vx1 = min(sbx + r, G - 1);
  const int vy0 = max(sby - r, 0), vy1 = min(sby + r, G - 1);
  auto block = [&](int lev, int &x0, int &y0, int &x1, int &y1) {
    const int nx = sbx >> lev, ny = sby >> lev;
    x0 = max((nx - 1) << lev, 0);
    x1 = min(((nx + 2) << lev) - 1, G - 1);
    y0 = max((ny - 1) << lev, 0);
    y1 = min(((ny + 2) << lev) - 1, G - 1);
    return x0 <= vx0 && x1 >= vx1 && y0 <= vy0 && y1 >= vy1;  // holds the visited square
  };
  bool ok = true;
  float dist = 0.0f;
  int bx0, by0, bx1, by1;
  if (l <= g.L && block(l, bx0, by0, bx1, by1)) {
    int x0 = vx0, y0 = vy0, x1 = vx1, y1 = vy1;
    if (l > 0 && block(l - 1, bx0, by0, bx1, by1)) {
      x0 = bx0; y0 = by0; x1 = bx1; y1 = by1;
    }
    double D = kInf;
    if (x0 > 0) D = fmin(D, yx - (g.x0 + x0 * g.h));
    if (x1 < G - 1) D = fmin(D, g.x0 + (x1 + 1) * g.h - yx);
    if (y0 > 0) D = fmin(D, yy - (g.y0 + y0 * g.h));
    if (y1 < G - 1) D = fmin(D, g.y0 + (y1 + 1) * g.h - yy);
    if (D != kInf) {
      const double Wb = pyr3[off.o[l] + morton2((uint32_t)(sbx >> l), (uint32_t)(sby >> l))];
      ok = Wb == -kInf || (D > 0.0 && far_enough(D * D, C.rho2(), Wb, wk));
      if (!ok && r >= kWalkFrom) {
        const float dw = (float)((Wb - wk) * (C.ih * C.ih));
        dist = __builtin_amdgcn_sqrtf(C.rb) + __builtin_amdgcn_sqrtf(fmaxf(C.rb + dw, 0.0f));
      }
    }
  }
  if (C.mask(!ok) == 0u) return true;
  need = r >= kWalkFrom ? row_max_nonneg(dist) : 0.0f;
  return false;
}

// -0.0 exactly (an edge integral no fragment has touched)
__device__ inline bool is_neg_zero(double x) {
  return (unsigned long long)__double_as_longlong(x) == 0x8000000000000000ull;
}

// Counts the lanes of the wave with flag set: one atomic per wave, issued by
// the lowest such lane.
template <class T>
__device__ inline void wave_count(T *dst, bool flag) {
  const unsigned long long bal = __ballot(flag);
  if (bal && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)bal) - 1))
    atomicAdd(dst, (T)__popcll(bal));
}

// Whether some Dirac j of a pyramid node may cut the polygon C of the Dirac at
// (cx, cy) (about the grid's centre): with Y = y_j - y_k in the node's box [x0,
// x0 + side] x [y0, y0 + side] (bins, from the Dirac) and the node's plane,
//   pi_j - pi_k = |Y|^2 + w_k - w_j - 2 X.Y
//               >= b + a.y_k - |y_k|^2 + w_k + (a - 2 y_k - 2 X).Y  at a vertex X,
// in FP32 and bins, with the rounding of its terms allowed for.  One lane tests
// one node against all vertices of its group's polygon.
template <class R>
__device__ inline bool node_reaches(const Plane &p, const Cell<R> &C, double wk, double cx,
                                    double cy, float x0, float y0, float side) {
  const double ih2 = C.ih * C.ih, d = p.ax * cx + p.ay * cy, q = cx * cx + cy * cy;
  const float c0 = (float)((p.b + d - q + wk) * ih2);
  const float gx = (float)((p.ax - 2.0 * cx) * C.ih), gy = (float)((p.ay - 2.0 * cy) * C.ih);
  const float x1 = x0 + side, y1 = y0 + side;
  const float vx = (float)(C.x * (R)C.ih), vy = (float)(C.y * (R)C.ih);
  float m = INFINITY;
#define MA_VERTEX(v)                                                       \
  {                                                                        \
    const float tx = gx - 2.0f * dpp<kDppBcast + v>(vx);                   \
    const float ty = gy - 2.0f * dpp<kDppBcast + v>(vy);                   \
    m = fminf(m, fminf(tx * x0, tx * x1) + fminf(ty * y0, ty * y1));       \
  }
  MA_VERTEX(0) MA_VERTEX(1) MA_VERTEX(2) MA_VERTEX(3) MA_VERTEX(4) MA_VERTEX(5)
  if (C.n > 6) {
    MA_VERTEX(6) MA_VERTEX(7) MA_VERTEX(8)
    if (C.n > 9) {
      MA_VERTEX(9) MA_VERTEX(10) MA_VERTEX(11) MA_VERTEX(12) MA_VERTEX(13) MA_VERTEX(14)
      MA_VERTEX(15)
    }
  }
#undef MA_VERTEX
  const float far = fmaxf(fabsf(x0), fabsf(x1)) + fmaxf(fabsf(y0), fabsf(y1));
  const float err = 2e-6f * (fabsf(c0) + (fabsf(gx) + fabsf(gy) + 2.0f * __builtin_amdgcn_sqrtf(C.rb)) * far) +
                    (float)(1e-14 * (fabs(p.b) + fabs(d) + q + fabs(wk)) * ih2);
  return !(c0 + m > err);
}

// Site-centric construction: the starting box is clipped by the Diracs of the
// bins in Chebyshev rings 0..rmax around the Dirac's own bin (rings 0 and 1
// together).  A lane takes a bin; from ring 2 on a bin whose maximum weight
// and distance cannot reach the polygon is skipped.  After each ring the cell
// is final if every unvisited Dirac is far_enough (certify_levels).  Otherwise
// the remaining Diracs are reached through the pyramids: a depth-first walk
// that tests the 16 grandchildren of a node at once, skips nodes inside the
// visited square, prunes nodes that are far_enough for their own maximum weight
// or whose plane does not reach the polygon (node_reaches) and clips by the
// Diracs of the nodes it keeps.  Pruning uses the polygon at the time of the
// test, which only shrinks, so every pruned Dirac stays unable to cut the final
// cell.
template <class R>
__global__ void __launch_bounds__(kCellThreads) k_cell_local(CellArgs a, const double *pyr,
                                                             const double *pyr3,
                                                             const Plane *__restrict__ planes,
                                                             PyrOff off, int rmax) {
  __shared__ uint32_t stacks[kCellGroups][kWalkStack];
  const int64_t k = xcd_block<kCellXcdRun>(blockIdx.x, gridDim.x) * kCellGroups +
                    threadIdx.x / kGroup;
  if (k >= a.n) return;
  const Grid &g = a.g;
  Cell<R> C(g);
  const int l = C.l;
  const bool lead = l == 0;
  if (lead) zero_cell_outputs(a, k);
  if (a.force_general) {
    if (lead) {
      a.pn[k] = -1;
      a.tcount[k] = 0;
      atomicOr(&a.flags[3], 1);
      if (sizeof(R) == sizeof(double)) a.far[k] = 0;
    }
    return;
  }
  const int lane16 = (int)((k >> 6) & 15);
  if (sizeof(R) == sizeof(double) && a.use_far && a.far[k]) {
    // far from its Dirac at the last weights: the per-bin candidate owners
    // build it exactly (the site-centric search would only run over budget)
    wave_count(&a.stripes[(16 + lane16) * 16], lead);
    if (lead) {
      a.pn[k] = -2;
      a.tcount[k] = 0;
    }
    return;
  }
  const double yx = a.pos[2 * k], yy = a.pos[2 * k + 1], wk = a.w[k];
  bool fail = !C.init(a.dom[0] - yx, a.dom[1] - yy, a.dom[2] - yx, a.dom[3] - yy, a.box_half);
  bool certified = false;
  // squared distance of y_k to the box of nodes [x, x + 2^lev) x [y, y + 2^lev)
  auto dist2 = [&](int x, int y, int lev) {
    const double X0 = g.x0 + x * g.h, X1 = g.x0 + (x + (1 << lev)) * g.h;
    const double Y0 = g.y0 + y * g.h, Y1 = g.y0 + (y + (1 << lev)) * g.h;
    const double dx = fmax(fmax(X0 - yx, yx - X1), 0.0);
    const double dy = fmax(fmax(Y0 - yy, yy - Y1), 0.0);
    return dx * dx + dy * dy;
  };
  const int sbx = bin_coord(yx, g.x0, g.h, g.G), sby = bin_coord(yy, g.y0, g.h, g.G);
  int r = min(rmax, 1);
  for (; r <= rmax && C.n > 0 && !fail; r++) {
    // positions of the ring, counter-clockwise from its lower-left corner
    // (r <= 1: the bins of the 3 x 3 block, or the Dirac's own)
    const int len = r == 0 ? 1 : r == 1 ? 9 : 8 * r;
    for (int p0 = 0; p0 < len && C.n > 0 && !fail; p0 += kGroup) {
      const int p = p0 + l;
      int bx = sbx, by = sby;
      if (r == 1) {
        bx += p % 3 - 1;
        by += p / 3 - 1;
      } else if (r > 1) {
        const int sd = (p >= 2 * r) + (p >= 4 * r) + (p >= 6 * r), o = p - sd * 2 * r;
        bx += sd == 0 ? o - r : sd == 1 ? r : sd == 2 ? r - o : -r;
        by += sd == 0 ? -r : sd == 1 ? o - r : sd == 2 ? r : r - o;
      }
      int32_t lo = 0;
      int cnt = 0;
      if (p < len && bx >= 0 && bx < g.G && by >= 0 && by < g.G) {
        const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
        if (r <= 1 || !far_enough(dist2(bx, by, 0), C.rho2(), pyr[b], wk)) {
          lo = a.bin_start[b];
          cnt = a.bin_start[b + 1] - lo;
        }
      }
      clip_ranges<float, false>(a, k, yx, yy, wk, lo, cnt, nullptr, C, fail);
    }
    if (C.n == 0 || fail) break;
    float need = 0.0f;
    if (certify_levels(g, pyr3, off, sbx, sby, r, yx, yy, C, wk, need)) {
      certified = true;
      break;
    }
    if (need > (float)r + kWalkAhead && need > kWalkWeight * __builtin_amdgcn_sqrtf(C.rb)) {
      r++;  // many more rings, because of the weights: the walk is cheaper
      break;
    }
  }
  const bool walk = !certified && C.n > 0 && !fail;
  bool over_budget = false;
  if (walk) {
    // bins [sbx - rr, sbx + rr] x [sby - rr, sby + rr] have been visited
    const int rr = r - 1;
    const int vx0 = sbx - rr, vx1 = sbx + rr, vy0 = sby - rr, vy1 = sby + rr;
    uint32_t *stack = stacks[threadIdx.x / kGroup];
    int sp = 0, visits = 0;
    uint32_t ent = (uint32_t)g.L << 27;
    // position about the grid's centre, and in bins from its corner
    const double half = 0.5 * g.h * (double)g.G;
    const double cx = yx - g.x0 - half, cy = yy - g.y0 - half;
    const double bx = (yx - g.x0) * C.ih, by = (yy - g.y0) * C.ih;
    while (true) {
      const int lev = (int)(ent >> 27), st = min(lev, 2), cl = lev - st;
      const uint32_t ch = ((ent & ((1u << 27) - 1u)) << (2 * st)) | (uint32_t)l;
      const int nch = 1 << (2 * st);
      visits += nch;
      if (visits > a.walk_budget) {
        // weights with a large spread leave many nodes unprunable: the cell
        // is rebuilt from the per-bin candidate owners instead
        over_budget = true;
        break;
      }
      bool descend = false;
      int32_t lo = 0;
      int cnt = 0;
      const int nx = (int)(compact1by1(ch) << cl), ny = (int)(compact1by1(ch >> 1) << cl);
      const int sd = 1 << cl;
      bool live = l < nch && !(nx >= vx0 && nx + sd - 1 <= vx1 && ny >= vy0 && ny + sd - 1 <= vy1);
      if (live) {
        const double W = pyr[off.o[cl] + ch];
        live = W != -kInf && !far_enough(dist2(nx, ny, cl), C.rho2(), W, wk);
      }
      if (C.mask(live)) {
        const Plane p = live ? planes[off.o[cl] + ch] : Plane{0.0, 0.0, 0.0, 0.0};
        // (every lane of the group takes part: it reads their vertices)
        const bool reaches =
            node_reaches(p, C, wk, cx, cy, (float)(nx - bx), (float)(ny - by), (float)sd);
        if (live && reaches) {
          // the Diracs of a node are one contiguous Morton range: a node
          // holding few of them (sparse regions) is taken whole
          lo = a.bin_start[(int64_t)ch << (2 * cl)];
          cnt = a.bin_start[((int64_t)ch + 1) << (2 * cl)] - lo;
          if (cl > 0 && cnt > kNodeDiracs) {
            descend = true;
            cnt = 0;
          }
        }
      }
      const unsigned dm = C.mask(descend);
      if (descend) stack[sp + __popc(dm & ((1u << l) - 1u))] = ((uint32_t)cl << 27) | ch;
      sp += __popc(dm);
      clip_ranges<float, true>(a, k, yx, yy, wk, lo, cnt, nullptr, C, fail);
      if (sp == 0 || C.n == 0 || fail) break;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the lanes' stack entries
      ent = stack[--sp];
    }
  }
  // a cell still touching the starting box is larger than that box (or lies
  // beyond it): in FP64 it is rebuilt from the per-bin candidate owners, in
  // FP32 by the FP64 kernels
  if (!fail && !over_budget && C.touches_cut()) {
    if (sizeof(R) == sizeof(double))
      over_budget = true;
    else
      fail = true;
  }
  wave_count(&a.stripes[lane16 * 16], lead && walk);  // cells that needed the pyramid walk
  wave_count(&a.stripes[(16 + lane16) * 16], lead && over_budget && !fail);  // left to the bin path
  wave_count(&a.stripes[(32 + lane16) * 16], lead && fail);  // left to the general kernels
  if (Tol<R>::redo > R(0)) {
    const int redo = row_sum(C.nredo);
    if (lead && redo > 0) atomicAdd(&a.counters[5], (unsigned long long)redo);
  }
  if (lead && sizeof(R) == sizeof(double) && !fail) a.far[k] = over_budget ? 1 : 0;
  if (fail || over_budget) {
    if (lead) {
      a.pn[k] = fail ? -1 : -2;
      a.tcount[k] = 0;
      if (fail) atomicOr(&a.flags[3], 1);
    }
    return;
  }
  polish(a, k, yx, yy, wk, C);
  write_cell(a, k, yx, yy, C);
}

// Bin-candidate construction for the cells listed in `list` (those whose
// pyramid walk ran over budget): the bin rectangle of the Dirac is clipped by
// the candidate owners of its bins.  The rectangle covers every bin where the
// Dirac may own a point and the owners of every point of these bins are among
// the candidates, so no certificate is needed.
template <class R>
__global__ void __launch_bounds__(kCellThreads) k_cell_bins(CellArgs a, const int32_t *list,
                                                            const int32_t *nlist) {
  const int64_t idx = blockIdx.x * (int64_t)kCellGroups + threadIdx.x / kGroup;
  if (idx >= *nlist) return;
  const Grid &g = a.g;
  Cell<R> C(g);
  const int l = C.l;
  const bool lead = l == 0;
  const int64_t k = list[idx];
  const int rx0 = a.rect[4 * k], ry0 = a.rect[4 * k + 1], rx1 = a.rect[4 * k + 2],
            ry1 = a.rect[4 * k + 3];
  if (rx0 > rx1) {
    if (lead) {
      a.pn[k] = 0;
      a.tcount[k] = 0;
    }
    return;
  }
  const int W = rx1 - rx0 + 1;
  if ((int64_t)W * (ry1 - ry0 + 1) > kBigRect) {
    // many bins: left to the workgroup-per-cell kernel
    if (lead) {
      a.pn[k] = -1;
      a.tcount[k] = 0;
      atomicOr(&a.flags[3], 1);
    }
    return;
  }
  const int nb = W * (ry1 - ry0 + 1);
  const double yx = a.pos[2 * k], yy = a.pos[2 * k + 1], wk = a.w[k];
  bool fail = !C.init(g.x0 + rx0 * g.h - yx, g.y0 + ry0 * g.h - yy,
                      g.x0 + (rx1 + 1) * g.h - yx, g.y0 + (ry1 + 1) * g.h - yy,
                      sizeof(R) == sizeof(float) ? a.box_half : kInf);  // FP64: the rectangle bounds it
  for (int t0 = 0; t0 < nb && C.n > 0 && !fail; t0 += kGroup) {
    const int t = t0 + l;
    int32_t lo = 0;
    int cnt = 0;
    if (t < nb) {
      const int64_t b = morton2((uint32_t)(rx0 + t % W), (uint32_t)(ry0 + t / W));
      lo = a.cand_start[b];
      cnt = a.cand_start[b + 1] - lo;
    }
    clip_ranges<R, true>(a, k, yx, yy, wk, lo, cnt, a.cand, C, fail);
  }
  if (Tol<R>::redo > R(0)) {
    const int redo = row_sum(C.nredo);
    if (lead && redo > 0) atomicAdd(&a.counters[5], (unsigned long long)redo);
  }
  if (!fail && C.touches_cut()) fail = true;
  if (sizeof(R) == sizeof(double) && !fail) {
    // back within the site-centric search's starting box: the next
    // evaluation tries that search again
    const double half = a.box_half;
    const bool out = l < C.n && !(fabs((double)C.x) < half && fabs((double)C.y) < half);
    const bool any = C.mask(out) != 0u;
    if (lead) a.far[k] = any ? 1 : 0;
  }
  if (fail) {
    if (lead) {
      a.pn[k] = -1;
      a.tcount[k] = 0;
      atomicOr(&a.flags[3], 1);
    }
    return;
  }
  polish(a, k, yx, yy, wk, C);
  write_cell(a, k, yx, yy, C);
}

// Exact owners of the bins.  Candidate entry i (Dirac j listed by bin b) is
// kept only if the part of b (grown by 1e-6 of its side) where j beats every
// other candidate of b has positive area: the grown bin square clipped by the
// power half-planes of those candidates (coordinates local to y_j, strict tie
// rule, the coincident-Dirac rule of clip_batch) is not empty.  The owners of
// every point of b are among its candidates, so the kept Diracs are those
// whose cells meet the grown bin in positive area (entries whose clip
// overflows or breaks on rounding are kept: a superfluous candidate costs
// time, not correctness).  A Dirac's bin rectangle then spans only the bins
// its cell meets, instead of every bin where its power merely comes close to
// one competitor's.
__global__ void __launch_bounds__(kCellThreads) k_cand_refine(CellArgs a, const int32_t *cbin,
                                                              int64_t ncand, int32_t *keep) {
  const int64_t i = xcd_block<kCellXcdRun>(blockIdx.x, gridDim.x) * kCellGroups +
                    threadIdx.x / kGroup;
  if (i >= ncand) return;
  const Grid &g = a.g;
  Cell<double> C(g);
  const int32_t b = cbin[i], j = a.cand[i];
  const double yx = a.pos[2 * j], yy = a.pos[2 * j + 1];
  const uint32_t bx = compact1by1((uint32_t)b), by = compact1by1((uint32_t)b >> 1);
  // the bin grown by a margin: a neighbour across an edge of j's cell that
  // lies on a bin side owns a strip of the grown bin, so the bins of j's
  // rectangle still list every neighbour of j (Hessian entries along bin
  // sides, e.g. on a lattice of exact ties)
  const double eps = 1e-6 * g.h;
  const double x0 = g.x0 + bx * g.h - eps, y0 = g.y0 + by * g.h - eps;
  const double x1 = g.x0 + (bx + 1) * g.h + eps, y1 = g.y0 + (by + 1) * g.h + eps;
  bool fail = !C.init(x0 - yx, y0 - yy, x1 - yx, y1 - yy, kInf);
  const int32_t q0 = a.cand_start[b];
  const int cnt = a.cand_start[b + 1] - q0;
  clip_ranges<double, false>(a, j, yx, yy, a.w[j], q0, C.l == 0 ? cnt : 0, a.cand, C, fail);
  if (C.l == 0) keep[i] = (C.n > 0 || fail) ? 1 : 0;
}

ma_status refine_candidates(ma_engine *e, int64_t total) {
  EvalBuffers &B = e->eb;
  CellArgs a{};
  a.g = e->grid;
  a.pos = e->pos.p;
  a.w = B.w_s.p;
  a.wlo = B.wlo();
  a.perm = e->perm.p;
  a.cand_start = B.cand_cnt.p;
  a.cand = B.cand.p;
  hipLaunchKernelGGL(k_cand_refine, dim3(nblocks(total, kCellGroups)), dim3(kCellThreads), 0,
                     e->stream, a, B.cbin.p, total, B.ckeep.p);
  MA_HIP_TRY(hipGetLastError());
  return MA_OK;
}

// (cell, triangle) pairs: the 16 lanes of a group write the segment of one
// cell, the segments of consecutive cells being consecutive.  Cells with more
// than kPadTri candidates were not kept by the cell kernel; their group scans
// the triangle bins again.  Bound by HBM (8 B written and 4 B read a pair): 1M
// cells, 10.4M pairs 107 us (one thread per cell's count and a search for each
// slot's cell, at 1.2 waves per SIMD: 248 us).
__global__ void __launch_bounds__(kCellThreads) k_pairs(CellArgs a, const int32_t *poff,
                                                        int32_t *pair_cell, int32_t *pair_tri) {
  const int64_t k = xcd_block<kCellXcdRun>(blockIdx.x, gridDim.x) * kCellGroups +
                    threadIdx.x / kGroup;
  if (k >= a.n) return;
  const int l = (int)threadIdx.x & (kGroup - 1), base = (int)threadIdx.x & 48;
  const int cnt = a.tcount[k];
  const int32_t o = poff[k];
  if (cnt <= kPadTri) {
    for (int c = l; c < cnt; c += kGroup) {
      pair_cell[o + c] = (int32_t)k;
      pair_tri[o + c] = a.ptri[k * kPadTri + c];
    }
    return;
  }
  const double *bb = a.bbox + 4 * k;
  group_triangles(a, base, l, bb[0], bb[1], bb[2], bb[3], [&](int32_t ti, int i) {
    pair_cell[o + i] = (int32_t)k;
    pair_tri[o + i] = ti;
  });
}

// ---------------------------------------------------------------------------
// Streaming Sutherland-Hodgman stage: clips by the closed half-plane left of
// a -> b.  Each vertex carries the label of its outgoing edge.
// ---------------------------------------------------------------------------
template <class R>
struct SV {
  R x, y;
  int lab;
};
template <class R>
struct Stage {
  R ax, ay, ex, ey, elen;
  bool started;
  SV<R> first, prev;
  R fs, ps;
  __device__ void init(R x0, R y0, R x1, R y1) {
    ax = x0;
    ay = y0;
    ex = x1 - x0;
    ey = y1 - y0;
    elen = sqrt(ex * ex + ey * ey);
    started = false;
  }
  // Side of v w.r.t. the edge line; values within rounding of zero count as
  // on the line (inside: the triangle is closed), so a cell edge lying on a
  // mesh edge stays with the triangle on the cell's side.
  __device__ R side(const SV<R> &v) const {
    const R dx = v.x - ax, dy = v.y - ay;
    const R s = ex * dy - ey * dx;
    return fabs(s) <= Tol<R>::snap * elen * (fabs(v.x) + fabs(v.y) + fabs(dx) + fabs(dy)) ? R(0)
                                                                                          : s;
  }
  __device__ static SV<R> cross_pt(const SV<R> &p, R sp, const SV<R> &c, R sc, int lab) {
    const R tt = sp / (sp - sc);
    SV<R> r;
    r.x = p.x + tt * (c.x - p.x);
    r.y = p.y + tt * (c.y - p.y);
    r.lab = lab;
    return r;
  }
  // edge p -> c: emits up to two vertices
  __device__ int edge(const SV<R> &p, R sp, const SV<R> &c, R sc, SV<R> &o0, SV<R> &o1) const {
    if (sp >= R(0)) {
      if (sc >= R(0)) {
        o0 = c;
        return 1;
      }
      o0 = cross_pt(p, sp, c, sc, -1);
      return 1;
    }
    if (sc >= R(0)) {
      o0 = cross_pt(p, sp, c, sc, p.lab);
      o1 = c;
      return 2;
    }
    return 0;
  }
  __device__ int push(const SV<R> &c, SV<R> &o0, SV<R> &o1) {
    const R s = side(c);
    if (!started) {
      started = true;
      first = c;
      fs = s;
      prev = c;
      ps = s;
      return 0;
    }
    const int m = edge(prev, ps, c, s, o0, o1);
    prev = c;
    ps = s;
    return m;
  }
  __device__ int flush(SV<R> &o0, SV<R> &o1) const {
    if (!started) return 0;
    return edge(prev, ps, first, fs, o0, o1);
  }
};

// s += v; FP32 sums carry a Kahan compensation c (the true sum is s - c).
template <class R>
__device__ inline void acc_add(R &s, R &c, R v) {
  if (sizeof(R) == sizeof(float)) {
    const R y = v - c;
    const R t = s + y;
    c = (t - s) - y;
    s = t;
  } else {
    s += v;
  }
}

// Integrals over a fragment, as a fan of triangles (coordinates local to the
// Dirac).  MODE 0: mass and int rho |x - y|^2; MODE 1: mass and first moments;
// MODE 2: MODE 1 plus, per triangle vertex v, the integral of (|x - y_k|^2 -
// w_k) phi_v(x) over the fragment (phi_v: P1 hat function of v, linear on the
// triangle), the derivative of the dual value w.r.t. the density value at v;
// MODE 3: MODE 1 plus the second moments.  The integrands are products of
// functions linear on the fan triangle, whose integrals are closed forms in
// the vertex values: with A the area, S the sum of the vertices p_k and R that
// of the density values r_k there, int rho = A R / 3, int rho x = A/12 (R S +
// sum r_k p_k), int rho x x^T = A/60 (R (S S^T + sum p_k p_k^T) + W S^T + S W^T
// + 2 sum r_k p_k p_k^T), W = sum r_k p_k.  (Exact as the 6-point rule of the
// reference is, at a third of its instructions.)
template <int MODE, class R>
struct Quad {
  R area, mass, intg, mx, my;
  R sxx, syy, sxy;    // second moments (MODE 3)
  R cmass, cintg;     // Kahan compensations (FP32)
  // rho(Dirac + X) = r0 + ga (X - tx) + gb (Y - ty): the linear density
  // anchored at the triangle's first vertex (tx, ty), so that its values
  // inside the triangle carry no cancellation from extrapolating to the Dirac
  R r0, ga, gb, tx, ty;
  double wk;          // weight of the Dirac (MODE 2)
  double la[3], lb[3], lc[3];  // barycentric coordinates la X + lb Y + lc (MODE 2)
  double dv[3];
  // extent of the fragment, for the degeneracy test
  R xlo, xhi, ylo, yhi, cmax;

  struct V {
    R x, y, r, n;  // density and |x|^2 there
  };
  __device__ R rho(R x, R y) const { return r0 + ga * (x - tx) + gb * (y - ty); }
  __device__ V vertex(R x, R y) const { return {x, y, rho(x, y), x * x + y * y}; }
  __device__ void extend(const V &v) {
    xlo = fmin(xlo, v.x);
    xhi = fmax(xhi, v.x);
    ylo = fmin(ylo, v.y);
    yhi = fmax(yhi, v.y);
    cmax = fmax(cmax, fmax(fabs(v.x), fabs(v.y)));
  }
  // A fragment counts only if its area is positive: the reference clips the
  // closed triangle by the open cell (ties excluded), so a cell touching a
  // triangle only along an edge or at a point yields nothing.  Exactly
  // degenerate fragments come out with areas at rounding level, hence the
  // scale-aware threshold.
  __device__ bool positive() const {
    return area > Tol<R>::area * ((xhi - xlo) + (yhi - ylo)) * cmax;
  }
  // int rho ds along the edge a -> b
  __device__ R edge(R ax, R ay, R ra, R bx, R by, R rb) const {
    const R ex = bx - ax, ey = by - ay;
    return sqrt(ex * ex + ey * ey) * (R(0.5) * (ra + rb));
  }
  __device__ void fan(const V &a, const V &b, const V &c) {
    const R ar = R(0.5) * ((b.x - a.x) * (c.y - a.y) - (c.x - a.x) * (b.y - a.y));
    const R Rs = a.r + b.r + c.r, Sx = a.x + b.x + c.x, Sy = a.y + b.y + c.y;
    const R Wx = a.r * a.x + b.r * b.x + c.r * c.x, Wy = a.r * a.y + b.r * b.y + c.r * c.y;
    area += ar;
    acc_add(mass, cmass, ar * (Rs * R(1.0 / 3.0)));
    if (MODE == 0) {
      const R q = Rs * (Sx * Sx + Sy * Sy + (a.n + b.n + c.n)) +
                  R(2) * (Wx * Sx + Wy * Sy + (a.r * a.n + b.r * b.n + c.r * c.n));
      acc_add(intg, cintg, ar * (q * R(1.0 / 60.0)));
    } else {
      mx += ar * (R(1.0 / 12.0) * (Rs * Sx + Wx));
      my += ar * (R(1.0 / 12.0) * (Rs * Sy + Wy));
    }
    if (MODE == 3) {
      const R xx = a.x * a.x + b.x * b.x + c.x * c.x, yy = a.y * a.y + b.y * b.y + c.y * c.y;
      const R xy = a.x * a.y + b.x * b.y + c.x * c.y;
      const R rxx = a.r * a.x * a.x + b.r * b.x * b.x + c.r * c.x * c.x;
      const R ryy = a.r * a.y * a.y + b.r * b.y * b.y + c.r * c.y * c.y;
      const R rxy = a.r * a.x * a.y + b.r * b.x * b.y + c.r * c.x * c.y;
      const R f = ar * R(1.0 / 60.0);
      sxx += f * (Rs * (Sx * Sx + xx) + R(2) * (Wx * Sx + rxx));
      syy += f * (Rs * (Sy * Sy + yy) + R(2) * (Wy * Sy + ryy));
      sxy += f * (Rs * (Sx * Sy + xy) + Wx * Sy + Wy * Sx + R(2) * rxy);
    }
    if (MODE == 2) {
      const double N = a.n + b.n + c.n, S2 = Sx * Sx + Sy * Sy;
#pragma unroll
      for (int v = 0; v < 3; v++) {
        const double fa = la[v] * a.x + lb[v] * a.y + lc[v], fb = la[v] * b.x + lb[v] * b.y + lc[v];
        const double fc = la[v] * c.x + lb[v] * c.y + lc[v], F = fa + fb + fc;
        const double Fx = fa * a.x + fb * b.x + fc * c.x, Fy = fa * a.y + fb * b.y + fc * c.y;
        const double Fn = fa * a.n + fb * b.n + fc * c.n;
        dv[v] += ar * ((1.0 / 60.0) * (F * (S2 + N) + 2.0 * (Fx * Sx + Fy * Sy + Fn)) -
                       (1.0 / 3.0) * wk * F);
      }
    }
  }
};

// Streaming integration for k_frag_wide: fragment vertices arrive in order.
template <int MODE, class R>
struct Integrator : Quad<MODE, R> {
  using Base = Quad<MODE, R>;
  using V = typename Base::V;
  int cnt;
  V first, prev;
  int first_lab, prev_lab;
  // Edge integrals are buffered until the area is known (named registers
  // rather than arrays, so nothing spills to scratch).
  int nb;
  int bl0, bl1, bl2, bl3;
  R bv0, bv1, bv2, bv3;
  double *eacc;
  int64_t k;
  __device__ void commit(int lab, R r) { atomicAdd(&eacc[k * kMaxFast + lab], (double)r); }
  __device__ void edge(const V &a, int lab, const V &b) {
    if (MODE != 0 || lab < 0) return;
    if (b.x == a.x && b.y == a.y) return;  // zero-length piece from a snapped vertex
    const R r = Base::edge(a.x, a.y, a.r, b.x, b.y, b.r);
    if (nb == 0) {
      bl0 = lab;
      bv0 = r;
    } else if (nb == 1) {
      bl1 = lab;
      bv1 = r;
    } else if (nb == 2) {
      bl2 = lab;
      bv2 = r;
    } else if (nb == 3) {
      bl3 = lab;
      bv3 = r;
    } else {
      // a degenerate fragment has at most one cell edge of positive length
      // (plus zero-length edges at tie vertices): five or more means a
      // genuine fragment
      commit(lab, r);
    }
    nb++;
  }
  __device__ void push(const SV<R> &v) {
    const V c = Base::vertex(v.x, v.y);
    Base::extend(c);
    if (cnt == 0) {
      first = c;
      first_lab = v.lab;
    } else {
      edge(prev, prev_lab, c);
      if (cnt >= 2) Base::fan(first, prev, c);
    }
    prev = c;
    prev_lab = v.lab;
    cnt++;
  }
  __device__ void finish() {
    if (cnt >= 2) edge(prev, prev_lab, first);
    if (Base::positive()) {
      if (nb > 0) commit(bl0, bv0);
      if (nb > 1) commit(bl1, bv1);
      if (nb > 2) commit(bl2, bv2);
      if (nb > 3) commit(bl3, bv3);
    }
  }
};

// Corners of triangle t in coordinates local to Dirac k (formed in FP64, then
// rounded once) and the quadrature of the pair.
template <class R>
struct LocalTri {
  R x[3], y[3];
};
template <int MODE, class R>
__device__ inline void quad_setup(const CellArgs &a, int64_t k, const TriData &t, LocalTri<R> &T,
                                  Quad<MODE, R> &I) {
  const double yx = a.pos[2 * k], yy = a.pos[2 * k + 1];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    T.x[c] = (R)(t.x[c] - yx);
    T.y[c] = (R)(t.y[c] - yy);
  }
  I.area = I.mass = I.intg = I.mx = I.my = R(0);
  I.sxx = I.syy = I.sxy = R(0);
  I.cmass = I.cintg = R(0);
  I.r0 = (R)(t.a * t.x[0] + t.b * t.y[0] + t.c);  // the value at vertex 0
  I.ga = (R)t.a;
  I.gb = (R)t.b;
  I.tx = T.x[0];
  I.ty = T.y[0];
  I.xlo = I.ylo = R(kInf);
  I.xhi = I.yhi = R(-kInf);
  I.cmax = R(0);
  if (MODE == 2) {
    // barycentric coordinates of the triangle in coordinates local to the Dirac
    const double X0 = t.x[0] - yx, Y0 = t.y[0] - yy, X1 = t.x[1] - yx, Y1 = t.y[1] - yy;
    const double X2 = t.x[2] - yx, Y2 = t.y[2] - yy;
    const double inv = 1.0 / ((X1 - X0) * (Y2 - Y0) - (X2 - X0) * (Y1 - Y0));
    I.la[0] = (Y1 - Y2) * inv; I.lb[0] = (X2 - X1) * inv; I.lc[0] = (X1 * Y2 - X2 * Y1) * inv;
    I.la[1] = (Y2 - Y0) * inv; I.lb[1] = (X0 - X2) * inv; I.lc[1] = (X2 * Y0 - X0 * Y2) * inv;
    I.la[2] = (Y0 - Y1) * inv; I.lb[2] = (X1 - X0) * inv; I.lc[2] = (X0 * Y1 - X1 * Y0) * inv;
    I.wk = a.w[k];
    I.dv[0] = I.dv[1] = I.dv[2] = 0.0;
  }
}
// Sets up the three clip stages (one per triangle edge) and the integrator of
// pair (cell k, triangle t) for k_frag_wide.
template <int MODE, class R>
__device__ inline void frag_setup(const CellArgs &a, int64_t k, const TriData &t, Stage<R> &s1,
                                  Stage<R> &s2, Stage<R> &s3, Integrator<MODE, R> &I) {
  LocalTri<R> T;
  quad_setup<MODE, R>(a, k, t, T, I);
  s1.init(T.x[0], T.y[0], T.x[1], T.y[1]);
  s2.init(T.x[1], T.y[1], T.x[2], T.y[2]);
  s3.init(T.x[2], T.y[2], T.x[0], T.y[0]);
  I.cnt = 0;
  I.nb = 0;
  I.eacc = a.eacc;
  I.k = k;
}

// Vertex v of the cell polygon of k (label: v, or -1 on a domain edge) from
// the evaluation's polygon arrays.
template <class R>
struct PolyGlobal {
  const CellArgs &a;
  int64_t k;
  __device__ void operator()(int v, SV<R> &c) const {
    const int64_t at = k * kMaxFast + v;
    c.x = CellBuf<R>::px(a)[at];
    c.y = CellBuf<R>::py(a)[at];
    c.lab = (a.plab[at] >= 0) ? v : -1;
  }
};

// Streams the n-vertex cell polygon of k through the three clip stages;
// src(v, c) fetches vertex v, sink(v) receives the fragment's vertices in
// order.
template <class R, class Src, class Sink>
__device__ inline void frag_clip(const Src &src, int n, Stage<R> &s1, Stage<R> &s2, Stage<R> &s3,
                                 Sink &&sink) {
  SV<R> o0, o1, q0, q1, r0, r1;
  auto to3 = [&](const SV<R> &v) {
    const int m3 = s3.push(v, r0, r1);
    if (m3 > 0) sink(r0);
    if (m3 > 1) sink(r1);
  };
  auto to2 = [&](const SV<R> &v) {
    const int m2 = s2.push(v, q0, q1);
    if (m2 > 0) to3(q0);
    if (m2 > 1) to3(q1);
  };
  for (int v = 0; v < n; v++) {
    SV<R> c;
    src(v, c);
    const int m1 = s1.push(c, o0, o1);
    if (m1 > 0) to2(o0);
    if (m1 > 1) to2(o1);
  }
  const int m1 = s1.flush(o0, o1);
  if (m1 > 0) to2(o0);
  if (m1 > 1) to2(o1);
  const int m2 = s2.flush(q0, q1);
  if (m2 > 0) to3(q0);
  if (m2 > 1) to3(q1);
  const int m3 = s3.flush(r0, r1);
  if (m3 > 0) sink(r0);
  if (m3 > 1) sink(r1);
}

// Vertices per thread that k_frag's LDS holds (FP32 / FP64): cells and
// fragments with more go to k_frag_wide.  12 is what the label word holds; in
// FP64 10 keep four workgroups on a compute unit (1M Diracs: 0.78 ms with
// k_frag_wide, 0.86 with 12, 1.04 with 9).
template <class R>
struct FragCap {
  static constexpr int value = sizeof(R) == sizeof(float) ? 12 : 10;
};
// The polygon of one thread of k_frag: vertex slots in LDS (a column per
// thread), their order packed in a word of 4 bits a vertex and the labels of
// the edges leaving them (the cell edge's index, kNoLabel on a triangle or
// domain edge) in one of 5 bits.  A clip rotates the two words and moves no
// vertex; the slots past the last vertex of the order word are free.
constexpr int kNoLabel = 31;
template <class R>
struct FragPoly {
  R *px, *py;  // this thread's column, 256 apart
  uint64_t order, labels;
  int m;

  __device__ int slot(int i) const { return (int)(order >> (4 * i)) & 15; }
  __device__ int label(int i) const { return (int)(labels >> (5 * i)) & 31; }
  __device__ R x(int i) const { return px[slot(i) * 256]; }
  __device__ R y(int i) const { return py[slot(i) * 256]; }
  // Clip by the closed half-plane left of (ax, ay) -> (bx, by).  Side values
  // within rounding of zero count as on the line (inside: the triangle is
  // closed), so a cell edge lying on a mesh edge stays with the triangle on
  // the cell's side.  Returns false when the polygon outgrows its slots or
  // rounding breaks the single run of vertices inside.
  __device__ bool clip(R ax, R ay, R bx, R by) {
    const R ex = bx - ax, ey = by - ay;
    const R tol = Tol<R>::snap * sqrt(ex * ex + ey * ey);
    auto side = [&](R vx, R vy) -> R {
      const R dx = vx - ax, dy = vy - ay;
      const R v = ex * dy - ey * dx;
      return fabs(v) <= tol * (fabs(vx) + fabs(vy) + fabs(dx) + fabs(dy)) ? R(0) : v;
    };
    unsigned in = 0u;
    for (int i = 0; i < m; i++) in |= (side(x(i), y(i)) >= R(0) ? 1u : 0u) << i;
    const unsigned full = (1u << m) - 1u;
    if (in == full) return true;
    if (in == 0u) {
      m = 0;
      return true;
    }
    const int kept = __popc(in), out = 32 - __clz((int)(~in & full));
    const int s0 = (in & 1u) ? (out == m ? 0 : out) : __ffs((int)in) - 1;
    const unsigned run = ((1u << kept) - 1u) << s0;
    if (((run | (run >> m)) & full) != in || kept + 2 > FragCap<R>::value) return false;
    // the run first, then the vertices cut off, then the free slots
    const uint64_t om = (1ull << (4 * m)) - 1ull, lm = (1ull << (5 * m)) - 1ull;
    const uint64_t lo = order & om, ll = labels & lm;
    order = (order & ~om) | (((lo >> (4 * s0)) | (lo << (4 * (m - s0)))) & om);
    labels = ((ll >> (5 * s0)) | (ll << (5 * (m - s0)))) & lm;
    // edge kept - 1 -> kept leaves, edge m - 1 -> 0 comes back
    const R ux = x(kept - 1), uy = y(kept - 1), vx = x(kept), vy = y(kept);
    const R wx = x(m - 1), wy = y(m - 1), zx = x(0), zy = y(0);
    const R su = side(ux, uy), sv = side(vx, vy), sw = side(wx, wy), sz = side(zx, zy);
    const R t0 = ratio(su, su - sv), t1 = ratio(sw, sw - sz);
    const int el = label(m - 1), s1 = slot(kept), s2 = slot(kept + 1);
    px[s1 * 256] = ux + t0 * (vx - ux);
    py[s1 * 256] = uy + t0 * (vy - uy);
    px[s2 * 256] = wx + t1 * (zx - wx);
    py[s2 * 256] = wy + t1 * (zy - wy);
    const int at = 5 * kept;
    labels = (labels & ((1ull << at) - 1ull)) |
             ((uint64_t)(unsigned)(kNoLabel | (el << 5)) << at);
    m = kept + 2;
    return true;
  }
};

// One thread per pair: the cell polygon, in LDS, clipped by the triangle's
// three edges, then integrated in one loop over the fragment.  Every lane runs
// the same sequence (classify, two crossings, rotate), so the wave is bound by
// its longest polygon only; a pipeline that streamed the vertices through the
// three edges took a different branch on every lane (26 % of the lanes active
// per instruction, 3700 VALU instructions a wave against 2100 and 47 % here).
// VALU issue bounds it (75 - 84 % busy).  At 10.4M pairs, before and after:
// FP64 1.38 and 0.68 ms, FP32 0.86 and 0.48 ms (0.70 while every workgroup
// counted its fragments at one address).
template <int MODE, class R>
__global__ void __launch_bounds__(256) k_frag(CellArgs a, int64_t npairs,
                                              const int32_t *__restrict__ pair_cell,
                                              const int32_t *__restrict__ pair_tri) {
  // every thread stays to the end (block-level sums below); threads past
  // the last pair take the last pair with an empty polygon (nothing)
  const int64_t p0 = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool valid = p0 < npairs;
  const int64_t p = valid ? p0 : npairs - 1;
  const int64_t k = pair_cell[p];
  const TriData t = a.tri[pair_tri[p]];
  const int n = valid ? a.pn[k] : 0;
  Quad<MODE, R> I;
  LocalTri<R> T;
  quad_setup<MODE, R>(a, k, t, T, I);
  // the same LDS holds the per-cell sums at the end
  constexpr int kCap = FragCap<R>::value;
  constexpr int kStageBytes = kCap * 256 * 2 * (int)sizeof(R);
  constexpr int kRedBytes = 256 * 4 + 6 * 256 * 8 + 16;
  __shared__ __align__(16) unsigned char lds[kStageBytes > kRedBytes ? kStageBytes : kRedBytes];
  const int tt = (int)threadIdx.x;
  FragPoly<R> F;
  F.px = reinterpret_cast<R *>(lds) + tt;
  F.py = F.px + kCap * 256;
  F.order = 0xFEDCBA9876543210ull;
  F.labels = 0ull;
  F.m = min(n, kCap);
  for (int i = 0; i < F.m; i++) {
    const int64_t at = k * kMaxFast + i;
    F.px[i * 256] = CellBuf<R>::px(a)[at];
    F.py[i * 256] = CellBuf<R>::py(a)[at];
    F.labels |= (uint64_t)(a.plab[at] >= 0 ? i : kNoLabel) << (5 * i);
  }
  bool wide = n > kCap;
  if (wide) F.m = 0;
#pragma unroll 1
  for (int c = 0; c < 3; c++) {
    const int d = c == 2 ? 0 : c + 1;
    const R ax = c == 0 ? T.x[0] : c == 1 ? T.x[1] : T.x[2];
    const R ay = c == 0 ? T.y[0] : c == 1 ? T.y[1] : T.y[2];
    const R bx = d == 0 ? T.x[0] : d == 1 ? T.x[1] : T.x[2];
    const R by = d == 0 ? T.y[0] : d == 1 ? T.y[1] : T.y[2];
    if (F.m > 0 && !F.clip(ax, ay, bx, by)) {
      wide = true;
      F.m = 0;
    }
  }
  const int nout = F.m;
  if (wide) a.ovf[atomicAdd(a.novf, 1)] = (int32_t)p;
  if (nout > 0) {
    using V = typename Quad<MODE, R>::V;
    const V first = I.vertex(F.x(0), F.y(0));
    I.extend(first);
    V prev = first;
    for (int i = 1; i < nout; i++) {
      const V v = I.vertex(F.x(i), F.y(i));
      I.extend(v);
      if (i > 1) I.fan(first, prev, v);
      prev = v;
    }
  }
  const bool counted = valid && nout >= 3 && I.positive();
  if (MODE == 0 && counted) {
    // Hessian edge integrals (include/MA/kantorovich.hpp:109-122)
    double *eacc = a.eacc + k * kMaxFast;
    for (int i = 0; i < nout; i++) {
      const int lab = F.label(i);
      if (lab == kNoLabel) continue;
      const int i1 = i + 1 == nout ? 0 : i + 1;
      const R ax = F.x(i), ay = F.y(i), bx = F.x(i1), by = F.y(i1);
      if (ax == bx && ay == by) continue;  // zero-length piece from a snapped vertex
      atomicAdd(&eacc[lab], (double)I.edge(ax, ay, I.rho(ax, ay), bx, by, I.rho(bx, by)));
    }
  }
  if (MODE == 1 && a.fo.count != nullptr) {
    // fragment polygons from the staging (every thread takes part)
    auto gx = [&](int i) { return F.x(i); };
    auto gy = [&](int i) { return F.y(i); };
    const double eps = frag_eps(I.xlo, I.xhi, I.ylo, I.yhi);
    const int m = counted ? frag_distinct(nout, eps, gx, gy) : 0;
    unsigned long long f, v;
    frag_reserve_block(a.fo, m, f, v);
    if (m > 0)
      frag_write(a.fo, f, v, m, a.perm[k], pair_tri[p], a.pos[2 * k], a.pos[2 * k + 1], nout,
                 eps, gx, gy);
  }
  if (counted && MODE == 2) {
    const int64_t ti = pair_tri[p];
#pragma unroll
    for (int v = 0; v < 3; v++) atomicAdd(&a.dval[a.triv[3 * ti + v]], I.dv[v]);
  }
  // Per-cell sums: pairs come sorted by cell, so the threads of a block
  // holding the same cell are contiguous.  Each thread's contributions go to
  // LDS; the last thread of each run sums its run and issues one atomic per
  // quantity (instead of one per fragment).  Every thread reaches the
  // barriers (no early return above).
  constexpr int kQ = MODE == 0 ? 2 : MODE == 3 ? 6 : 3;
  __syncthreads();  // every thread is done with its staged vertices
  int *skey = reinterpret_cast<int *>(lds);
  double (*sval)[256] = reinterpret_cast<double (*)[256]>(lds + 256 * 4);
  {
    double q[kQ];
    if (MODE == 0) {
      q[0] = (double)I.mass - (double)I.cmass;
      q[1] = (double)I.intg - (double)I.cintg;
    } else {
      q[0] = (double)I.mass;
      q[1] = (double)I.mx;
      q[2] = (double)I.my;
      if (MODE == 3) {
        q[3 % kQ] = (double)I.sxx;
        q[4 % kQ] = (double)I.syy;
        q[5 % kQ] = (double)I.sxy;
      }
    }
    const int t = (int)threadIdx.x;
    skey[t] = counted ? (int)k : (valid ? -2 - (int)(k & 0x3fffffff) : -1);
#pragma unroll
    for (int c = 0; c < kQ; c++) sval[c][t] = counted ? q[c] : 0.0;
    // fragment count: per wave into LDS, one global atomic per block (a
    // same-address atomic per wave serialises across the whole grid)
    int *wcnt = reinterpret_cast<int *>(lds + 256 * 4 + 6 * 256 * 8);
    const unsigned long long bal = __ballot(counted);
    if ((t & 63) == 0) wcnt[t >> 6] = __popcll(bal);
    __syncthreads();
    if (t == 0) {
      const int c4 = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
      if (c4) atomicAdd(counter_stripe(a.counters, 0, blockIdx.x), (unsigned long long)c4);
    }
    // runs are keyed by cell; uncounted fragments keep their cell's run
    // boundaries (key -2 - k) but contribute nothing
    const int mykey = valid ? (int)k : -1;
    auto cell_of = [&](int j) {
      const int kk = skey[j];
      return kk >= 0 ? kk : (kk == -1 ? -1 : -2 - kk);
    };
    const bool last = t == 255 || cell_of(t + 1) != mykey;
    if (valid && last) {
      double acc[kQ];
#pragma unroll
      for (int c = 0; c < kQ; c++) acc[c] = 0.0;
      bool any = false;
      for (int j = t; j >= 0 && cell_of(j) == mykey; j--) {
        any |= skey[j] >= 0;
#pragma unroll
        for (int c = 0; c < kQ; c++) acc[c] += sval[c][j];
      }
      if (any) {
        if (MODE == 0) {
          atomicAdd(&a.mass[k], acc[0]);
          atomicAdd(&a.intg[k], acc[1]);
        } else {
          atomicAdd(&a.mass[k], acc[0]);
          atomicAdd(&a.mom[2 * k], acc[1]);
          atomicAdd(&a.mom[2 * k + 1], acc[2]);
          if (MODE == 3) {
            atomicAdd(&a.mom2[3 * k], acc[3 % kQ]);
            atomicAdd(&a.mom2[3 * k + 1], acc[4 % kQ]);
            atomicAdd(&a.mom2[3 * k + 2], acc[5 % kQ]);
          }
        }
      }
    }
  }
}

// The pairs whose fragment outgrew k_frag's staging: streaming integration,
// one pair per thread, grid-stride over the list.
// Bound by the serial chain of a thread, so that single waves all over the chip
// take the list (64 workgroups of 256 threads: 18, 73 and 95 us for the calls
// of 1k, 100k with output and 1M cells, now 17, 67 and 41).
template <int MODE, class R>
__global__ void __launch_bounds__(256) k_frag_wide(CellArgs a, const int32_t *__restrict__ pair_cell,
                                                   const int32_t *__restrict__ pair_tri) {
  const int cnt = *a.novf;
  for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < cnt; idx += gridDim.x * blockDim.x) {
    const int64_t p = a.ovf[idx];
    const int64_t k = pair_cell[p];
    const TriData t = a.tri[pair_tri[p]];
    Stage<R> s1, s2, s3;
    Integrator<MODE, R> I;
    frag_setup<MODE, R>(a, k, t, s1, s2, s3, I);
    frag_clip<R>(PolyGlobal<R>{a, k}, a.pn[k], s1, s2, s3, [&](const SV<R> &v) { I.push(v); });
    I.finish();
    if (!(I.cnt >= 3 && I.positive())) continue;
    if (MODE == 1 && a.fo.count != nullptr) {
      // the fragment twice more: its distinct vertices counted, then written
      const double eps = frag_eps(I.xlo, I.xhi, I.ylo, I.yhi);
      DistinctRun d(eps);
      Integrator<MODE, R> J;  // (I still holds this pair's sums)
      frag_setup<MODE, R>(a, k, t, s1, s2, s3, J);
      frag_clip<R>(PolyGlobal<R>{a, k}, a.pn[k], s1, s2, s3,
                   [&](const SV<R> &q) { d.take((double)q.x, (double)q.y); });
      const int m = d.count();
      unsigned long long f, v;
      frag_reserve(a.fo, m, f, v);
      if (f < (unsigned long long)a.fo.cap_frag && v + m <= (unsigned long long)a.fo.cap_vert) {
        a.fo.cell[f] = a.perm[k];
        a.fo.tri[f] = pair_tri[p];
        a.fo.nv[f] = m;
        a.fo.start[f] = (int64_t)v;
        const double ox = a.pos[2 * k], oy = a.pos[2 * k + 1];
        DistinctRun dw(eps);
        frag_setup<MODE, R>(a, k, t, s1, s2, s3, J);
        frag_clip<R>(PolyGlobal<R>{a, k}, a.pn[k], s1, s2, s3, [&](const SV<R> &q) {
          const int at = dw.cnt;
          if (dw.take((double)q.x, (double)q.y) && at < m) {
            a.fo.xy[2 * (v + at)] = (double)q.x + ox;
            a.fo.xy[2 * (v + at) + 1] = (double)q.y + oy;
          }
        });
      }
    }
    if (MODE == 0) {
      atomicAdd(&a.mass[k], (double)I.mass - (double)I.cmass);
      atomicAdd(&a.intg[k], (double)I.intg - (double)I.cintg);
    } else {
      atomicAdd(&a.mass[k], (double)I.mass);
      atomicAdd(&a.mom[2 * k], (double)I.mx);
      atomicAdd(&a.mom[2 * k + 1], (double)I.my);
    }
    if (MODE == 3) {
      atomicAdd(&a.mom2[3 * k], (double)I.sxx);
      atomicAdd(&a.mom2[3 * k + 1], (double)I.syy);
      atomicAdd(&a.mom2[3 * k + 2], (double)I.sxy);
    }
    if (MODE == 2) {
      const int64_t ti = pair_tri[p];
      for (int v = 0; v < 3; v++) atomicAdd(&a.dval[a.triv[3 * ti + v]], I.dv[v]);
    }
    atomicAdd(&a.counters[0], 1ull);
  }
}

// Hessian rows of the fast-path cells (include/MA/kantorovich.hpp:109-122):
// H_kj = -int_{e_kj} rho ds / (2 |y_k - y_j|), H_kk = -sum_j H_kj, in FP64.
// The lanes of a group hold the edges of one cell.  k_row_count finds how many
// entries each row has; once these are scanned, k_row_fill writes the rows
// into the CSR arrays, each entry at its rank among the labels.  Two short
// passes over the edges (12 B an edge and pass) instead of sorted rows staged
// by one thread per cell and copied by another kernel: 1M cells 77 and 112 us
// against 364 and 104.
struct RowLane {
  int l, base;
  int32_t j = -1;        // neighbour, -1: no entry
  bool lead = false;     // the first lane with this neighbour
  __device__ RowLane() : l((int)threadIdx.x & (kGroup - 1)), base((int)threadIdx.x & 48) {}
  __device__ unsigned mask(bool p) const { return (unsigned)(__ballot(p) >> base) & 0xffffu; }
  // calls f(o) with o = 1..15 as compile-time constants, for row rotations
  template <class F>
  __device__ static void rotations(F &&f) {
    f(std::integral_constant<int, 1>{}); f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{}); f(std::integral_constant<int, 4>{});
    f(std::integral_constant<int, 5>{}); f(std::integral_constant<int, 6>{});
    f(std::integral_constant<int, 7>{}); f(std::integral_constant<int, 8>{});
    f(std::integral_constant<int, 9>{}); f(std::integral_constant<int, 10>{});
    f(std::integral_constant<int, 11>{}); f(std::integral_constant<int, 12>{});
    f(std::integral_constant<int, 13>{}); f(std::integral_constant<int, 14>{});
    f(std::integral_constant<int, 15>{});
  }
  // edge l of cell k (n vertices); returns its integral (all slots are read,
  // so that the loads do not wait for n)
  __device__ double load(const CellArgs &a, int64_t k, int n) {
    const int32_t label = a.plab[k * kMaxFast + l];
    const double e = a.eacc[k * kMaxFast + l];
    // -0.0: edge met by no fragment
    j = l < n && label >= 0 && !is_neg_zero(e) ? label : -1;
    const int key = j >= 0 ? j : -1 - l;
    lead = j >= 0;
    rotations([&](auto o) {  // lane l sees lane l - o
      if (dpp<kDppRor + decltype(o)::value>(key) == key && l >= decltype(o)::value) lead = false;
    });
    return j >= 0 ? e : 0.0;
  }
};

__global__ void __launch_bounds__(kCellThreads) k_row_count(CellArgs a, double *fval_part,
                                                            int32_t *row_cnt, int per) {
  int my_max = 0, my_empty = 0, my_nv = 0;
  const int64_t k0 = ((int64_t)blockIdx.x * kCellGroups + threadIdx.x / kGroup) * per;
  for (int64_t k = k0; k < min(k0 + per, a.n); k++) {
    const int n = a.pn[k];
    RowLane L;
    (void)L.load(a, k, n);
    if (n < 0) continue;  // the general kernels write this row's count
    const int cnt = __popc(L.mask(L.lead));
    if (L.l == 0) {
      row_cnt[k] = cnt > 0 ? cnt + 1 : 0;
      const double m = a.mass[k];
      fval_part[k] = (a.wlo ? a.w[k] + a.wlo[k] : a.w[k]) * m - a.intg[k];
      my_max = max(my_max, n);
      my_empty += m <= 0.0;
      my_nv += n;
    }
  }
  __shared__ int s_max, s_empty, s_nv;
  if (threadIdx.x == 0) s_max = s_empty = s_nv = 0;
  __syncthreads();
  if ((threadIdx.x & (kGroup - 1)) == 0) {
    atomicMax(&s_max, my_max);
    atomicAdd(&s_empty, my_empty);
    atomicAdd(&s_nv, my_nv);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // (the largest cell is soon known, and few cells are empty)
    if ((unsigned long long)s_max > __hip_atomic_load(&a.counters[2], __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(&a.counters[2], (unsigned long long)s_max);
    if (s_empty) atomicAdd(&a.counters[3], (unsigned long long)s_empty);
    atomicAdd(counter_stripe(a.counters, 1, blockIdx.x), (unsigned long long)s_nv);
  }
}

__global__ void __launch_bounds__(kCellThreads) k_row_fill(CellArgs a, const int32_t *ptr,
                                                           int32_t *col, double *val) {
  const int64_t k = xcd_block<kCellXcdRun>(blockIdx.x, gridDim.x) * kCellGroups +
                    threadIdx.x / kGroup;
  if (k >= a.n) return;
  const int n = a.pn[k];
  if (n < 0) return;
  const int32_t o = ptr[k];
  if (ptr[k + 1] == o) return;
  RowLane L;
  const double e = L.load(a, k, n);
  double v = 0.0;
  if (L.j >= 0) {
    const double dx = a.pos[2 * k] - a.pos[2 * L.j], dy = a.pos[2 * k + 1] - a.pos[2 * L.j + 1];
    v = e / (2.0 * sqrt(dx * dx + dy * dy));
  }
  const double diag = row_sum(v);
  if (L.mask(L.lead != (L.j >= 0))) {
    // a label on several edges (degenerate edges): their integrals are one entry
    double s = v;
    RowLane::rotations([&](auto r) {
      const int jr = dpp<kDppRor + decltype(r)::value>(L.j);
      const double vr = dpp<kDppRor + decltype(r)::value>(v);
      if (jr == L.j) s += vr;
    });
    v = s;
  }
  const int key = L.lead ? L.j : INT_MAX;
  int rank = L.lead && L.j > (int32_t)k ? 1 : 0;
  RowLane::rotations([&](auto r) { rank += dpp<kDppRor + decltype(r)::value>(key) < key; });
  if (L.lead) {
    col[o + rank] = L.j;
    val[o + rank] = -v;
  }
  const int below = __popc(L.mask(L.lead && L.j < (int32_t)k));
  if (L.l == 0) {
    col[o + below] = (int32_t)k;
    val[o + below] = diag;
  }
}

// moments: local (relative to the Dirac) -> absolute; with `second`, the
// second moments too (from the local first moments, before those change):
// int rho x^2 = S_uu + 2 y_x M_u + y_x^2 m, int rho x y = S_uv + y_x M_v + y_y M_u + y_x y_y m
__global__ void k_mom_finalize(CellArgs a, int second) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= a.n || a.pn[k] < 0) return;
  const double m = a.mass[k], yx = a.pos[2 * k], yy = a.pos[2 * k + 1];
  const double mu = a.mom[2 * k], mv = a.mom[2 * k + 1];
  if (second) {
    a.mom2[3 * k] += 2.0 * yx * mu + yx * yx * m;
    a.mom2[3 * k + 1] += 2.0 * yy * mv + yy * yy * m;
    a.mom2[3 * k + 2] += yx * mv + yy * mu + yx * yy * m;
  }
  a.mom[2 * k] = mu + yx * m;
  a.mom[2 * k + 1] = mv + yy * m;
}

// Lists the cells whose vertex count holds the marker `value`.
__global__ void k_collect(int64_t n, const int32_t *pn, int32_t value, int32_t *list,
                          int32_t *count) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  if (pn[k] == value) list[atomicAdd(count, 1)] = (int32_t)k;
}

}  // namespace ma

namespace ma {

ma_status run_bin_candidates(ma_engine *e, const int32_t *pn, const unsigned char *mask);

// Bins within kMaskBins (Chebyshev) of the Diracs whose cells the site-centric
// kernel left to other kernels (pn < 0): the starting box of that kernel
// (at most kBoxWide) and one more ring.
constexpr int kMaskBins = (int)kBoxWide + 1;
// One thread per Dirac finds such cells; the wave's 64 lanes mark the square of
// one of them at a time (2000 cells of 2M: 167 us when each thread marked its
// own 35 x 35 bins).
__global__ void k_mark_bins(Grid g, int64_t n, const double *pos, const int32_t *pn,
                            unsigned char *mask) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const bool marks = k < n && pn[k] < 0;
  int bx = 0, by = 0;
  if (marks) {
    bx = bin_coord(pos[2 * k], g.x0, g.h, g.G);
    by = bin_coord(pos[2 * k + 1], g.y0, g.h, g.G);
  }
  constexpr int kSide = 2 * kMaskBins + 1;
  for (unsigned long long m = __ballot(marks); m; m &= m - 1) {
    const int c = __ffsll((long long)m) - 1;
    const int cx = __shfl(bx, c, 64) - kMaskBins, cy = __shfl(by, c, 64) - kMaskBins;
    for (int t = (int)(threadIdx.x & 63); t < kSide * kSide; t += 64) {
      const int x = cx + t % kSide, y = cy + t / kSide;
      if (x >= 0 && x < g.G && y >= 0 && y < g.G) mask[morton2((uint32_t)x, (uint32_t)y)] = 1;
    }
  }
}
// *out = 1 if the bin rectangle of a cell with pn < 0 reaches the outer ring
// of its own square of marked bins (its cell may extend past the bins whose
// lists were built).  Sides on the grid's border need no margin.
__global__ void k_mask_check(Grid g, int64_t n, const double *pos, const int32_t *pn,
                             const int32_t *rect, int32_t *out) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n || pn[k] >= 0) return;
  const int rx0 = rect[4 * k], ry0 = rect[4 * k + 1], rx1 = rect[4 * k + 2], ry1 = rect[4 * k + 3];
  if (rx0 > rx1) return;  // listed nowhere: an empty cell
  const int bx = bin_coord(pos[2 * k], g.x0, g.h, g.G), by = bin_coord(pos[2 * k + 1], g.y0, g.h, g.G);
  const bool bad = (rx0 <= bx - kMaskBins && rx0 > 0) || (ry0 <= by - kMaskBins && ry0 > 0) ||
                   (rx1 >= bx + kMaskBins && rx1 < g.G - 1) ||
                   (ry1 >= by + kMaskBins && ry1 < g.G - 1);
  if (bad) atomicOr(out, 1);
}

// mode: 0 Kantorovich, 1 first moments, 2 adjoint; fp32: FP32 geometry for
// mode 0 (mixed precision).
ma_status run_cells(ma_engine *e, int mode, bool fp32, int32_t *npairs_out,
                    int32_t *ngeneral_out) {
  EvalBuffers &B = e->eb;
  const int64_t n = e->n;
  if (mode != 0) fp32 = false;
  if (fp32) {
    MA_HIP_TRY(B.pxf.ensure((size_t)kMaxFast * n));
    MA_HIP_TRY(B.pyf.ensure((size_t)kMaxFast * n));
  } else {
    MA_HIP_TRY(B.px.ensure((size_t)kMaxFast * n));
    MA_HIP_TRY(B.py.ensure((size_t)kMaxFast * n));
  }
  MA_HIP_TRY(B.eacc.ensure((size_t)kMaxFast * n));
  MA_HIP_TRY(B.plab.ensure((size_t)kMaxFast * n));
  MA_HIP_TRY(B.pn.ensure((size_t)n));
  MA_HIP_TRY(B.bbox.ensure((size_t)(4 * n)));
  MA_HIP_TRY(B.tcount.ensure((size_t)n + 1));
  MA_HIP_TRY(B.poff.ensure((size_t)n + 1));
  MA_HIP_TRY(B.glist.ensure((size_t)n + 1));
  CellArgs a;
  a.g = e->grid;
  a.n = n;
  a.pos = e->pos.p;
  a.w = B.w_s.p;
  a.wlo = B.wlo();
  a.perm = e->perm.p;
  a.rect = B.rect.p;
  a.cand_start = B.cand_cnt.p;
  a.cand = B.cand.p;
  a.tbin_start = e->tbin_start.p;
  a.tbin_items = e->tbin_items.p;
  a.tri = e->tri.p;
  a.tbox = e->tbox.p;
  a.px = B.px.p;
  a.py = B.py.p;
  a.pxf = B.pxf.p;
  a.pyf = B.pyf.p;
  a.plab = B.plab.p;
  a.pn = B.pn.p;
  a.bbox = B.bbox.p;
  a.tcount = B.tcount.p;
  a.mass = B.mass_s.p;
  a.intg = B.intg_s.p;
  a.mom = B.mom_s.p;
  if (mode == 3) MA_HIP_TRY(B.mom2_s.ensure((size_t)(3 * n)));
  a.mom2 = mode == 3 ? B.mom2_s.p : nullptr;
  a.eacc = B.eacc.p;
  a.flags = B.flags.p;
  a.counters = B.counters.p;
  a.force_general = e->force_general;
  // in the far-cell regime the per-bin lists are built anyway, and a cell
  // whose walk runs long mostly ends on the bin path after it: give up early
  a.walk_budget = e->many_far ? std::min(e->walk_budget, kFarWalkBudget) : e->walk_budget;
  MA_HIP_TRY(B.ptri.ensure((size_t)kPadTri * n));
  a.ptri = B.ptri.p;
  MA_HIP_TRY(B.stripes.ensure(48 * 16));
  MA_HIP_TRY(hipMemsetAsync(B.stripes.p, 0, sizeof(unsigned long long) * 48 * 16, e->stream));
  a.stripes = B.stripes.p;
  a.bin_start = e->bin_start.p;
  MA_HIP_TRY(B.far.ensure((size_t)n));
  a.far = B.far.p;
  // only when many cells were far (C4-like: clustered Diracs over a spread
  // density); a few far cells cost the site-centric search less than the
  // bin path they would keep
  a.use_far = (e->far_valid && e->many_far && !fp32 && e->far_cells > 0) ? 1 : 0;
  a.box_half = (e->many_far ? kBoxNarrow : kBoxWide) * e->grid.h;
  a.triv = e->triv.p;
  a.dval = B.dval.p;
  a.fo = e->fo;
  if (mode != 1) a.fo.count = nullptr;
  for (int i = 0; i < 4; i++) a.dom[i] = e->dom[i];
  PyrOff po{};
  for (int l = 0; l <= e->grid.L; l++) po.o[l] = e->pyr_off[l];
  const Plane *planes = reinterpret_cast<const Plane *>(B.plane.p);
  MA_HIP_TRY(hipEventRecord(e->ev[10], e->stream));
  if (fp32)
    hipLaunchKernelGGL(k_cell_local<float>, dim3(nblocks(n, kCellGroups)), dim3(kCellThreads), 0,
                       e->stream, a, B.pyr.p, B.pyr3.p, planes, po, e->local_rings);
  else
    hipLaunchKernelGGL(k_cell_local<double>, dim3(nblocks(n, kCellGroups)), dim3(kCellThreads), 0,
                       e->stream, a, B.pyr.p, B.pyr3.p, planes, po, e->local_rings);
  MA_HIP_TRY(hipEventRecord(e->ev[11], e->stream));
  {
    int32_t fl0[4];
    unsigned long long ct0[8], st[48 * 16];
    MA_HIP_TRY(read_back(e, {{fl0, B.flags.p, sizeof fl0},
                             {ct0, B.counters.p, sizeof ct0},
                             {st, B.stripes.p, sizeof st}}));
    unsigned long long nwalk = 0, nbins = 0, nfail = 0;
    for (int i = 0; i < 16; i++) {
      nwalk += st[i * 16];
      nbins += st[(16 + i) * 16];
      nfail += st[(32 + i) * 16];
    }
    ct0[6] = nbins;
    e->info.nbinpath = (int64_t)nwalk;
    e->info.nbincand = (int64_t)nbins;
    e->ran_candidates = false;
    if (!fp32 && !(fl0[3] || ct0[6])) e->many_far = false;
    if (fl0[3] || ct0[6]) {
      // cells over the walk budget or overflowing the fast path: per-bin
      // candidate owners (and bin rectangles of those cells)
      MA_HIP_TRY(hipEventRecord(e->ev[8], e->stream));
      // few such cells (e.g. the heavy cells at converged weights): candidate
      // lists only for the bins within kMaskBins of their Diracs, accepted
      // when every such cell's bin rectangle stays inside its own square
      // (then its cell does too, and the lists of its bins are complete)
      // (not tried again on the same Diracs once it has fallen through: the
      // cells left over then tend to stay larger than the squares)
      const bool masked = !e->force_general && e->mask_ok &&
                          (int64_t)(nbins + nfail) <= std::max<int64_t>(64, e->grid.nbins / 256);
      // exact per-bin owners pay off when many cells take the bin path (far
      // from their Diracs, with long candidate lists and large rectangles)
      e->refine = (int64_t)nbins >= n / 16;
      if (!fp32) e->many_far = e->refine;
      ma_status s = MA_OK;
      if (masked) {
        MA_HIP_TRY(B.binmask.ensure((size_t)e->grid.nbins));
        MA_HIP_TRY(hipMemsetAsync(B.binmask.p, 0, (size_t)e->grid.nbins, e->stream));
        hipLaunchKernelGGL(k_mark_bins, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, e->grid, n,
                           e->pos.p, B.pn.p, B.binmask.p);
        s = run_bin_candidates(e, B.pn.p, B.binmask.p);
        if (s != MA_OK) return s;
        int32_t outside = 0;
        MA_HIP_TRY(hipMemsetAsync(B.flags.p + 2, 0, sizeof(int32_t), e->stream));
        hipLaunchKernelGGL(k_mask_check, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, e->grid, n,
                           e->pos.p, B.pn.p, B.rect.p, B.flags.p + 2);
        MA_HIP_TRY(read_back(e, {{&outside, B.flags.p + 2, sizeof(int32_t)}}));
        if (outside) {
          e->mask_ok = false;
          s = run_bin_candidates(e, B.pn.p, nullptr);
        }
      } else {
        s = run_bin_candidates(e, B.pn.p, nullptr);
      }
      if (s != MA_OK) return s;
      a.cand_start = B.cand_cnt.p;  // (re)allocated by the candidate search
      a.cand = B.cand.p;
      if (ct0[6]) {
        MA_HIP_TRY(hipMemsetAsync(B.glist.p + n, 0, sizeof(int32_t), e->stream));
        hipLaunchKernelGGL(k_collect, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, n, B.pn.p,
                           -2, B.glist.p, B.glist.p + n);
        const unsigned nb = nblocks((int64_t)ct0[6], kCellGroups);
        if (fp32)
          hipLaunchKernelGGL(k_cell_bins<float>, dim3(nb), dim3(kCellThreads), 0, e->stream, a,
                             B.glist.p, B.glist.p + n);
        else
          hipLaunchKernelGGL(k_cell_bins<double>, dim3(nb), dim3(kCellThreads), 0, e->stream, a,
                             B.glist.p, B.glist.p + n);
      }
      MA_HIP_TRY(hipEventRecord(e->ev[9], e->stream));
      e->ran_candidates = true;
    }
  }
  MA_HIP_TRY(hipEventRecord(e->ev[3], e->stream));
  MA_HIP_TRY(exclusive_scan(e, B.tcount.p, B.poff.p, n));
  int32_t np = 0, fl[4];
  MA_HIP_TRY(read_back(e, {{&np, B.poff.p + n, sizeof np}, {fl, B.flags.p, sizeof fl}}));
  MA_HIP_TRY(B.pair_cell.ensure((size_t)np + 1));
  MA_HIP_TRY(B.pair_tri.ensure((size_t)np + 1));
  hipLaunchKernelGGL(k_pairs, dim3(nblocks(n, kCellGroups)), dim3(kCellThreads), 0, e->stream, a,
                     B.poff.p, B.pair_cell.p, B.pair_tri.p);
  MA_HIP_TRY(hipEventRecord(e->ev[4], e->stream));
  if (np > 0) {
    // list of the pairs whose fragment outgrows k_frag's staging (count at [np])
    MA_HIP_TRY(B.ovf.ensure((size_t)np + 1));
    MA_HIP_TRY(hipMemsetAsync(B.ovf.p + np, 0, sizeof(int32_t), e->stream));
    a.ovf = B.ovf.p;
    a.novf = B.ovf.p + np;
    const dim3 grid(nblocks(np, 256)), block(256), wgrid(1024), wblock(64);
    const int32_t *pc = B.pair_cell.p, *pt = B.pair_tri.p;
    if (mode == 0 && fp32) {
      hipLaunchKernelGGL((k_frag<0, float>), grid, block, 0, e->stream, a, (int64_t)np, pc, pt);
      hipLaunchKernelGGL((k_frag_wide<0, float>), wgrid, wblock, 0, e->stream, a, pc, pt);
    } else if (mode == 0) {
      hipLaunchKernelGGL((k_frag<0, double>), grid, block, 0, e->stream, a, (int64_t)np, pc, pt);
      hipLaunchKernelGGL((k_frag_wide<0, double>), wgrid, wblock, 0, e->stream, a, pc, pt);
    } else if (mode == 1) {
      hipLaunchKernelGGL((k_frag<1, double>), grid, block, 0, e->stream, a, (int64_t)np, pc, pt);
      hipLaunchKernelGGL((k_frag_wide<1, double>), wgrid, wblock, 0, e->stream, a, pc, pt);
    } else if (mode == 3) {
      hipLaunchKernelGGL((k_frag<3, double>), grid, block, 0, e->stream, a, (int64_t)np, pc, pt);
      hipLaunchKernelGGL((k_frag_wide<3, double>), wgrid, wblock, 0, e->stream, a, pc, pt);
    } else {
      hipLaunchKernelGGL((k_frag<2, double>), grid, block, 0, e->stream, a, (int64_t)np, pc, pt);
      hipLaunchKernelGGL((k_frag_wide<2, double>), wgrid, wblock, 0, e->stream, a, pc, pt);
    }
  }
  MA_HIP_TRY(hipEventRecord(e->ev[5], e->stream));
  if (mode == 0) {
    // cells per group: enough workgroups to fill the chip, few enough that
    // their counters' atomics do not queue up
    const int per = (int)std::min<int64_t>(8, std::max<int64_t>(1, n / (2048 * kCellGroups)));
    hipLaunchKernelGGL(k_row_count, dim3(nblocks(n, kCellGroups * per)), dim3(kCellThreads), 0,
                       e->stream, a, B.fval_part.p, B.row_cnt.p, per);
  }
  if (mode == 1 || mode == 3)  // mode 2 keeps the moments about the Dirac
    hipLaunchKernelGGL(k_mom_finalize, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, a,
                       (int)(mode == 3));
  int32_t ng = 0;
  if (fl[3]) {
    MA_HIP_TRY(hipMemsetAsync(B.glist.p + n, 0, sizeof(int32_t), e->stream));
    hipLaunchKernelGGL(k_collect, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, n, B.pn.p, -1,
                       B.glist.p, B.glist.p + n);
    MA_HIP_TRY(read_back(e, {{&ng, B.glist.p + n, sizeof(int32_t)}}));
  }
  MA_HIP_TRY(hipGetLastError());
  *npairs_out = np;
  *ngeneral_out = ng;
  return MA_OK;
}

// The CSR rows of the fast-path cells of the last run_cells (mode 0), at the
// offsets csr_ptr.
ma_status fill_rows(ma_engine *e) {
  EvalBuffers &B = e->eb;
  CellArgs a{};
  a.n = e->n;
  a.pos = e->pos.p;
  a.pn = B.pn.p;
  a.plab = B.plab.p;
  a.eacc = B.eacc.p;
  hipLaunchKernelGGL(k_row_fill, dim3(nblocks(e->n, kCellGroups)), dim3(kCellThreads), 0, e->stream, a,
                     B.csr_ptr.p, B.csr_col.p, B.csr_val.p);
  MA_HIP_TRY(hipGetLastError());
  return MA_OK;
}

}  // namespace ma
