// Geometry kernels of the gfx950 engine: Dirac/triangle binning, the
// max-weight pyramid, per-bin candidate owners, power-cell construction,
// cell x triangle fragments with exact P1 quadrature, and CSR assembly.
//
// Reference behaviour reproduced (paths relative to the MongeAmpere++ tree):
//   fragments and their edge labels   include/MA/voronoi_triangulation_intersection.hpp:42-199
//   strict tie rule                    include/MA/predicates.hpp:85-86
//   mass / value / Hessian per fragment include/MA/kantorovich.hpp:93-135
//   quadrature rules                   include/MA/quadrature.hpp:23-42,69-85,122-143
//   first moments                      include/MA/lloyd.hpp:30-69
#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>

#include "geom_common.h"
#include "lanes.h"

namespace ma {

// ---------------------------------------------------------------------------
// Exclusive prefix sum of int32 (wave64 shuffles, 1024 elements per block).
// ---------------------------------------------------------------------------
// (entries from nin on count as 0)
__global__ void __launch_bounds__(256) k_scan_block(const int32_t *in, int64_t nin, int32_t *out,
                                                     int32_t *sums, int64_t n) {
  __shared__ int32_t ws[8];
  const int tid = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * 1024 + tid * 4;
  int v[4];
  int s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int64_t idx = base + i;
    v[i] = idx < nin ? in[idx] : 0;
    s += v[i];
  }
  const int lane = tid & 63, wid = tid >> 6;
  int x = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) ws[wid] = x;
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int k = 0; k < 4; k++) {
      int t = ws[k];
      ws[k] = acc;
      acc += t;
    }
    ws[4] = acc;
  }
  __syncthreads();
  int excl = x - s + ws[wid];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int64_t idx = base + i;
    if (idx < n) out[idx] = excl;
    excl += v[i];
  }
  if (tid == 0 && sums) sums[blockIdx.x] = ws[4];
}

__global__ void __launch_bounds__(256) k_scan_add(int32_t *out, const int32_t *offs, int64_t n) {
  const int64_t base = (int64_t)blockIdx.x * 1024 + threadIdx.x * 4;
  const int32_t o = offs[blockIdx.x];
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (base + i < n) out[base + i] += o;
}

hipError_t exclusive_scan(ma_engine *e, const int32_t *in, int32_t *out, int64_t n) {
  std::vector<int64_t> len{n + 1};
  while (len.back() > 1024) len.push_back((len.back() + 1023) / 1024);
  int64_t tmp = 0;
  for (size_t l = 1; l < len.size(); l++) tmp += len[l];
  MA_HIP_RET(e->eb.scan_tmp.ensure((size_t)tmp + 1));
  std::vector<int32_t *> buf(len.size());
  buf[0] = out;
  int64_t off = 0;
  for (size_t l = 1; l < len.size(); l++) {
    buf[l] = e->eb.scan_tmp.p + off;
    off += len[l];
  }
  for (size_t l = 0; l < len.size(); l++) {
    const int32_t *src = (l == 0) ? in : buf[l];
    int32_t *sums = (l + 1 < len.size()) ? buf[l + 1] : nullptr;
    hipLaunchKernelGGL(k_scan_block, dim3((unsigned)((len[l] + 1023) / 1024)), dim3(256), 0,
                       e->stream, src, l == 0 ? n : len[l], buf[l], sums, len[l]);
  }
  for (size_t l = len.size() - 1; l-- > 0;) {
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)((len[l] + 1023) / 1024)), dim3(256), 0,
                       e->stream, buf[l], buf[l + 1], len[l]);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Small helpers
// ---------------------------------------------------------------------------
struct ReadSrc {
  const uint32_t *src[kReadParts];
  int words[kReadParts];
};
__global__ void __launch_bounds__(256) k_read_back(ReadSrc s, uint32_t *out) {
  for (int k = 0; k < kReadParts; out += s.words[k++])
    for (int i = threadIdx.x; i < s.words[k]; i += 256) out[i] = s.src[k][i];
}
hipError_t read_back(ma_engine *e, std::initializer_list<ReadPart> parts) {
  ReadSrc s{};
  int k = 0;
  size_t bytes = 0;
  for (const ReadPart &p : parts) {
    bytes += p.bytes;
    if (k == kReadParts || bytes > kReadBytes || p.bytes % 4) return hipErrorInvalidValue;
    s.src[k] = static_cast<const uint32_t *>(p.src);
    s.words[k++] = (int)(p.bytes / 4);
  }
  hipLaunchKernelGGL(k_read_back, dim3(1), dim3(256), 0, e->stream, s, e->pinned);
  MA_HIP_RET(hipGetLastError());
  MA_HIP_RET(hipStreamSynchronize(e->stream));
  const char *h = reinterpret_cast<const char *>(e->pinned);
  for (const ReadPart &p : parts) {
    std::memcpy(p.dst, h, p.bytes);
    h += p.bytes;
  }
  return hipSuccess;
}
__global__ void k_fill_i32(int32_t *p, int32_t v, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_gather_f64(const double *src, const int32_t *perm, double *dst, int64_t n) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) dst[k] = src[perm[k]];
}
__global__ void k_scatter_f64(const double *src, const int32_t *perm, double *dst, int64_t n) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) dst[perm[k]] = src[k];
}

hipError_t to_morton(ma_engine *e, const double *src, double *dst, bool src_on_device) {
  const double *s = src;
  if (!src_on_device) {
    MA_HIP_RET(e->sb.stage.ensure((size_t)e->n));
    MA_HIP_RET(hipMemcpyAsync(e->sb.stage.p, src, sizeof(double) * e->n, hipMemcpyHostToDevice,
                              e->stream));
    s = e->sb.stage.p;
  }
  hipLaunchKernelGGL(k_gather_f64, dim3(nblocks(e->n)), dim3(kBlock), 0, e->stream, s,
                     e->perm.p, dst, e->n);
  return hipGetLastError();
}

hipError_t from_morton(ma_engine *e, const double *src, double *dst, bool dst_on_device) {
  if (dst_on_device) {
    hipLaunchKernelGGL(k_scatter_f64, dim3(nblocks(e->n)), dim3(kBlock), 0, e->stream, src,
                       e->perm.p, dst, e->n);
    return hipGetLastError();
  }
  MA_HIP_RET(e->sb.stage.ensure((size_t)e->n));
  hipLaunchKernelGGL(k_scatter_f64, dim3(nblocks(e->n)), dim3(kBlock), 0, e->stream, src,
                     e->perm.p, e->sb.stage.p, e->n);
  MA_HIP_RET(hipMemcpyAsync(dst, e->sb.stage.p, sizeof(double) * e->n, hipMemcpyDeviceToHost,
                            e->stream));
  return hipStreamSynchronize(e->stream);
}

// ---------------------------------------------------------------------------
// Dirac binning (counting sort by Morton bin, then by caller index).
// ---------------------------------------------------------------------------
__global__ void k_dirac_bin(const double *X, int64_t n, Grid g, int32_t *bin, int32_t *cnt) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int bx = bin_coord(X[2 * i], g.x0, g.h, g.G), by = bin_coord(X[2 * i + 1], g.y0, g.h, g.G);
  int32_t b = (int32_t)morton2((uint32_t)bx, (uint32_t)by);
  bin[i] = b;
  atomicAdd(&cnt[b], 1);
}
// cnt counts down to 0 (k_sort_bins orders the bin afterwards)
__global__ void k_dirac_scatter(const int32_t *bin, int64_t n, const int32_t *start, int32_t *cnt,
                                int32_t *perm) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t b = bin[i];
  perm[start[b] + atomicSub(&cnt[b], 1) - 1] = (int32_t)i;
}
// Sort each bin's item list ascending (lists are short; insertion sort).
__global__ void k_sort_bins(const int32_t *start, int64_t nb, int32_t *items) {
  int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (b >= nb) return;
  int32_t s = start[b], t = start[b + 1];
  for (int32_t i = s + 1; i < t; i++) {
    int32_t v = items[i];
    int32_t j = i - 1;
    while (j >= s && items[j] > v) {
      items[j + 1] = items[j];
      j--;
    }
    items[j + 1] = v;
  }
}
__global__ void k_gather_pos(const double *X, const int32_t *perm, int64_t n, double *pos,
                             int32_t *iperm) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  int32_t i = perm[k];
  pos[2 * k] = X[2 * i];
  pos[2 * k + 1] = X[2 * i + 1];
  iperm[i] = (int32_t)k;
}
__global__ void k_colmajor_to_xy(const double *Xc, int64_t n, double *Xi) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  Xi[2 * i] = Xc[i];
  Xi[2 * i + 1] = Xc[n + i];
}

hipError_t build_dirac_grid(ma_engine *e, const double *d_X, int layout) {
  const int64_t n = e->n;
  const Grid &g = e->grid;
  DBuf<double> &xi = e->cb.xi;
  DBuf<int32_t> &bin = e->cb.bin, &cnt = e->cb.cnt;
  const double *X = d_X;
  if (layout == MA_XY_COLMAJOR) {
    MA_HIP_RET(xi.ensure((size_t)(2 * n)));
    hipLaunchKernelGGL(k_colmajor_to_xy, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, d_X, n,
                       xi.p);
    X = xi.p;
  }
  MA_HIP_RET(bin.ensure((size_t)n));
  MA_HIP_RET(cnt.ensure((size_t)g.nbins + 1));
  MA_HIP_RET(e->bin_start.ensure((size_t)g.nbins + 1));
  MA_HIP_RET(e->perm.ensure((size_t)n));
  MA_HIP_RET(e->iperm.ensure((size_t)n));
  MA_HIP_RET(e->pos.ensure((size_t)(2 * n)));
  MA_HIP_RET(hipMemsetAsync(cnt.p, 0, sizeof(int32_t) * g.nbins, e->stream));
  hipLaunchKernelGGL(k_dirac_bin, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, X, n, g, bin.p,
                     cnt.p);
  MA_HIP_RET(exclusive_scan(e, cnt.p, e->bin_start.p, g.nbins));
  hipLaunchKernelGGL(k_dirac_scatter, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, bin.p, n,
                     e->bin_start.p, cnt.p, e->perm.p);
  hipLaunchKernelGGL(k_sort_bins, dim3(nblocks(g.nbins)), dim3(kBlock), 0, e->stream,
                     e->bin_start.p, g.nbins, e->perm.p);
  hipLaunchKernelGGL(k_gather_pos, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, X, e->perm.p, n,
                     e->pos.p, e->iperm.p);
  MA_HIP_RET(hipGetLastError());
  return hipStreamSynchronize(e->stream);
}

// ---------------------------------------------------------------------------
// Triangle bins: every triangle is listed in each bin its bounding box meets.
// ---------------------------------------------------------------------------
template <bool FILL>
// A triangle is listed in every bin its FP32 (outward-rounded) bounding box
// meets (the box group_triangles tests).
__global__ void k_tbin(const float4 *tbox, int64_t nt, Grid g, int32_t *cnt,
                       const int32_t *start, int32_t *items) {
  int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (f >= nt) return;
  const float4 tb = tbox[f];
  const double x0 = tb.x, y0 = tb.y, x1 = tb.z, y1 = tb.w;
  int bx0 = bin_coord(x0, g.x0, g.h, g.G), bx1 = bin_coord(x1, g.x0, g.h, g.G);
  int by0 = bin_coord(y0, g.y0, g.h, g.G), by1 = bin_coord(y1, g.y0, g.h, g.G);
  for (int by = by0; by <= by1; by++)
    for (int bx = bx0; bx <= bx1; bx++) {
      uint32_t b = morton2((uint32_t)bx, (uint32_t)by);
      if (FILL) {
        const int32_t s = start[b] + atomicSub(&cnt[b], 1) - 1;
        items[s] = ((int32_t)f << kTriShift) | (bx == bx0 ? kTriFirstX : 0) |
                   (by == by0 ? kTriFirstY : 0);
      } else {
        atomicAdd(&cnt[b], 1);
      }
    }
}

hipError_t build_triangle_bins(ma_engine *e) {
  const Grid &g = e->grid;
  DBuf<int32_t> &cnt = e->cb.cnt;
  MA_HIP_RET(cnt.ensure((size_t)g.nbins + 1));
  MA_HIP_RET(e->tbin_start.ensure((size_t)g.nbins + 1));
  MA_HIP_RET(hipMemsetAsync(cnt.p, 0, sizeof(int32_t) * g.nbins, e->stream));
  hipLaunchKernelGGL(k_tbin<false>, dim3(nblocks(e->nt)), dim3(kBlock), 0, e->stream, e->tbox.p,
                     e->nt, g, cnt.p, nullptr, nullptr);
  MA_HIP_RET(exclusive_scan(e, cnt.p, e->tbin_start.p, g.nbins));
  int32_t total = 0;
  MA_HIP_RET(read_back(e, {{&total, e->tbin_start.p + g.nbins, sizeof(int32_t)}}));
  MA_HIP_RET(e->tbin_items.ensure((size_t)total + 1));
  hipLaunchKernelGGL(k_tbin<true>, dim3(nblocks(e->nt)), dim3(kBlock), 0, e->stream, e->tbox.p,
                     e->nt, g, cnt.p, e->tbin_start.p, e->tbin_items.p);
  hipLaunchKernelGGL(k_sort_bins, dim3(nblocks(g.nbins)), dim3(kBlock), 0, e->stream,
                     e->tbin_start.p, g.nbins, e->tbin_items.p);
  MA_HIP_RET(hipGetLastError());
  return hipStreamSynchronize(e->stream);
}

// ---------------------------------------------------------------------------
// Pyramids over the bins: level l node m covers the 4^l bins with Morton codes
// [m 4^l, (m+1) 4^l).  pyr: the largest weight of the node's Diracs (-inf: no
// Diracs); pyr3: the largest over the 3 x 3 nodes around it; and the planes
// (lanes.h).
// ---------------------------------------------------------------------------
// Neighbourhood maxima, all levels in one launch.
__global__ void k_pyr3(Grid g, PyrOff off, int64_t nodes, const double *__restrict__ pyr,
                       double *out) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nodes) return;
  int l = 0;
  while (l < g.L && i >= off.o[l + 1]) l++;
  const double *lvl = pyr + off.o[l];
  const uint32_t m = (uint32_t)(i - off.o[l]);
  const int side = g.G >> l, x = (int)compact1by1(m), y = (int)compact1by1(m >> 1);
  double v = -kInf;
  for (int dy = -1; dy <= 1; dy++)
    for (int dx = -1; dx <= 1; dx++) {
      const int xx = x + dx, yy = y + dy;
      if (xx >= 0 && xx < side && yy >= 0 && yy < side)
        v = fmax(v, lvl[morton2((uint32_t)xx, (uint32_t)yy)]);
    }
  out[i] = v;
}

// lower bound of v_j - 2 x.y_j over the node's Diracs, rounding allowed for
__device__ inline double plane_bound(const Plane &p, const NodeBox &q, double x, double y) {
  double mag;
  const double m = box_min(q, p.ax - 2.0 * x, p.ay - 2.0 * y, mag);
  return p.b + m - kPlaneEps * (fabs(p.b) + mag);
}

// A bound with infinite terms may be no number: then it bounds nothing.  A node
// with Diracs stays below the +inf that marks the empty ones.
__device__ inline double node_bound(double t) { return t != t ? -kInf : fmin(t, DBL_MAX); }

// One group per node of level lev + 2 (lev + 1 when that is the top: step 1);
// lane c takes its descendant c of level lev.  lev = 0: from the Diracs of the
// bins; above: from the records of level lev.  Writes planes and largest
// weights.  Weights need not be finite: -inf (or NaN) is no Dirac here, as in
// pyr; +inf gives its nodes the bound -inf; neither enters the fits.
__global__ void __launch_bounds__(kCellThreads) k_plane(Grid g, int lev, int step,
                                                        const int32_t *__restrict__ bin_start,
                                                        const double *__restrict__ pos,
                                                        const double *__restrict__ w, PyrOff off,
                                                        Plane *pl, NodeSums *sums,
                                                        double *pyr) {
  const int top = lev + step;
  const int64_t node = blockIdx.x * (int64_t)kCellGroups + threadIdx.x / kGroup;
  if (node >= (int64_t)1 << (2 * (g.L - top))) return;
  const int l = (int)threadIdx.x & (kGroup - 1), base4 = 4 * ((int)threadIdx.x & 48);
  const bool on = l < (1 << (2 * step));
  const uint32_t m = ((uint32_t)node << (2 * step)) | (uint32_t)(on ? l : 0);
  const double hx = g.x0 + 0.5 * g.h * g.G, hy = g.y0 + 0.5 * g.h * g.G;
  NodeSums s{0.0, 0.0, 0.0, 0.0};
  double W = -kInf;  // largest weight
  int32_t q0 = 0, q1 = 0;
  if (on && lev == 0) {
    q0 = bin_start[m];
    q1 = bin_start[m + 1];
    for (int32_t q = q0; q < q1; q++) {
      const double x = pos[2 * q] - hx, y = pos[2 * q + 1] - hy, wq = w[q];
      const bool fits = fabs(wq) < kInf;  // (selects: a branch would hold up the loads)
      s.n += fits ? 1.0 : 0.0;
      s.x += fits ? x : 0.0;
      s.y += fits ? y : 0.0;
      s.w += fits ? wq : 0.0;
      W = fmax(W, wq);
    }
    pyr[off.o[0] + m] = W;
  } else if (on) {
    s = sums[off.o[lev] + m];
    W = pyr[off.o[lev] + m];
  }
  // gradient of the weights: least squares over the lanes' means
  const double N = row_sum(s.n), Sx = row_sum(s.x), Sy = row_sum(s.y), Sw = row_sum(s.w);
  double gx = 0.0, gy = 0.0;
  {
    const double in = N > 0.0 ? 1.0 / N : 0.0, im = s.n > 0.0 ? 1.0 / s.n : 0.0;
    const double dx = s.x * im - Sx * in, dy = s.y * im - Sy * in, dw = s.w * im - Sw * in;
    const double xx = row_sum(s.n * dx * dx), xy = row_sum(s.n * dx * dy);
    const double yy = row_sum(s.n * dy * dy);
    const double xw = row_sum(s.n * dx * dw), yw = row_sum(s.n * dy * dw);
    const double det = xx * yy - xy * xy;
    if (det > 1e-6 * xx * yy) {  // else (Diracs on a line, or one): constant weights
      gx = (xw * yy - yw * xy) / det;
      gy = (yw * xx - xw * xy) / det;
    }
    // (finite weights may be too large for their sums)
    if (!(fabs(gx) + fabs(gy) < kInf)) gx = gy = 0.0;
  }
  auto gradient = [&](const NodeBox &q, Plane &p) {
    p.ax = (q.x0 + q.x1) - gx;
    p.ay = (q.y0 + q.y1) - gy;
    p.pad = 0.0;
  };
  Plane p{0.0, 0.0, kInf, 0.0};
  NodeBox q = node_box(g, m, lev);
  if (lev == 0) {
    gradient(q, p);
    for (int32_t i = q0; i < q1; i++) {
      const double x = pos[2 * i] - hx, y = pos[2 * i + 1] - hy;
      const double wi = w[i], v = x * x + y * y - wi, d = p.ax * x + p.ay * y;
      const double t = node_bound(v - d - kPlaneEps * (x * x + y * y + fabs(wi) +
                                                       fabs(p.ax * x) + fabs(p.ay * y)));
      p.b = fmin(p.b, wi > -kInf ? t : kInf);
    }
    if (on) pl[off.o[0] + m] = p;
  } else if (on) {
    p = pl[off.o[lev] + m];
  }
  // one and two levels up: the children's bounds moved to the parent's gradient
  uint32_t mm = m;
  for (int k = 1; k <= step; k++) {
    mm >>= 2;
    Plane u{0.0, 0.0, kInf, 0.0};
    const NodeBox up = node_box(g, mm, lev + k);
    gradient(up, u);
    double t = kInf;
    if (on && p.b < kInf) {
      double mag;
      const double d = box_min(q, p.ax - u.ax, p.ay - u.ay, mag);
      t = node_bound(p.b + d - kPlaneEps * (fabs(p.b) + mag));
    }
    const int st = k == 1 ? 1 : 4;  // lanes of the children: l, l ^ st, ...
    t = fmin(t, row_get(t, base4, l ^ st));
    t = fmin(t, row_get(t, base4, l ^ (2 * st)));
    u.b = t;
    W = fmax(W, row_get(W, base4, l ^ st));
    W = fmax(W, row_get(W, base4, l ^ (2 * st)));
    if (on && (l & (4 * st - 1)) == 0) {
      pl[off.o[lev + k] + mm] = u;
      pyr[off.o[lev + k] + mm] = W;
    }
    p = u;
    q = up;
  }
  if (l == 0) sums[off.o[top] + node] = NodeSums{N, Sx, Sy, Sw};
}

// true if pi_j - pi_k (affine) can be <= 0 somewhere in the bin (min over
// corners); corners in absolute coordinates.  Beside an infinite weight only
// the order counts: a Dirac of weight -inf, or beside one of weight +inf, owns
// nothing and is not listed.
__device__ inline bool may_beat(double x0, double y0, double h, double jx, double jy, double wj,
                                double kx, double ky, double wk) {
  bool ok = false;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const double cx = x0 + (c & 1 ? h : 0.0), cy = y0 + (c & 2 ? h : 0.0);
    const double dj = (cx - jx) * (cx - jx) + (cy - jy) * (cy - jy) - wj;
    const double dk = (cx - kx) * (cx - kx) + (cy - ky) * (cy - ky) - wk;
    ok |= fabs(dj) < kInf && fabs(dk) < kInf ? (dj - dk) <= 1e-12 * (fabs(dj) + fabs(dk))
                                             : dj < dk;
  }
  return ok;
}

// Depth-first walk of the plane pyramid by the 16 lanes of a group: the
// grandchildren of a node are tested at once (keep(plane, box)), nodes of few
// Diracs are taken whole, and visit(q, valid) gets 16 Diracs at a time.
constexpr int kWalkTake = 16;
template <class Keep, class Visit>
__device__ inline void row_walk(const Grid &g, const int32_t *bin_start, const Plane *pl,
                                const PyrOff &off, uint32_t *stack, int base, int l, Keep &&keep,
                                Visit &&visit) {
  int sp = 0;
  uint32_t ent = (uint32_t)g.L << 27;
  while (true) {
    const int lev = (int)(ent >> 27), st = min(lev, 2), cl = lev - st;
    const uint32_t ch = ((ent & ((1u << 27) - 1u)) << (2 * st)) | (uint32_t)l;
    bool descend = false;
    int32_t lo = 0;
    int cnt = 0;
    if (l < (1 << (2 * st))) {
      const Plane p = pl[off.o[cl] + ch];
      if (p.b < kInf && keep(p, node_box(g, ch, cl))) {
        lo = bin_start[(int64_t)ch << (2 * cl)];
        cnt = bin_start[((int64_t)ch + 1) << (2 * cl)] - lo;
        if (cl > 0 && cnt > kWalkTake) {
          descend = true;
          cnt = 0;
        }
      }
    }
    const unsigned dm = (unsigned)(__ballot(descend) >> base) & 0xffffu;
    if (descend) stack[sp + __popc(dm & ((1u << l) - 1u))] = ((uint32_t)cl << 27) | ch;
    sp += __popc(dm);
    for_ranges(base, l, lo, cnt, []() { return true; },
               [&](int32_t q, int, bool valid) { visit(q, valid); });
    if (sp == 0) break;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the lanes' stack entries
    ent = stack[--sp];
  }
}

// Candidate owners of a bin: with k the owner of the bin's centre, the Diracs
// j with pi_j <= pi_k at some corner (pi_j - pi_k is affine, so no other Dirac
// owns a point of the bin).  Counting pass, 16 lanes per bin: a first walk
// finds k (starting from the previous evaluation's, or from a greedy descent),
// a second one counts the candidates and keeps the first kCandStage of them
// (stage[b * kCandStage + i], 512 B per bin, allocated only when lists are
// built).  Filling pass, into exactly sized CSR lists: copies those, and walks
// again only for the bins with more (48 kept candidates left C2's converged
// cells a third slower).  VALU work of the node tests bounds it (81 % busy,
// 77 % of the lanes active; the count of all bins at one address hides behind
// it).  200k clustered Diracs, 512 x 512 bins: 16.5 ms with one thread per bin
// walking the max-weight pyramid, 3.1 ms with a group per bin on that pyramid,
// 0.93 ms with the planes (their five launches take 0.03 ms).
constexpr int kCandStage = 128;
template <bool FILL>
__global__ void __launch_bounds__(kCellThreads) k_cand_list(
    Grid g, const int32_t *__restrict__ tbin_start, const int32_t *__restrict__ bin_start,
    const double *__restrict__ pos, const double *__restrict__ w, const Plane *__restrict__ pl,
    PyrOff off, int32_t *owner, int32_t *cand_start, int32_t *cand, int32_t *cbin, int32_t *stage,
    unsigned long long *counters, const unsigned char *__restrict__ mask) {
  __shared__ uint32_t stacks[kCellGroups][kWalkStack];
  const int64_t b = xcd_block<kCellXcdRun>(blockIdx.x, gridDim.x) * kCellGroups +
                    threadIdx.x / kGroup;
  if (b >= g.nbins) return;
  const int l = (int)threadIdx.x & (kGroup - 1), base = (int)threadIdx.x & 48;
  uint32_t *stack = stacks[threadIdx.x / kGroup];
  if (FILL) {
    const int32_t o = cand_start[b], c = cand_start[b + 1] - o;
    if (c <= kCandStage) {
      for (int i = l; i < c; i += kGroup) {
        cand[o + i] = stage[b * kCandStage + i];
        cbin[o + i] = (int32_t)b;
      }
      return;
    }
  } else if (tbin_start[b + 1] == tbin_start[b] || (mask && !mask[b])) {
    if (l == 0) cand_start[b] = 0;  // no triangle (or not needed): no candidates
    return;
  }
  const NodeBox B = node_box(g, (uint32_t)b, 0);
  const double hx = g.x0 + 0.5 * g.h * g.G, hy = g.y0 + 0.5 * g.h * g.G;
  int best = owner[b];
  if (!FILL) {
    const double mx = 0.5 * (B.x0 + B.x1), my = 0.5 * (B.y0 + B.y1);
    // v - 2 x.y of a Dirac at the bin's centre x
    auto value = [&](int32_t q) {
      const double x = pos[2 * q] - hx, y = pos[2 * q + 1] - hy;
      return x * x + y * y - w[q] - 2.0 * (mx * x + my * y);
    };
    double U = kInf;
    auto better = [&](int32_t q, bool valid) {
      const double h = valid ? value(q) : kInf;
      const double m = row_min(h);
      if (m < U) {
        U = m;
        best = row_get(q, 4 * base, __ffs((unsigned)(__ballot(h == m) >> base) & 0xffffu) - 1);
      }
    };
    if (best >= 0) U = value(best);
    if (!(U < kInf)) {  // no last owner, or its weight is -inf or NaN now
      U = kInf;
      best = -1;
      // greedy descent to the bin with the smallest lower bound
      uint32_t m = 0;
      for (int lev = g.L; lev > 0;) {
        const int st = min(lev, 2);
        lev -= st;
        const uint32_t ch = (m << (2 * st)) | (uint32_t)l;
        double v = kInf;
        if (l < (1 << (2 * st))) {
          const Plane p = pl[off.o[lev] + ch];
          if (p.b < kInf) v = plane_bound(p, node_box(g, ch, lev), mx, my);
        }
        const unsigned eq = (unsigned)(__ballot(v == row_min(v)) >> base) & 0xffffu;
        m = (m << (2 * st)) | (uint32_t)(eq ? __ffs(eq) - 1 : 0);
      }
      const int32_t q0 = bin_start[m], q1 = bin_start[m + 1];
      for (int32_t q = q0; q < q1; q += kGroup) better(q + l, q + l < q1);
    }
    row_walk(g, bin_start, pl, off, stack, base, l,
             [&](const Plane &p, const NodeBox &q) { return !(plane_bound(p, q, mx, my) > U); },
             better);
    if (l == 0) owner[b] = best;
    if (best < 0) {  // no Dirac has a weight above -inf
      if (l == 0) cand_start[b] = 0;
      return;
    }
  }
  const double kx = pos[2 * best], ky = pos[2 * best + 1], kw = w[best];
  // the owner's v - 2 x.y at the corners, rounding allowed for (weight +inf:
  // only its like may share the bin)
  double thr[4];
  {
    const double x = kx - hx, y = ky - hy, v = x * x + y * y - kw;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const double cx = c & 1 ? B.x1 : B.x0, cy = c & 2 ? B.y1 : B.y0;
      thr[c] = kw < kInf ? v - 2.0 * (cx * x + cy * y) +
                               kPlaneEps * (x * x + y * y + fabs(kw) +
                                            2.0 * (fabs(cx * x) + fabs(cy * y)))
                         : -kInf;
    }
  }
  const double ox = B.x0 + hx, oy = B.y0 + hy;  // the bin's lower corner
  int cnt = 0;
  const int32_t o = FILL ? cand_start[b] : 0;
  row_walk(g, bin_start, pl, off, stack, base, l,
           [&](const Plane &p, const NodeBox &q) {
             bool any = false;
#pragma unroll
             for (int c = 0; c < 4; c++)
               any |= !(plane_bound(p, q, c & 1 ? B.x1 : B.x0, c & 2 ? B.y1 : B.y0) > thr[c]);
             return any;
           },
           [&](int32_t q, bool valid) {
             const bool hit = valid && (q == best || may_beat(ox, oy, g.h, pos[2 * q],
                                                              pos[2 * q + 1], w[q], kx, ky, kw));
             const unsigned hm = (unsigned)(__ballot(hit) >> base) & 0xffffu;
             const int at = cnt + __popc(hm & ((1u << l) - 1u));
             if (hit && FILL) {
               cand[o + at] = q;
               cbin[o + at] = (int32_t)b;
             } else if (hit && at < kCandStage) {
               stage[b * kCandStage + at] = q;
             }
             cnt += __popc(hm);
           });
  if (!FILL && l == 0) {
    cand_start[b] = cnt;
    atomicAdd(&counters[1], (unsigned long long)cnt);
  }
}

// Compaction of the refined candidate lists: pos is the exclusive prefix sum
// of the keep flags (an entry is kept iff pos[i + 1] > pos[i]).
__global__ void k_refine_starts(int64_t nb, const int32_t *start, const int32_t *pos,
                                int32_t *nstart) {
  const int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (b <= nb) nstart[b] = pos[start[b]];
}
__global__ void k_refine_move(int64_t nc, const int32_t *pos, const int32_t *cand,
                              int32_t *ncand) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < nc && pos[i + 1] > pos[i]) ncand[pos[i]] = cand[i];
}

__global__ void k_rect_init(int32_t *r, int64_t n) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  r[4 * k] = INT_MAX;
  r[4 * k + 1] = INT_MAX;
  r[4 * k + 2] = -1;
  r[4 * k + 3] = -1;
}

// Bin rectangle of every Dirac: bounding box (in bin coordinates) of the bins
// listing it as a candidate.
// Only Diracs marked pn[q] < 0 (uncertified by the site-centric search, or
// overflowing it) are needed.
__global__ void k_rect(Grid g, const int32_t *tbin_start, const int32_t *cand_start,
                       const int32_t *cand, const int32_t *pn, int32_t *rect) {
  const int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (b >= g.nbins) return;
  if (tbin_start[b + 1] == tbin_start[b]) return;
  const int bx = (int)compact1by1((uint32_t)b), by = (int)compact1by1((uint32_t)(b >> 1));
  for (int32_t i = cand_start[b]; i < cand_start[b + 1]; i++) {
    int32_t q = cand[i];
    if (pn[q] >= 0) continue;
    atomicMin(&rect[4 * q + 0], bx);
    atomicMin(&rect[4 * q + 1], by);
    atomicMax(&rect[4 * q + 2], bx);
    atomicMax(&rect[4 * q + 3], by);
  }
}

// ---------------------------------------------------------------------------
// Per-Dirac cell construction and integration.
// ---------------------------------------------------------------------------
struct Poly {
  int n;
  double x[kMaxPoly], y[kMaxPoly];
  int lab[kMaxPoly];  // label of edge k -> k+1
};

// Keep L(X) = kk - 2 X.Y > 0 (strict tie rule).  Vertex-based
// Sutherland-Hodgman; each vertex carries the label of its outgoing edge.
// Returns false on capacity overflow.
__device__ inline bool clip_cell(Poly &P, Poly &Q, double Yx, double Yy, double kk, int label) {
  const int n = P.n;
  double s[kMaxPoly];
  int nin = 0;
  for (int i = 0; i < n; i++) {
    s[i] = kk - 2.0 * (P.x[i] * Yx + P.y[i] * Yy);
    nin += s[i] > 0.0;
  }
  if (nin == n) return true;
  if (nin == 0) {
    P.n = 0;
    return true;
  }
  int m = 0;
  for (int i = 0; i < n; i++) {
    const int i1 = (i + 1 == n) ? 0 : i + 1;
    if (m + 2 > kMaxPoly) return false;
    if (s[i] > 0.0) {
      Q.x[m] = P.x[i];
      Q.y[m] = P.y[i];
      Q.lab[m] = P.lab[i];
      m++;
      if (!(s[i1] > 0.0)) {
        const double t = s[i] / (s[i] - s[i1]);
        Q.x[m] = P.x[i] + t * (P.x[i1] - P.x[i]);
        Q.y[m] = P.y[i] + t * (P.y[i1] - P.y[i]);
        Q.lab[m] = label;
        m++;
      }
    } else if (s[i1] > 0.0) {
      const double t = s[i] / (s[i] - s[i1]);
      Q.x[m] = P.x[i] + t * (P.x[i1] - P.x[i]);
      Q.y[m] = P.y[i] + t * (P.y[i1] - P.y[i]);
      Q.lab[m] = P.lab[i];
      m++;
    }
  }
  for (int i = 0; i < m; i++) {
    P.x[i] = Q.x[i];
    P.y[i] = Q.y[i];
    P.lab[i] = Q.lab[i];
  }
  P.n = m;
  return true;
}

// Clip a fragment by the closed half-plane left of (ax,ay)->(bx,by).
// Degenerate (zero-area) results are discarded by the caller.
__device__ inline bool clip_tri_edge(const Poly &P, Poly &Q, double ax, double ay, double bx,
                                     double by) {
  const int n = P.n;
  double s[kMaxPoly];
  const double ex = bx - ax, ey = by - ay;
  const double elen = sqrt(ex * ex + ey * ey);
  int nin = 0;
  for (int i = 0; i < n; i++) {
    const double dx = P.x[i] - ax, dy = P.y[i] - ay;
    s[i] = ex * dy - ey * dx;
    // within rounding of the line: on it (see Stage::side)
    if (fabs(s[i]) <= kSnap * elen * (fabs(P.x[i]) + fabs(P.y[i]) + fabs(dx) + fabs(dy)))
      s[i] = 0.0;
    nin += s[i] >= 0.0;
  }
  if (nin == 0) {
    Q.n = 0;
    return true;
  }
  if (nin == n) {
    for (int i = 0; i < n; i++) {
      Q.x[i] = P.x[i];
      Q.y[i] = P.y[i];
      Q.lab[i] = P.lab[i];
    }
    Q.n = n;
    return true;
  }
  int m = 0;
  for (int i = 0; i < n; i++) {
    const int i1 = (i + 1 == n) ? 0 : i + 1;
    if (m + 2 > kMaxPoly) return false;
    if (s[i] >= 0.0) {
      Q.x[m] = P.x[i];
      Q.y[m] = P.y[i];
      Q.lab[m] = P.lab[i];
      m++;
      if (s[i1] < 0.0) {
        const double t = s[i] / (s[i] - s[i1]);
        Q.x[m] = P.x[i] + t * (P.x[i1] - P.x[i]);
        Q.y[m] = P.y[i] + t * (P.y[i1] - P.y[i]);
        Q.lab[m] = -1;
        m++;
      }
    } else if (s[i1] >= 0.0) {
      const double t = s[i] / (s[i] - s[i1]);
      Q.x[m] = P.x[i] + t * (P.x[i1] - P.x[i]);
      Q.y[m] = P.y[i] + t * (P.y[i1] - P.y[i]);
      Q.lab[m] = P.lab[i];
      m++;
    }
  }
  Q.n = m;
  return true;
}

// Integrals over one convex fragment (vertices (qx, qy)[0..m), coordinates
// local to the Dirac) of triangle t, added to S: mass and int rho |x|^2
// (MODE 0), or mass and first moments (MODE 1, 2); MODE 2 also returns in dv
// the integrals of (|x|^2 - w_k) phi_v for the triangle's three hat functions.
// Fan from vertex 0 (include/MA/quadrature.hpp:122-143); the mass by the
// centroid rule, the rest by the Albrecht-Collatz points (exact for the
// cubic integrands).
struct FragSums {
  double mass = 0.0, intg = 0.0, momx = 0.0, momy = 0.0;
  double sxx = 0.0, syy = 0.0, sxy = 0.0;  // second moments (MODE 3)
};
template <int MODE>
__device__ inline void frag_integrals(const double *qx, const double *qy, int m,
                                      const TriData &t, double yx, double yy, double wk,
                                      FragSums &S, double dv[3]) {
  const double r0 = t.a * yx + t.b * yy + t.c;  // rho at the Dirac
  double la[3], lb[3], lc[3];
  if (MODE == 2) {
    // barycentric coordinates of the triangle as affine functions
    const double ax = t.x[0] - yx, ay = t.y[0] - yy, bx = t.x[1] - yx, by = t.y[1] - yy;
    const double cx = t.x[2] - yx, cy = t.y[2] - yy;
    const double inv = 1.0 / ((bx - ax) * (cy - ay) - (cx - ax) * (by - ay));
    la[0] = (by - cy) * inv; lb[0] = (cx - bx) * inv; lc[0] = (bx * cy - cx * by) * inv;
    la[1] = (cy - ay) * inv; lb[1] = (ax - cx) * inv; lc[1] = (cx * ay - ax * cy) * inv;
    la[2] = (ay - by) * inv; lb[2] = (bx - ax) * inv; lc[2] = (ax * by - bx * ay) * inv;
  }
  for (int i = 1; i + 1 < m; i++) {
    const double x0 = qx[0], y0 = qy[0], x1 = qx[i], y1 = qy[i];
    const double x2 = qx[i + 1], y2 = qy[i + 1];
    const double area = 0.5 * ((x1 - x0) * (y2 - y0) - (x2 - x0) * (y1 - y0));
    const double gx = (x0 + x1 + x2) / 3.0, gy = (y0 + y1 + y2) / 3.0;
    S.mass += area * (r0 + t.a * gx + t.b * gy);
    AC6 qp;
    ac6_points(x0, y0, x1, y1, x2, y2, qp);
    double s1 = 0.0, s9 = 0.0, m1x = 0.0, m9x = 0.0, m1y = 0.0, m9y = 0.0;
    double q1[3] = {0.0, 0.0, 0.0}, q9[3] = {0.0, 0.0, 0.0};  // MODE 3: xx, yy, xy
    double c1[3] = {0.0, 0.0, 0.0}, c9[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < 6; p++) {
      const double rp = r0 + t.a * qp.px[p] + t.b * qp.py[p];
      if (MODE == 2) {
        const double c = qp.px[p] * qp.px[p] + qp.py[p] * qp.py[p] - wk;
#pragma unroll
        for (int v = 0; v < 3; v++) {
          const double f = c * (la[v] * qp.px[p] + lb[v] * qp.py[p] + lc[v]);
          if (p < 3) c1[v] += f; else c9[v] += f;
        }
      }
      if (MODE == 3) {
        const double fx = rp * qp.px[p], fy = rp * qp.py[p];
        const double t[3] = {fx * qp.px[p], fy * qp.py[p], fx * qp.py[p]};
#pragma unroll
        for (int v = 0; v < 3; v++) {
          if (p < 3) q1[v] += t[v]; else q9[v] += t[v];
        }
      }
      if (MODE == 0) {
        const double f = rp * (qp.px[p] * qp.px[p] + qp.py[p] * qp.py[p]);
        if (p < 3) s1 += f; else s9 += f;
      } else {
        if (p < 3) {
          m1x += rp * qp.px[p];
          m1y += rp * qp.py[p];
        } else {
          m9x += rp * qp.px[p];
          m9y += rp * qp.py[p];
        }
      }
    }
    if (MODE == 0) {
      S.intg += area * (s1 * (1.0 / 30.0) + s9 * (9.0 / 30.0));
    } else {
      S.momx += area * (m1x * (1.0 / 30.0) + m9x * (9.0 / 30.0));
      S.momy += area * (m1y * (1.0 / 30.0) + m9y * (9.0 / 30.0));
    }
    if (MODE == 3) {
      S.sxx += area * (q1[0] * (1.0 / 30.0) + q9[0] * (9.0 / 30.0));
      S.syy += area * (q1[1] * (1.0 / 30.0) + q9[1] * (9.0 / 30.0));
      S.sxy += area * (q1[2] * (1.0 / 30.0) + q9[2] * (9.0 / 30.0));
    }
    if (MODE == 2) {
#pragma unroll
      for (int v = 0; v < 3; v++) dv[v] += area * (c1[v] * (1.0 / 30.0) + c9[v] * (9.0 / 30.0));
    }
  }
}

// General per-Dirac kernel (polygons up to kMaxPoly vertices in private
// memory) for the cells listed in `list`: the rare cells that overflow the
// register/LDS fast path.
// MODE 0: Kantorovich, 1: first moments, 2: first moments + density-value
// adjoint (integrals of (|x - y_k|^2 - w_k) phi_v, accumulated into dval),
// 3: first and second moments (include/MA/lloyd.hpp:71-123).
template <int MODE>
__global__ void __launch_bounds__(kBlock) k_cells_general(
    const int32_t *__restrict__ list, const int32_t *__restrict__ nlist,
    Grid g, int64_t n, const double *__restrict__ pos, const double *__restrict__ w,
    const double *wlo, const int32_t *__restrict__ perm, const int32_t *__restrict__ rect,
    const int32_t *__restrict__ cand_start, const int32_t *__restrict__ cand,
    const int32_t *__restrict__ tbin_start, const int32_t *__restrict__ tbin_items,
    const TriData *__restrict__ tri, double *mass_out, double *intg_out, double *fval_part,
    double *mom_out, double *mom2_out, int32_t *row_cnt, int32_t *row_col, double *row_val,
    int cap_row, const int32_t *__restrict__ triv, double *dval, int32_t *hlist, int force_huge,
    int32_t *flags, unsigned long long *counters) {
  const int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (idx >= *nlist) return;
  const int64_t k = list[idx];
  const int rx0 = rect[4 * k], ry0 = rect[4 * k + 1], rx1 = rect[4 * k + 2], ry1 = rect[4 * k + 3];
  if (rx0 <= rx1 && (int64_t)(rx1 - rx0 + 1) * (ry1 - ry0 + 1) > kBigRect) {
    hlist[atomicAdd(&hlist[n], 1)] = (int32_t)k;  // k_cell_huge
    return;
  }
  const double yx = pos[2 * k], yy = pos[2 * k + 1], wk = w[k];
  Poly P, Q, F;
  P.n = 0;
  if (rx0 <= rx1) {
    const double X0 = g.x0 + rx0 * g.h - yx, X1 = g.x0 + (rx1 + 1) * g.h - yx;
    const double Y0 = g.y0 + ry0 * g.h - yy, Y1 = g.y0 + (ry1 + 1) * g.h - yy;
    P.n = 4;
    P.x[0] = X0; P.y[0] = Y0; P.lab[0] = -1;
    P.x[1] = X1; P.y[1] = Y0; P.lab[1] = -1;
    P.x[2] = X1; P.y[2] = Y1; P.lab[2] = -1;
    P.x[3] = X0; P.y[3] = Y1; P.lab[3] = -1;
  }
  bool overflow = false;
  double rho2 = 0.0;
  for (int v = 0; v < P.n; v++) rho2 = fmax(rho2, P.x[v] * P.x[v] + P.y[v] * P.y[v]);
  // bins in Chebyshev rings around the Dirac's bin (clamped into the
  // rectangle): near candidates first keep the intermediate polygons small
  const int sbx = min(max(bin_coord(yx, g.x0, g.h, g.G), rx0), rx1);
  const int sby = min(max(bin_coord(yy, g.y0, g.h, g.G), ry0), ry1);
  const int maxr = max(max(sbx - rx0, rx1 - sbx), max(sby - ry0, ry1 - sby));
  for (int r = 0; r <= maxr && P.n > 0; r++)
  for (int by = max(sby - r, ry0); by <= min(sby + r, ry1) && P.n > 0; by++)
    for (int bx = max(sbx - r, rx0); bx <= min(sbx + r, rx1) && P.n > 0; bx++) {
      if (by != sby - r && by != sby + r && bx != sbx - r && bx != sbx + r) continue;
      const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
      for (int32_t i = cand_start[b]; i < cand_start[b + 1] && P.n > 0; i++) {
        const int32_t j = cand[i];
        if (j == k) continue;
        bool seen = false;
        for (int v = 0; v < P.n; v++) seen |= (P.lab[v] == j);
        if (seen) continue;
        const double Yx = pos[2 * j] - yx, Yy = pos[2 * j + 1] - yy, wj = w[j];
        const double d2 = Yx * Yx + Yy * Yy;
        const double dw = wdiff(wlo, wk, k, wj, j);  // w_k - w_j
        if (d2 == 0.0) {
          // coincident Diracs: the larger weight (then the smaller caller
          // index) hides the other
          if (dw < 0.0 || (dw == 0.0 && perm[j] < perm[k])) P.n = 0;
          continue;
        }
        const double d = sqrt(d2), rho = sqrt(rho2);
        if (d2 - 2.0 * rho * d + dw > 1e-12 * (d2 + fabs(wk) + fabs(wj))) continue;
        if (!clip_cell(P, Q, Yx, Yy, d2 + dw, j)) {
          overflow = true;
          P.n = 0;
        }
        rho2 = 0.0;
        for (int v = 0; v < P.n; v++) rho2 = fmax(rho2, P.x[v] * P.x[v] + P.y[v] * P.y[v]);
      }
    }
  // cells beyond this kernel's capacity go to k_cell_huge (a fragment of an
  // n-gon has at most n + 3 vertices, a row at most n + 1 entries)
  if (overflow || P.n > kMaxPoly - 4 || force_huge) {
    hlist[atomicAdd(&hlist[n], 1)] = (int32_t)k;
    return;
  }

  FragSums S;
  double acc[kMaxPoly];
  uint64_t touched = 0u;
  int nfrag = 0;
  const int np = P.n;
  for (int v = 0; v < np; v++) acc[v] = 0.0;
  if (np > 0) {
    double px0 = kInf, py0 = kInf, px1 = -kInf, py1 = -kInf;
    for (int v = 0; v < np; v++) {
      px0 = fmin(px0, P.x[v]);
      px1 = fmax(px1, P.x[v]);
      py0 = fmin(py0, P.y[v]);
      py1 = fmax(py1, P.y[v]);
    }
    px0 += yx; px1 += yx; py0 += yy; py1 += yy;  // absolute bounding box
    const int qx0 = max(bin_coord(px0, g.x0, g.h, g.G), rx0);
    const int qx1 = min(bin_coord(px1, g.x0, g.h, g.G), rx1);
    const int qy0 = max(bin_coord(py0, g.y0, g.h, g.G), ry0);
    const int qy1 = min(bin_coord(py1, g.y0, g.h, g.G), ry1);
    for (int by = qy0; by <= qy1; by++)
      for (int bx = qx0; bx <= qx1; bx++) {
        const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
        for (int32_t q = tbin_start[b]; q < tbin_start[b + 1]; q++) {
          const TriData t = tri[tbin_items[q] >> kTriShift];
          double tx0, ty0, tx1, ty1;
          tri_bbox(t, tx0, ty0, tx1, ty1);
          if (tx1 < px0 || tx0 > px1 || ty1 < py0 || ty0 > py1) continue;
          // visit each triangle once: in the bin holding the lower-left
          // corner of the overlap of the two bounding boxes
          const int ox = max(bin_coord(fmax(tx0, px0), g.x0, g.h, g.G), qx0);
          const int oy = max(bin_coord(fmax(ty0, py0), g.y0, g.h, g.G), qy0);
          if (ox != bx || oy != by) continue;
          // local triangle
          const double ax = t.x[0] - yx, ay = t.y[0] - yy;
          const double bxx = t.x[1] - yx, byy = t.y[1] - yy;
          const double cx = t.x[2] - yx, cy = t.y[2] - yy;
          // fragment = cell clipped by the three triangle edges; cell edges
          // are labelled by their index in P, triangle edges by -1
          F.n = np;
          for (int v = 0; v < np; v++) {
            F.x[v] = P.x[v];
            F.y[v] = P.y[v];
            F.lab[v] = v;
          }
          if (!clip_tri_edge(F, Q, ax, ay, bxx, byy) || !clip_tri_edge(Q, F, bxx, byy, cx, cy) ||
              !clip_tri_edge(F, Q, cx, cy, ax, ay)) {
            overflow = true;
            continue;
          }
          const int m = Q.n;
          if (m < 3) continue;
          {
            // fragments of zero area (cell touching the triangle along an
            // edge or at a point) do not count; see Integrator::positive
            double ar2 = 0.0, xlo = kInf, xhi = -kInf, ylo = kInf, yhi = -kInf, cm = 0.0;
            for (int i = 0; i < m; i++) {
              const int i1 = (i + 1 == m) ? 0 : i + 1;
              ar2 += Q.x[i] * Q.y[i1] - Q.x[i1] * Q.y[i];
              xlo = fmin(xlo, Q.x[i]);
              xhi = fmax(xhi, Q.x[i]);
              ylo = fmin(ylo, Q.y[i]);
              yhi = fmax(yhi, Q.y[i]);
              cm = fmax(cm, fmax(fabs(Q.x[i]), fabs(Q.y[i])));
            }
            if (!(0.5 * ar2 > 1e-13 * ((xhi - xlo) + (yhi - ylo)) * cm)) continue;
          }
          nfrag++;
          const double r0 = t.a * yx + t.b * yy + t.c;  // rho at the Dirac
          double dv[3] = {0.0, 0.0, 0.0};
          frag_integrals<MODE>(Q.x, Q.y, m, t, yx, yy, wk, S, dv);
          if (MODE == 2) {
            const int64_t ti = tbin_items[q] >> kTriShift;
#pragma unroll
            for (int v = 0; v < 3; v++) atomicAdd(&dval[triv[3 * ti + v]], dv[v]);
          }
          if (MODE == 0) {
            // Hessian contributions of the fragment's cell edges
            // (include/MA/kantorovich.hpp:109-122)
            for (int i = 0; i < m; i++) {
              const int lab = Q.lab[i];
              if (lab < 0 || P.lab[lab] < 0) continue;
              const int i1 = (i + 1 == m) ? 0 : i + 1;
              const double ex = Q.x[i1] - Q.x[i], ey = Q.y[i1] - Q.y[i];
              if (ex == 0.0 && ey == 0.0) continue;  // piece from a snapped vertex
              const double mx = 0.5 * (Q.x[i] + Q.x[i1]), my = 0.5 * (Q.y[i] + Q.y[i1]);
              acc[lab] += sqrt(ex * ex + ey * ey) * (r0 + t.a * mx + t.b * my);
              touched |= 1ull << lab;
            }
          }
        }
      }
  }
  if (MODE == 0) {
    mass_out[k] = S.mass;
    intg_out[k] = S.intg;
    fval_part[k] = (wlo ? wk + wlo[k] : wk) * S.mass - S.intg;
    // row: off-diagonals sorted by column, duplicates summed, diagonal last-in
    int32_t cols[kMaxPoly + 1];
    double vals[kMaxPoly + 1];
    int nr = 0;
    double diag = 0.0;
    for (int v = 0; v < np; v++) {
      if (!((touched >> v) & 1ull)) continue;
      const int32_t j = P.lab[v];
      const double dx = yx - pos[2 * j], dy = yy - pos[2 * j + 1];
      const double val = acc[v] / (2.0 * sqrt(dx * dx + dy * dy));
      diag += val;
      int p = 0;
      while (p < nr && cols[p] < j) p++;
      if (p < nr && cols[p] == j) {  // duplicate label (degenerate edge): merge
        vals[p] -= val;
        continue;
      }
      for (int r = nr; r > p; r--) {
        cols[r] = cols[r - 1];
        vals[r] = vals[r - 1];
      }
      cols[p] = j;
      vals[p] = -val;
      nr++;
    }
    if (nr + 1 > cap_row) {  // more neighbours than the row staging holds
      overflow = true;
      nr = 0;
    }
    int cnt = 0;
    if (nr > 0) {
      int32_t *oc = row_col + k * (int64_t)cap_row;
      double *ov = row_val + k * (int64_t)cap_row;
      bool placed = false;
      for (int r = 0; r < nr; r++) {
        if (!placed && cols[r] > k) {
          oc[cnt] = (int32_t)k;
          ov[cnt++] = diag;
          placed = true;
        }
        oc[cnt] = cols[r];
        ov[cnt++] = vals[r];
      }
      if (!placed) {
        oc[cnt] = (int32_t)k;
        ov[cnt++] = diag;
      }
    }
    row_cnt[k] = cnt;
  } else {
    mass_out[k] = S.mass;
    // mode 2 keeps the moments about the Dirac
    // modes 1 and 3 return absolute moments, mode 2 keeps them about the Dirac
    const bool absm = MODE == 1 || MODE == 3;
    mom_out[2 * k] = S.momx + (absm ? yx * S.mass : 0.0);
    mom_out[2 * k + 1] = S.momy + (absm ? yy * S.mass : 0.0);
    if (MODE == 3) {
      mom2_out[3 * k] = S.sxx + 2.0 * yx * S.momx + yx * yx * S.mass;
      mom2_out[3 * k + 1] = S.syy + 2.0 * yy * S.momy + yy * yy * S.mass;
      mom2_out[3 * k + 2] = S.sxy + yx * S.momy + yy * S.momx + yx * yy * S.mass;
    }
  }
  if (overflow) atomicOr(&flags[0], 1);
  atomicAdd(&counters[0], (unsigned long long)nfrag);
  atomicMax(&counters[2], (unsigned long long)np);
}

// ---------------------------------------------------------------------------
// Cells beyond the general kernel (more than kMaxPoly - 4 vertices, or a bin
// rectangle of more than kBigRect bins: e.g. a cell in a sparse region
// bordering a dense cluster, or far displaced from its Dirac), one workgroup
// per cell.  The polygon (LDS, up to kHugePoly vertices) is clipped by the
// owners listed in the rectangle's bins, batch by batch, deepest cut first,
// each clip a parallel Sutherland-Hodgman step: every thread classifies four consecutive vertices, emits 0..2 output
// vertices for each, and a block prefix sum places them.  Fragments are the
// triangles of the cell's bins clipped by the cell's edge lines, one
// triangle per thread; Hessian edge integrals are summed in LDS.
// ---------------------------------------------------------------------------
constexpr int kHugeChunk = kHugePoly / kHugeBlock;  // vertices per thread
constexpr int kFragCap = 48;                         // fragment vertices per thread
constexpr int kHugeMaxClips = 1 << 16;               // clips of one cell

static_assert(kHugeChunk * kHugeBlock == kHugePoly, "chunking");

// Exclusive prefix sum over the block (kHugeBlock threads); *total gets the sum.
__device__ inline int huge_scan(int v, int *tmp, int *total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) tmp[wid] = x;
  __syncthreads();
  int off = 0, tot = 0;
  for (int i = 0; i < kHugeBlock / 64; i++) {
    off += (i < wid) ? tmp[i] : 0;
    tot += tmp[i];
  }
  __syncthreads();
  *total = tot;
  return off + x - v;
}

// Block-wide sum (op 0) or max (op 1) of a double.
template <int OP>
__device__ inline double huge_reduce(double v, double *tmp) {
  for (int o = 32; o > 0; o >>= 1) {
    const double y = __shfl_xor(v, o, 64);
    v = OP == 0 ? v + y : fmax(v, y);
  }
  if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = tmp[0];
  for (int i = 1; i < kHugeBlock / 64; i++) r = OP == 0 ? r + tmp[i] : fmax(r, tmp[i]);
  __syncthreads();
  return r;
}

// Clip of a thread's fragment (triangle piece, FP64 local coordinates) by the
// closed half-plane N.(X - A) >= 0 of cell edge `label`; points within
// rounding of the line count as on it.  Returns false on capacity overflow.
__device__ inline bool clip_frag(int &m, double *fx, double *fy, int *fl, double *gx, double *gy,
                                 int *gl, double Ax, double Ay, double Nx, double Ny, int label) {
  double s[kFragCap];
  int nin = 0;
  const double nn = fabs(Nx) + fabs(Ny);
  for (int i = 0; i < m; i++) {
    const double dx = fx[i] - Ax, dy = fy[i] - Ay;
    s[i] = Nx * dx + Ny * dy;
    if (fabs(s[i]) <= kSnap * nn * (fabs(fx[i]) + fabs(fy[i]) + fabs(dx) + fabs(dy))) s[i] = 0.0;
    nin += s[i] >= 0.0;
  }
  // a fragment edge lying on the line (e.g. a triangle edge along the cell
  // edge) is a piece of the cell edge
  for (int i = 0; i < m; i++)
    if (s[i] == 0.0 && s[(i + 1 == m) ? 0 : i + 1] == 0.0) fl[i] = label;
  if (nin == m) return true;
  if (nin == 0) {
    m = 0;
    return true;
  }
  int q = 0;
  for (int i = 0; i < m; i++) {
    const int i1 = (i + 1 == m) ? 0 : i + 1;
    if (q + 2 > kFragCap) return false;
    if (s[i] >= 0.0) {
      gx[q] = fx[i];
      gy[q] = fy[i];
      gl[q++] = fl[i];
      if (s[i1] < 0.0) {
        const double t = s[i] / (s[i] - s[i1]);
        gx[q] = fx[i] + t * (fx[i1] - fx[i]);
        gy[q] = fy[i] + t * (fy[i1] - fy[i]);
        gl[q++] = label;
      }
    } else if (s[i1] >= 0.0) {
      const double t = s[i] / (s[i] - s[i1]);
      gx[q] = fx[i] + t * (fx[i1] - fx[i]);
      gy[q] = fy[i] + t * (fy[i1] - fy[i]);
      gl[q++] = fl[i];
    }
  }
  for (int i = 0; i < q; i++) {
    fx[i] = gx[i];
    fy[i] = gy[i];
    fl[i] = gl[i];
  }
  m = q;
  return true;
}

// Edge labels of the bin-rectangle sides inside k_cell_huge (all negative,
// so never a neighbour): bottom, right, top, left.
constexpr int kHugeSide0 = -2;

template <int MODE>
__global__ void __launch_bounds__(kHugeBlock) k_cell_huge(
    const int32_t *__restrict__ hlist, Grid g, int64_t n, const double *__restrict__ pos,
    const double *__restrict__ w, const double *wlo, const int32_t *__restrict__ perm,
    const int32_t *__restrict__ rect, const int32_t *__restrict__ cand_start,
    const int32_t *__restrict__ cand, const int32_t *__restrict__ tbin_start,
    const int32_t *__restrict__ tbin_items, const TriData *__restrict__ tri, double *mass_out,
    double *intg_out, double *fval_part, double *mom_out, double *mom2_out, int32_t *row_cnt,
    int32_t *row_col,
    double *row_val, int cap_row, int32_t *hrow_col, double *hrow_val,
    const int32_t *__restrict__ triv, double *dval, int32_t *flags,
    unsigned long long *counters, FragOut fo) {
  __shared__ double sx[2][kHugePoly], sy[2][kHugePoly];
  __shared__ int sl[2][kHugePoly];
  __shared__ double sacc[kHugePoly];  // clip values while building, edge integrals after
  __shared__ unsigned char stouch[kHugePoly];
  __shared__ int itmp[kHugeBlock / 64];
  __shared__ double dtmp[kHugeBlock / 64];
  __shared__ int s_empty, s_best;
  const int tid = threadIdx.x;
  const int64_t k = hlist[blockIdx.x];
  const int rx0 = rect[4 * k], ry0 = rect[4 * k + 1], rx1 = rect[4 * k + 2], ry1 = rect[4 * k + 3];
  const double yx = pos[2 * k], yy = pos[2 * k + 1], wk = w[k];
  int np = 0, cur = 0;
  bool fail = false;
  double X0 = 0.0, X1 = 0.0, Y0 = 0.0, Y1 = 0.0;
  if (rx0 <= rx1) {
    X0 = g.x0 + rx0 * g.h - yx;
    X1 = g.x0 + (rx1 + 1) * g.h - yx;
    Y0 = g.y0 + ry0 * g.h - yy;
    Y1 = g.y0 + (ry1 + 1) * g.h - yy;
    if (tid == 0) {
      sx[0][0] = X0; sy[0][0] = Y0; sl[0][0] = kHugeSide0;
      sx[0][1] = X1; sy[0][1] = Y0; sl[0][1] = kHugeSide0 - 1;
      sx[0][2] = X1; sy[0][2] = Y1; sl[0][2] = kHugeSide0 - 2;
      sx[0][3] = X0; sy[0][3] = Y1; sl[0][3] = kHugeSide0 - 3;
    }
    np = 4;
  }
  if (tid == 0) s_empty = 0;
  __syncthreads();
  // Bins of the rectangle in Chebyshev rings around its centre, kHugeBlock
  // bins (one per thread) at a time; bins outside the bounding box of the
  // current polygon are skipped (the cell lies inside the polygon, so their
  // owners cannot border it).  Within a batch the polygon is clipped by the
  // candidate cutting deepest until no candidate cuts by more than rounding;
  // a half-plane already applied cannot cut again, so candidates listed in
  // several bins need no deduplication.
  const int v0 = tid * kHugeChunk;
  int nclip = 0;  // bound on the clips of one cell (every loop must end)
  const int cbx = (rx0 + rx1) >> 1, cby = (ry0 + ry1) >> 1;
  int qb[4] = {rx0, ry0, rx1, ry1};  // bin box of the polygon
  for (int r = 0; np > 0 && !fail; r++) {
    const int reach = max(max(cbx - qb[0], qb[2] - cbx), max(cby - qb[1], qb[3] - cby));
    if (r > reach) break;
    const int len = r == 0 ? 1 : 8 * r;  // ring positions, counter-clockwise from the corner
    for (int p0 = 0; p0 < len && np > 0 && !fail; p0 += kHugeBlock) {
      int32_t c0 = 0, c1 = 0;  // this thread's bin: candidates [c0, c1)
      const int pos_i = p0 + tid;
      if (pos_i < len) {
        int bx = cbx, by = cby;
        if (r > 0) {
          const int side = pos_i / (2 * r), o = pos_i % (2 * r);
          if (side == 0) { bx = cbx - r + o; by = cby - r; }
          else if (side == 1) { bx = cbx + r; by = cby - r + o; }
          else if (side == 2) { bx = cbx + r - o; by = cby + r; }
          else { bx = cbx - r; by = cby + r - o; }
        }
        if (bx >= qb[0] && bx <= qb[2] && by >= qb[1] && by <= qb[3]) {
          const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
          c0 = cand_start[b];
          c1 = cand_start[b + 1];
        }
      }
      // each (bin, candidate) entry clips at most once per batch: near-parallel
      // lines could otherwise trade rounding-level slivers forever
      uint64_t used = 0ull;
      while (true) {
        if (tid == 0) s_best = INT_MAX;
        double best = kInf;
        int32_t bj = -1, bi = -1;
        for (int32_t i = c0; i < c1; i++) {
          const int32_t j = cand[i];
          if (j == k) continue;
          if (i - c0 < 64 && ((used >> (i - c0)) & 1ull)) continue;
          const double Yx = pos[2 * j] - yx, Yy = pos[2 * j + 1] - yy;
          const double d2 = Yx * Yx + Yy * Yy;
          const double dw = wdiff(wlo, wk, k, w[j], j);  // w_k - w_j
          if (d2 == 0.0) {
            // coincident Diracs: the larger weight (then the smaller caller
            // index) hides the other
            if (dw < 0.0 || (dw == 0.0 && perm[j] < perm[k])) s_empty = 1;
            continue;
          }
          const double kk = d2 + dw;
          double dmin = kInf;
          for (int v = 0; v < np; v++) {
            const double tx = sx[cur][v] * Yx, ty = sy[cur][v] * Yy;
            const double sv = kk - 2.0 * (tx + ty);
            if (sv < -1e-14 * (fabs(kk) + 2.0 * (fabs(tx) + fabs(ty)))) dmin = fmin(dmin, sv);
          }
          const double depth = dmin / sqrt(d2);
          if (depth < best) {
            best = depth;
            bj = j;
            bi = i - c0;
          }
        }
        // deepest over the block; the smallest Dirac index among equals
        const double gbest = -huge_reduce<1>(-best, dtmp);
        if (bj >= 0 && best == gbest) atomicMin(&s_best, bj);
        __syncthreads();
        const int32_t j = s_best;
        if (s_empty) {
          np = 0;
          break;
        }
        if (j == INT_MAX) break;
        if (bj == j && bi < 64) used |= 1ull << bi;
        if (++nclip > kHugeMaxClips) {
          fail = true;
          break;
        }
        const double Yx = pos[2 * j] - yx, Yy = pos[2 * j + 1] - yy;
        const double kk = Yx * Yx + Yy * Yy + wdiff(wlo, wk, k, w[j], j);
        // clip values; those within rounding of zero are snapped onto the
        // line, so that a line through a vertex keeps that vertex instead of
        // adding a coincident copy (the region differs by measure zero)
        for (int c = 0; c < kHugeChunk; c++) {
          const int v = v0 + c;
          if (v < np) {
            const double tx = sx[cur][v] * Yx, ty = sy[cur][v] * Yy;
            const double sv = kk - 2.0 * (tx + ty);
            sacc[v] = (fabs(sv) <= 1e-14 * (fabs(kk) + 2.0 * (fabs(tx) + fabs(ty)))) ? 0.0 : sv;
          }
        }
        __syncthreads();
        // per vertex v and edge v -> v1: s_v > 0 keeps v (and adds the exit
        // point when s_v1 < 0); s_v = 0 keeps v, which starts the new edge
        // when s_v1 < 0; s_v < 0 adds the entry point when s_v1 > 0
        int emit[kHugeChunk], cnt = 0;
        for (int c = 0; c < kHugeChunk; c++) {
          const int v = v0 + c;
          emit[c] = 0;
          if (v < np) {
            const int v1 = (v + 1 == np) ? 0 : v + 1;
            const double s0 = sacc[v], s1 = sacc[v1];
            emit[c] = s0 > 0.0 ? (s1 < 0.0 ? 2 : 1) : s0 == 0.0 ? 1 : (s1 > 0.0 ? 1 : 0);
          }
          cnt += emit[c];
        }
        int total;
        int o = huge_scan(cnt, itmp, &total);
        if (total > kHugePoly) {
          fail = true;
          break;
        }
        const int nx = cur ^ 1;
        for (int c = 0; c < kHugeChunk; c++) {
          const int v = v0 + c;
          if (emit[c] == 0) continue;
          const int v1 = (v + 1 == np) ? 0 : v + 1;
          const double s0 = sacc[v], s1 = sacc[v1];
          if (s0 >= 0.0) {
            sx[nx][o] = sx[cur][v];
            sy[nx][o] = sy[cur][v];
            sl[nx][o++] = (s0 == 0.0 && s1 < 0.0) ? j : sl[cur][v];
            if (s0 > 0.0 && s1 < 0.0) {  // exit point: the new edge starts here
              const double t = s0 / (s0 - s1);
              sx[nx][o] = sx[cur][v] + t * (sx[cur][v1] - sx[cur][v]);
              sy[nx][o] = sy[cur][v] + t * (sy[cur][v1] - sy[cur][v]);
              sl[nx][o++] = j;
            }
          } else {  // entry point on edge v
            const double t = s0 / (s0 - s1);
            sx[nx][o] = sx[cur][v] + t * (sx[cur][v1] - sx[cur][v]);
            sy[nx][o] = sy[cur][v] + t * (sy[cur][v1] - sy[cur][v]);
            sl[nx][o++] = sl[cur][v];
          }
        }
        __syncthreads();
        cur = nx;
        np = total < 3 ? 0 : total;  // a point or a segment: no area
        if (np == 0) break;
      }
      // shrink the bin box to the polygon's
      if (np > 0 && !fail) {
        double ex0 = kInf, ey0 = kInf, ex1 = -kInf, ey1 = -kInf;
        for (int c = 0; c < kHugeChunk; c++) {
          const int v = v0 + c;
          if (v >= np) continue;
          ex0 = fmin(ex0, sx[cur][v]);
          ex1 = fmax(ex1, sx[cur][v]);
          ey0 = fmin(ey0, sy[cur][v]);
          ey1 = fmax(ey1, sy[cur][v]);
        }
        ex0 = -huge_reduce<1>(-ex0, dtmp);
        ey0 = -huge_reduce<1>(-ey0, dtmp);
        ex1 = huge_reduce<1>(ex1, dtmp);
        ey1 = huge_reduce<1>(ey1, dtmp);
        qb[0] = max(qb[0], bin_coord(ex0 + yx, g.x0, g.h, g.G));
        qb[1] = max(qb[1], bin_coord(ey0 + yy, g.y0, g.h, g.G));
        qb[2] = min(qb[2], bin_coord(ex1 + yx, g.x0, g.h, g.G));
        qb[3] = min(qb[3], bin_coord(ey1 + yy, g.y0, g.h, g.G));
      }
    }
  }
  if (fail) {
    if (tid == 0) {
      atomicOr(&flags[0], 1);
      counters[7] = ((unsigned long long)(uint32_t)k << 32) | ((unsigned long long)np << 16) |
                    (unsigned long long)min(nclip, 0xffff);
    }
    return;
  }
  // edge lines (a point A on the edge and an inward normal N) into the
  // spare buffer; edge integrals start at zero
  const int nb_ = cur ^ 1;
  double bx0 = kInf, by0 = kInf, bx1 = -kInf, by1 = -kInf;
  for (int c = 0; c < kHugeChunk; c++) {
    const int v = v0 + c;
    if (v >= np) continue;
    const int lab = sl[cur][v];
    double Nx, Ny;
    if (lab >= 0) {
      Nx = yx - pos[2 * lab];
      Ny = yy - pos[2 * lab + 1];
    } else {
      const int side = kHugeSide0 - lab;  // 0 bottom, 1 right, 2 top, 3 left
      Nx = side == 1 ? -1.0 : side == 3 ? 1.0 : 0.0;
      Ny = side == 0 ? 1.0 : side == 2 ? -1.0 : 0.0;
    }
    sx[nb_][v] = Nx;
    sy[nb_][v] = Ny;
    sacc[v] = 0.0;
    stouch[v] = 0;
    bx0 = fmin(bx0, sx[cur][v]);
    bx1 = fmax(bx1, sx[cur][v]);
    by0 = fmin(by0, sy[cur][v]);
    by1 = fmax(by1, sy[cur][v]);
  }
  bx0 = -huge_reduce<1>(-bx0, dtmp) + yx;
  by0 = -huge_reduce<1>(-by0, dtmp) + yy;
  bx1 = huge_reduce<1>(bx1, dtmp) + yx;
  by1 = huge_reduce<1>(by1, dtmp) + yy;
  FragSums S;
  int nfrag = 0;
  bool overflow = false;
  if (np > 0) {
    const int qx0 = max(bin_coord(bx0, g.x0, g.h, g.G), rx0);
    const int qx1 = min(bin_coord(bx1, g.x0, g.h, g.G), rx1);
    const int qy0 = max(bin_coord(by0, g.y0, g.h, g.G), ry0);
    const int qy1 = min(bin_coord(by1, g.y0, g.h, g.G), ry1);
    const int wx = qx1 - qx0 + 1;
    const int64_t nbins = (qx0 <= qx1 && qy0 <= qy1) ? (int64_t)wx * (qy1 - qy0 + 1) : 0;
    double fx[kFragCap], fy[kFragCap], gx[kFragCap], gy[kFragCap];
    int fl[kFragCap], gl[kFragCap];
    for (int64_t ib = tid; ib < nbins; ib += kHugeBlock) {
      const int bx = qx0 + (int)(ib % wx), by = qy0 + (int)(ib / wx);
      const int64_t b = morton2((uint32_t)bx, (uint32_t)by);
      for (int32_t q = tbin_start[b]; q < tbin_start[b + 1]; q++) {
        const TriData t = tri[tbin_items[q] >> kTriShift];
        double tx0, ty0, tx1, ty1;
        tri_bbox(t, tx0, ty0, tx1, ty1);
        if (tx1 < bx0 || tx0 > bx1 || ty1 < by0 || ty0 > by1) continue;
        // each triangle once: in the bin of the lower-left corner of the
        // overlap of the two bounding boxes
        const int ox = max(bin_coord(fmax(tx0, bx0), g.x0, g.h, g.G), qx0);
        const int oy = max(bin_coord(fmax(ty0, by0), g.y0, g.h, g.G), qy0);
        if (ox != bx || oy != by) continue;
        int m = 3;
        for (int c = 0; c < 3; c++) {
          fx[c] = t.x[c] - yx;
          fy[c] = t.y[c] - yy;
          fl[c] = -1;  // triangle edge
        }
        for (int v = 0; v < np && m > 0; v++)
          if (!clip_frag(m, fx, fy, fl, gx, gy, gl, sx[cur][v], sy[cur][v], sx[nb_][v],
                         sy[nb_][v], v)) {
            overflow = true;
            m = 0;
          }
        if (m < 3) continue;
        {
          double ar2 = 0.0, xlo = kInf, xhi = -kInf, ylo = kInf, yhi = -kInf, cm = 0.0;
          for (int i = 0; i < m; i++) {
            const int i1 = (i + 1 == m) ? 0 : i + 1;
            ar2 += fx[i] * fy[i1] - fx[i1] * fy[i];
            xlo = fmin(xlo, fx[i]);
            xhi = fmax(xhi, fx[i]);
            ylo = fmin(ylo, fy[i]);
            yhi = fmax(yhi, fy[i]);
            cm = fmax(cm, fmax(fabs(fx[i]), fabs(fy[i])));
          }
          if (!(0.5 * ar2 > 1e-13 * ((xhi - xlo) + (yhi - ylo)) * cm)) continue;
        }
        nfrag++;
        if (MODE == 1 && fo.count != nullptr) {
          auto gx = [&](int i) { return fx[i]; };
          auto gy = [&](int i) { return fy[i]; };
          const double eps = frag_eps_of(m, gx, gy);
          const int md = frag_distinct(m, eps, gx, gy);
          unsigned long long f, v;
          frag_reserve(fo, md, f, v);
          frag_write(fo, f, v, md, perm[k], tbin_items[q] >> kTriShift, yx, yy, m, eps, gx, gy);
        }
        double dv[3] = {0.0, 0.0, 0.0};
        frag_integrals<MODE>(fx, fy, m, t, yx, yy, wk, S, dv);
        if (MODE == 2) {
          const int64_t ti = tbin_items[q] >> kTriShift;
          for (int c = 0; c < 3; c++) atomicAdd(&dval[triv[3 * ti + c]], dv[c]);
        }
        if (MODE == 0) {
          const double r0 = t.a * yx + t.b * yy + t.c;
          for (int i = 0; i < m; i++) {
            const int lab = fl[i];
            if (lab < 0 || sl[cur][lab] < 0) continue;
            const int i1 = (i + 1 == m) ? 0 : i + 1;
            const double ex = fx[i1] - fx[i], ey = fy[i1] - fy[i];
            if (ex == 0.0 && ey == 0.0) continue;
            const double mx = 0.5 * (fx[i] + fx[i1]), my = 0.5 * (fy[i] + fy[i1]);
            atomicAdd(&sacc[lab], sqrt(ex * ex + ey * ey) * (r0 + t.a * mx + t.b * my));
            stouch[lab] = 1;
          }
        }
      }
    }
  }
  const double mass = huge_reduce<0>(S.mass, dtmp);
  const double intg = huge_reduce<0>(S.intg, dtmp);
  const double momx = huge_reduce<0>(S.momx, dtmp);
  const double momy = huge_reduce<0>(S.momy, dtmp);
  double sxx = 0.0, syy = 0.0, sxy = 0.0;
  if (MODE == 3) {
    sxx = huge_reduce<0>(S.sxx, dtmp);
    syy = huge_reduce<0>(S.syy, dtmp);
    sxy = huge_reduce<0>(S.sxy, dtmp);
  }
  const int nfr = (int)huge_reduce<0>((double)nfrag, dtmp);
  if (__syncthreads_or(overflow)) {
    if (tid == 0) atomicOr(&flags[0], 2);  // fragment capacity
    return;
  }
  if (MODE == 0) {
    // row: neighbour edges that carry a fragment edge; repeated labels
    // (degenerate edges) are merged into their first occurrence, entries
    // ranked by column, the diagonal inserted in order
    int keep[kHugeChunk];
    double val[kHugeChunk];
    double dsum = 0.0;
    for (int c = 0; c < kHugeChunk; c++) {
      const int v = v0 + c;
      keep[c] = 0;
      val[c] = 0.0;
      if (v >= np || !stouch[v] || sl[cur][v] < 0) continue;
      const int32_t j = sl[cur][v];
      const double dx = yx - pos[2 * j], dy = yy - pos[2 * j + 1];
      const double e = sacc[v] / (2.0 * sqrt(dx * dx + dy * dy));
      dsum += e;
      bool first = true;
      for (int u = 0; u < v && first; u++) first = !(stouch[u] && sl[cur][u] == j);
      keep[c] = first;
    }
    __syncthreads();
    // merged values: sum over the repeated labels
    for (int c = 0; c < kHugeChunk; c++) {
      const int v = v0 + c;
      if (!keep[c]) continue;
      const int32_t j = sl[cur][v];
      const double dx = yx - pos[2 * j], dy = yy - pos[2 * j + 1];
      const double inv = 1.0 / (2.0 * sqrt(dx * dx + dy * dy));
      double s = 0.0;
      for (int u = v; u < np; u++)
        if (stouch[u] && sl[cur][u] == j) s += sacc[u] * inv;
      val[c] = -s;
    }
    const double diag = huge_reduce<0>(dsum, dtmp);
    // kept flags to LDS (stouch is no longer needed) for the ranks
    for (int c = 0; c < kHugeChunk; c++) {
      const int v = v0 + c;
      if (v < np) stouch[v] = (unsigned char)keep[c];
    }
    __syncthreads();
    int nk = 0;
    for (int c = 0; c < kHugeChunk; c++) nk += keep[c];
    int nkept;
    (void)huge_scan(nk, itmp, &nkept);
    const int cnt = nkept > 0 ? nkept + 1 : 0;
    int32_t *oc = row_col + k * (int64_t)cap_row;
    double *ov = row_val + k * (int64_t)cap_row;
    if (cnt > cap_row) {
      // long row: staged in a slot of the long-row pool; the first regular
      // entry points there
      if (tid == 0) s_best = (int)atomicAdd(&counters[8], 1ull);
      __syncthreads();
      const int lslot = s_best;
      if (lslot >= kLongRows) {
        if (tid == 0) atomicOr(&flags[0], 4);
        return;
      }
      if (tid == 0) oc[0] = lslot;
      oc = hrow_col + (int64_t)lslot * kHugeRow;
      ov = hrow_val + (int64_t)lslot * kHugeRow;
    }
    for (int c = 0; c < kHugeChunk; c++) {
      if (!keep[c]) continue;
      const int32_t j = sl[cur][v0 + c];
      int rank = 0;
      for (int u = 0; u < np; u++) rank += (stouch[u] && sl[cur][u] < j);
      const int p = rank + (j > k ? 1 : 0);
      oc[p] = j;
      ov[p] = val[c];
    }
    if (cnt > 0) {
      int below = 0;
      for (int c = 0; c < kHugeChunk; c++) below += keep[c] && sl[cur][v0 + c] < k;
      int nbelow;
      (void)huge_scan(below, itmp, &nbelow);
      if (tid == 0) {
        oc[nbelow] = (int32_t)k;
        ov[nbelow] = diag;
      }
    }
    if (tid == 0) {
      row_cnt[k] = cnt;
      mass_out[k] = mass;
      intg_out[k] = intg;
      fval_part[k] = (wlo ? wk + wlo[k] : wk) * mass - intg;
    }
  } else if (tid == 0) {
    mass_out[k] = mass;
    const bool absm = MODE == 1 || MODE == 3;
    mom_out[2 * k] = momx + (absm ? yx * mass : 0.0);
    mom_out[2 * k + 1] = momy + (absm ? yy * mass : 0.0);
    if (MODE == 3) {
      mom2_out[3 * k] = sxx + 2.0 * yx * momx + yx * yx * mass;
      mom2_out[3 * k + 1] = syy + 2.0 * yy * momy + yy * yy * mass;
      mom2_out[3 * k + 2] = sxy + yx * momy + yy * momx + yx * yy * mass;
    }
  }
  if (tid == 0) {
    atomicAdd(&counters[0], (unsigned long long)nfr);
    atomicMax(&counters[2], (unsigned long long)np);
  }
}

// CSR rows of the cells evaluated by the general kernels (pn < 0), staged per
// Dirac in row_*; rows longer than cap_row entries (from k_cell_huge) are read
// from the long-row pool hrow_* at the slot stored in their first entry.
__global__ void k_csr_fill(int64_t n, const int32_t *pn, const int32_t *row_cnt,
                           const int32_t *row_col, const double *row_val, int cap_row,
                           const int32_t *hrow_col, const double *hrow_val, const int32_t *ptr,
                           int32_t *col, double *val) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n || pn[k] >= 0) return;
  const int c = row_cnt[k];
  const int32_t o = ptr[k];
  const int32_t *rc = row_col + k * (int64_t)cap_row;
  const double *rv = row_val + k * (int64_t)cap_row;
  if (c > cap_row) {
    const int64_t s = rc[0];
    rc = hrow_col + s * kHugeRow;
    rv = hrow_val + s * kHugeRow;
  }
  for (int i = 0; i < c; i++) {
    col[o + i] = rc[i];
    val[o + i] = rv[i];
  }
}

// Deterministic two-stage sum: partials per block, then one block.
__global__ void __launch_bounds__(256) k_sum_partials(const double *x, int64_t n, double *part) {
  __shared__ double s[256];
  double a = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a += x[i];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

hipError_t device_sum(ma_engine *e, const double *x, int64_t n, double *d_out) {
  MA_HIP_RET(e->eb.red_tmp.ensure(2048));
  hipLaunchKernelGGL(k_sum_partials, dim3(1024), dim3(256), 0, e->stream, x, n, e->eb.red_tmp.p);
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, e->stream, e->eb.red_tmp.p,
                     (int64_t)1024, d_out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// One evaluation.
// ---------------------------------------------------------------------------
ma_status run_cells(ma_engine *e, int mode, bool fp32, int32_t *npairs_out, int32_t *ngeneral_out);
ma_status fill_rows(ma_engine *e);
ma_status refine_candidates(ma_engine *e, int64_t total);

// Candidate owners of every domain bin (of the bins with mask[b] set, when
// mask is given) and the bin rectangles of the Diracs marked pn < 0 (see
// k_plane, k_cand_list, k_rect).
ma_status run_bin_candidates(ma_engine *e, const int32_t *pn, const unsigned char *mask) {
  const Grid &g = e->grid;
  const int64_t n = e->n;
  EvalBuffers &B = e->eb;
  PyrOff po{};
  for (int l = 0; l <= g.L; l++) po.o[l] = e->pyr_off[l];
  const Plane *pl = reinterpret_cast<const Plane *>(B.plane.p);
  MA_HIP_TRY(B.cand_cnt.ensure((size_t)g.nbins + 1));
  int32_t total = 0;
  // walks of the pyramid per bin: owners and counts (keeping the first
  // kCandStage candidates), then the lists of the bins with more (one walk
  // that records while the bound is still falling, and filters afterwards,
  // measured slower: it records far more)
  const dim3 grid(nblocks(g.nbins, kCellGroups)), block(kCellThreads);
  MA_HIP_TRY(B.cstage.ensure((size_t)g.nbins * kCandStage));
  hipLaunchKernelGGL(k_cand_list<false>, grid, block, 0, e->stream, g, e->tbin_start.p,
                     e->bin_start.p, e->pos.p, B.w_s.p, pl, po, B.owner.p, B.cand_cnt.p,
                     (int32_t *)nullptr, (int32_t *)nullptr, B.cstage.p, B.counters.p, mask);
  // offsets, and the total to the host
  MA_HIP_TRY(exclusive_scan(e, B.cand_cnt.p, B.cand_cnt.p, g.nbins));
  MA_HIP_TRY(read_back(e, {{&total, B.cand_cnt.p + g.nbins, sizeof(int32_t)}}));
  MA_HIP_TRY(B.cand.ensure((size_t)total + 1));
  MA_HIP_TRY(B.cbin.ensure((size_t)total + 1));
  hipLaunchKernelGGL(k_cand_list<true>, grid, block, 0, e->stream, g, e->tbin_start.p,
                     e->bin_start.p, e->pos.p, B.w_s.p, pl, po, B.owner.p, B.cand_cnt.p, B.cand.p,
                     B.cbin.p, B.cstage.p, B.counters.p, mask);
  if (total > 0 && e->refine) {
    // keep only the exact owners of each bin (refine_candidates), then
    // compact the lists
    MA_HIP_TRY(B.ckeep.ensure((size_t)total + 1));
    MA_HIP_TRY(B.cand2.ensure((size_t)total + 1));
    MA_HIP_TRY(B.cstart2.ensure((size_t)g.nbins + 1));
    ma_status rs = refine_candidates(e, total);
    if (rs != MA_OK) return rs;
    MA_HIP_TRY(exclusive_scan(e, B.ckeep.p, B.ckeep.p, total));
    hipLaunchKernelGGL(k_refine_starts, dim3(nblocks(g.nbins + 1)), dim3(kBlock), 0, e->stream,
                       g.nbins, B.cand_cnt.p, B.ckeep.p, B.cstart2.p);
    hipLaunchKernelGGL(k_refine_move, dim3(nblocks(total)), dim3(kBlock), 0, e->stream,
                       (int64_t)total, B.ckeep.p, B.cand.p, B.cand2.p);
    B.cand.swap(B.cand2);
    B.cand_cnt.swap(B.cstart2);
  }
  hipLaunchKernelGGL(k_rect_init, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, B.rect.p, n);
  hipLaunchKernelGGL(k_rect, dim3(nblocks(g.nbins)), dim3(kBlock), 0, e->stream, g,
                     e->tbin_start.p, B.cand_cnt.p, B.cand.p, pn, B.rect.p);
  MA_HIP_TRY(hipGetLastError());
  return MA_OK;
}

ma_status evaluate(ma_engine *e, int mode, double *fval_out, bool fp32) {
  const Grid &g = e->grid;
  const int64_t n = e->n;
  EvalBuffers &B = e->eb;
  // the outputs of the previous evaluation are overwritten from here on
  e->have_eval = false;
  e->have_hessian = false;
  // pyramid
  e->pyr_off.assign((size_t)g.L + 1, 0);
  int64_t tot = 0;
  for (int l = 0; l <= g.L; l++) {
    e->pyr_off[l] = tot;
    tot += (int64_t)1 << (2 * (g.L - l));
  }
  PyrOff po{};
  for (int l = 0; l <= g.L; l++) po.o[l] = e->pyr_off[l];
  MA_HIP_TRY(B.pyr.ensure((size_t)tot));
  MA_HIP_TRY(B.pyr3.ensure((size_t)tot));
  MA_HIP_TRY(B.cand_cnt.ensure((size_t)g.nbins + 1));
  MA_HIP_TRY(B.owner.ensure((size_t)g.nbins));
  MA_HIP_TRY(B.rect.ensure((size_t)(4 * n)));
  MA_HIP_TRY(B.mass_s.ensure((size_t)n));
  MA_HIP_TRY(B.intg_s.ensure((size_t)n));
  MA_HIP_TRY(B.fval_part.ensure((size_t)n));
  MA_HIP_TRY(B.mom_s.ensure((size_t)(2 * n)));
  MA_HIP_TRY(B.row_cnt.ensure((size_t)n + 1));
  MA_HIP_TRY(B.flags.ensure(4));
  MA_HIP_TRY(B.counters.ensure(kCounters));
  MA_HIP_TRY(B.red_tmp.ensure(2048));
  if (!e->owner_init) {
    hipLaunchKernelGGL(k_fill_i32, dim3(nblocks(g.nbins)), dim3(kBlock), 0, e->stream,
                       B.owner.p, -1, g.nbins);
    e->owner_init = true;
  }
  MA_HIP_TRY(hipEventRecord(e->ev[0], e->stream));
  MA_HIP_TRY(B.plane.ensure((size_t)(4 * tot)));
  MA_HIP_TRY(B.node_sums.ensure((size_t)(4 * tot)));
  for (int lev = 0; lev < g.L || lev == 0; lev += 2) {
    const int step = std::min(2, g.L - lev);
    hipLaunchKernelGGL(k_plane, dim3(nblocks((int64_t)1 << (2 * (g.L - lev - step)), kCellGroups)),
                       dim3(kCellThreads), 0, e->stream, g, lev, step, e->bin_start.p, e->pos.p,
                       B.w_s.p, po, reinterpret_cast<Plane *>(B.plane.p),
                       reinterpret_cast<NodeSums *>(B.node_sums.p), B.pyr.p);
  }
  hipLaunchKernelGGL(k_pyr3, dim3(nblocks(tot)), dim3(kBlock), 0, e->stream, g, po, tot, B.pyr.p,
                     B.pyr3.p);
  MA_HIP_TRY(hipEventRecord(e->ev[1], e->stream));
  MA_HIP_TRY(hipMemsetAsync(B.flags.p, 0, sizeof(int32_t) * 4, e->stream));
  MA_HIP_TRY(hipMemsetAsync(B.counters.p, 0, sizeof(unsigned long long) * kCounters, e->stream));
  MA_HIP_TRY(hipEventRecord(e->ev[2], e->stream));
  int32_t npairs = 0, ngen = 0;
  ma_status cs = run_cells(e, mode, fp32, &npairs, &ngen);
  if (cs != MA_OK) return cs;
  if (ngen > 0 && mode == 0) {  // staging of the general kernels' rows
    MA_HIP_TRY(B.row_col.ensure((size_t)n * e->cap_row));
    MA_HIP_TRY(B.row_val.ensure((size_t)n * e->cap_row));
  }
  int32_t nhuge = 0;
  const int32_t *hl = nullptr;  // list of the cells for k_cell_huge
  if (ngen > 0 && ((ngen <= kHugeRoute && e->force_general != 1) || e->fo.count != nullptr)) {
    // few cells: one workgroup each beats one thread each (whose candidate
    // loops run at memory latency).  Fragment output takes this route for
    // all of them: the general kernel can hand a cell on to the workgroup
    // kernel after it has met some of its fragments.
    nhuge = ngen;
    hl = B.glist.p;
  } else if (ngen > 0) {
    // cells that overflowed the fast path
    MA_HIP_TRY(B.hlist.ensure((size_t)n + 1));
    hl = B.hlist.p;
    MA_HIP_TRY(hipMemsetAsync(B.hlist.p + n, 0, sizeof(int32_t), e->stream));
    auto kern = mode == 0 ? k_cells_general<0> : mode == 1 ? k_cells_general<1>
                : mode == 2 ? k_cells_general<2> : k_cells_general<3>;
    hipLaunchKernelGGL(kern, dim3(nblocks(ngen)), dim3(kBlock), 0, e->stream, B.glist.p,
                       B.glist.p + n, g, n, e->pos.p, B.w_s.p, B.wlo(), e->perm.p, B.rect.p,
                       B.cand_cnt.p,
                       B.cand.p, e->tbin_start.p, e->tbin_items.p, e->tri.p,
                       B.mass_s.p, B.intg_s.p, B.fval_part.p, B.mom_s.p, B.mom2_s.p, B.row_cnt.p,
                       B.row_col.p, B.row_val.p, e->cap_row, e->triv.p, B.dval.p, B.hlist.p,
                       (int)(e->force_general == 2), B.flags.p, B.counters.p);
    MA_HIP_TRY(read_back(e, {{&nhuge, B.hlist.p + n, sizeof(int32_t)}}));
  }
  if (nhuge > 0) {
    // the few cells beyond the general kernel: one workgroup each
    if (mode == 0) {
      MA_HIP_TRY(B.hrow_col.ensure((size_t)kLongRows * kHugeRow));
      MA_HIP_TRY(B.hrow_val.ensure((size_t)kLongRows * kHugeRow));
    }
    auto kern = mode == 0 ? k_cell_huge<0> : mode == 1 ? k_cell_huge<1>
                : mode == 2 ? k_cell_huge<2> : k_cell_huge<3>;
    hipLaunchKernelGGL(kern, dim3(nhuge), dim3(kHugeBlock), 0, e->stream, hl, g, n,
                       e->pos.p, B.w_s.p, B.wlo(), e->perm.p, B.rect.p, B.cand_cnt.p, B.cand.p,
                       e->tbin_start.p, e->tbin_items.p, e->tri.p, B.mass_s.p, B.intg_s.p,
                       B.fval_part.p, B.mom_s.p, B.mom2_s.p, B.row_cnt.p, B.row_col.p, B.row_val.p,
                       e->cap_row, B.hrow_col.p, B.hrow_val.p, e->triv.p, B.dval.p, B.flags.p,
                       B.counters.p, mode == 1 ? e->fo : FragOut{});
  }
  MA_HIP_TRY(hipEventRecord(e->ev[6], e->stream));
  if (mode == 0) {
    MA_HIP_TRY(B.csr_ptr.ensure((size_t)n + 1));
    MA_HIP_TRY(exclusive_scan(e, B.row_cnt.p, B.csr_ptr.p, n));
    int32_t nnz = 0;
    MA_HIP_TRY(read_back(e, {{&nnz, B.csr_ptr.p + n, sizeof(int32_t)}}));
    MA_HIP_TRY(B.csr_col.ensure((size_t)nnz + 1));
    MA_HIP_TRY(B.csr_val.ensure((size_t)nnz + 1));
    const ma_status rs = fill_rows(e);
    if (rs != MA_OK) return rs;
    if (ngen > 0)
      hipLaunchKernelGGL(k_csr_fill, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, n, B.pn.p,
                         B.row_cnt.p, B.row_col.p, B.row_val.p, e->cap_row, B.hrow_col.p,
                         B.hrow_val.p, B.csr_ptr.p, B.csr_col.p, B.csr_val.p);
    MA_HIP_TRY(device_sum(e, B.fval_part.p, n, B.red_tmp.p + 1024));
    e->nnz = nnz;  // sizes the CSR buffers now holding this pass's rows
  }
  MA_HIP_TRY(hipEventRecord(e->ev[7], e->stream));
  MA_HIP_TRY(hipGetLastError());
  int32_t fl[4];
  unsigned long long ct[kCounters];
  double fv = 0.0;
  MA_HIP_TRY(read_back(e, {{fl, B.flags.p, sizeof fl},
                           {ct, B.counters.p, sizeof ct},
                           {&fv, B.red_tmp.p + 1024, mode == 0 ? sizeof fv : 0}}));
  float t[7] = {0, 0, 0, 0, 0, 0, 0}, tc = 0.0f;
  for (int i = 0; i < 7; i++) MA_HIP_TRY(hipEventElapsedTime(&t[i], e->ev[i], e->ev[i + 1]));
  if (e->ran_candidates) MA_HIP_TRY(hipEventElapsedTime(&tc, e->ev[8], e->ev[9]));
  float tk = 0.0f;
  MA_HIP_TRY(hipEventElapsedTime(&tk, e->ev[10], e->ev[11]));
  e->info.ms_cell_kernel = tk;
  e->info.ms_weights = t[0];
  e->info.ms_candidates = tc;
  e->info.ms_cell_build = t[2];
  e->info.ms_pairs = t[3];
  e->info.ms_frag = t[4];
  e->info.ms_cells = t[2] + t[3] + t[4] + t[5];
  e->info.ms_assemble = t[6];
  e->info.ms_total = t[0] + t[1] + t[2] + t[3] + t[4] + t[5] + t[6];
  for (int b = 0; b < kCounterStripes; b++) {
    ct[0] += *counter_stripe(ct, 0, b);
    ct[4] += *counter_stripe(ct, 1, b);
  }
  e->info.nfrag = (int64_t)ct[0];
  e->info.ncand = (int64_t)ct[1];
  e->info.max_poly = (int64_t)ct[2];
  e->info.empty_cells = (int64_t)ct[3];
  e->info.nvert = (int64_t)ct[4];
  e->info.nredecide = (int64_t)ct[5];
  e->info.npairs = npairs;
  e->info.ngeneral = ngen;
  e->info.nhuge = nhuge;
  e->info.nnz = e->nnz;
  if (fl[0]) {
    e->err = (fl[0] & 4) ? "more than " + std::to_string(kLongRows) +
                               " Hessian rows longer than " + std::to_string(kMaxRow) + " entries"
           : (fl[0] & 2) ? "a cell x triangle fragment exceeded " + std::to_string(kFragCap) +
                               " vertices"
                         : "a cell polygon exceeded " + std::to_string(kHugePoly) +
                               " vertices (or " + std::to_string(kHugeMaxClips) +
                               " clips): Morton cell " + std::to_string(ct[7] >> 32) + ", " +
                               std::to_string((ct[7] >> 16) & 0xffff) + " vertices after " +
                               std::to_string(ct[7] & 0xffff) + " clips";
    return MA_CAPACITY;
  }
  e->have_eval = true;
  e->have_hessian = mode == 0;
  if (!fp32 || mode != 0) e->far_valid = true;  // eb.far written by the FP64 cell kernel
  if (fval_out) *fval_out = fv;
  return MA_OK;
}

// ---------------------------------------------------------------------------
// CSR in the caller's order.
// ---------------------------------------------------------------------------
__global__ void k_caller_cnt(int64_t n, const int32_t *iperm, const int32_t *ptr, int32_t *cnt) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t k = iperm[i];
  cnt[i] = ptr[k + 1] - ptr[k];
}
// 16 lanes per row: every entry goes to its rank among the row's columns (all
// different).  Rows of up to 16 entries stay in registers; longer ones, rare,
// count ranks from memory.  (A thread per row that sorted by insertion in the
// output waited for its own stores: N = 1000 19.9 us instead of 3.7.)
__global__ void __launch_bounds__(kCellThreads)
    k_caller_fill(int64_t n, const int32_t *iperm, const int32_t *perm, const int32_t *ptr,
                  const int32_t *col, const double *val, const int32_t *optr, int32_t *ocol,
                  double *oval) {
  const int l = (int)threadIdx.x % kGroup, base = (int)threadIdx.x % 64 - l;
  const int64_t i = (int64_t)blockIdx.x * kCellGroups + threadIdx.x / kGroup;
  if (i >= n) return;
  const int32_t k = iperm[i];
  const int32_t s = ptr[k], c = ptr[k + 1] - s, o = optr[i];
  if (c <= kGroup) {
    const bool have = l < c;
    const int32_t j = have ? perm[col[s + l]] : INT32_MAX;
    int rank = 0;
    for (int q = 0; q < c; q++) rank += row_get(j, 4 * base, q) < j;
    if (have) {
      ocol[o + rank] = j;
      oval[o + rank] = val[s + l];
    }
    return;
  }
  for (int32_t r = l; r < c; r += kGroup) {
    const int32_t j = perm[col[s + r]];
    int rank = 0;
    for (int32_t q = 0; q < c; q++) rank += perm[col[s + q]] < j;
    ocol[o + rank] = j;
    oval[o + rank] = val[s + r];
  }
}

hipError_t csr_to_caller(ma_engine *e, int32_t *rowptr, int32_t *col, double *val) {
  const int64_t n = e->n;
  DBuf<int32_t> &optr = e->cb.ptr, &ocol = e->cb.col;
  DBuf<double> &oval = e->cb.val;
  MA_HIP_RET(optr.ensure((size_t)n + 1));
  MA_HIP_RET(ocol.ensure((size_t)e->nnz + 1));
  MA_HIP_RET(oval.ensure((size_t)e->nnz + 1));
  hipLaunchKernelGGL(k_caller_cnt, dim3(nblocks(n)), dim3(kBlock), 0, e->stream, n, e->iperm.p,
                     e->eb.csr_ptr.p, optr.p);
  MA_HIP_RET(exclusive_scan(e, optr.p, optr.p, n));
  hipLaunchKernelGGL(k_caller_fill, dim3(nblocks(n, kCellGroups)), dim3(kCellThreads), 0,
                     e->stream, n, e->iperm.p,
                     e->perm.p, e->eb.csr_ptr.p, e->eb.csr_col.p, e->eb.csr_val.p, optr.p,
                     ocol.p, oval.p);
  MA_HIP_RET(hipMemcpyAsync(rowptr, optr.p, sizeof(int32_t) * (n + 1), hipMemcpyDeviceToHost,
                            e->stream));
  MA_HIP_RET(hipMemcpyAsync(col, ocol.p, sizeof(int32_t) * e->nnz, hipMemcpyDeviceToHost,
                            e->stream));
  MA_HIP_RET(hipMemcpyAsync(val, oval.p, sizeof(double) * e->nnz, hipMemcpyDeviceToHost,
                            e->stream));
  return hipStreamSynchronize(e->stream);
}

}  // namespace ma
