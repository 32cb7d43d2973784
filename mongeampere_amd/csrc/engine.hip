// Engine object, C ABI entry points and the device-resident damped Newton
// solver (include/MA/optimal_transport.hpp:41-193 behaviour) with a
// Jacobi-preconditioned conjugate gradient on the gauge-fixed Laplacian.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <mutex>

#include "geom_common.h"
#include "lanes.h"

namespace ma {

hipError_t device_sum(ma_engine *e, const double *x, int64_t n, double *d_out);

constexpr int kVB = 256;      // threads per block for vector kernels
constexpr int kVGrid = 512;   // fixed grid => fixed number of partial sums

// ---------------------------------------------------------------------------
// Mesh preparation: ccw orientation and per-face linear density a x + b y + c
// (the plane through the three vertex values; include/MA/functions.hpp:55-80).
// ---------------------------------------------------------------------------
__global__ void k_tri_prep(const double *vxy, const double *vval, const int32_t *tri, int64_t nt,
                           TriData *out, int32_t *triv, float4 *tbox, int32_t *bad) {
  int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (f >= nt) return;
  int32_t id[3] = {tri[3 * f], tri[3 * f + 1], tri[3 * f + 2]};
  double x[3], y[3], v[3];
  for (int k = 0; k < 3; k++) {
    x[k] = vxy[2 * id[k]];
    y[k] = vxy[2 * id[k] + 1];
    v[k] = vval[id[k]];
  }
  double D = (x[1] - x[0]) * (y[2] - y[0]) - (x[2] - x[0]) * (y[1] - y[0]);
  if (D < 0) {
    double t;
    t = x[1]; x[1] = x[2]; x[2] = t;
    t = y[1]; y[1] = y[2]; y[2] = t;
    t = v[1]; v[1] = v[2]; v[2] = t;
    int32_t s = id[1]; id[1] = id[2]; id[2] = s;
    D = -D;
  }
  if (!(D > 0)) atomicOr(bad, 1);
  TriData T;
  for (int k = 0; k < 3; k++) {
    T.x[k] = x[k];
    T.y[k] = y[k];
  }
  const double f1 = v[1] - v[0], f2 = v[2] - v[0];
  const double ex1 = x[1] - x[0], ey1 = y[1] - y[0], ex2 = x[2] - x[0], ey2 = y[2] - y[0];
  T.a = (f1 * ey2 - f2 * ey1) / D;
  T.b = (ex1 * f2 - ex2 * f1) / D;
  T.c = v[0] - T.a * x[0] - T.b * y[0];
  out[f] = T;
  for (int k = 0; k < 3; k++) triv[3 * f + k] = id[k];
  tbox[f] = make_float4(__double2float_rd(fmin(x[0], fmin(x[1], x[2]))),
                        __double2float_rd(fmin(y[0], fmin(y[1], y[2]))),
                        __double2float_ru(fmax(x[0], fmax(x[1], x[2]))),
                        __double2float_ru(fmax(y[0], fmax(y[1], y[2]))));
}

// ---------------------------------------------------------------------------
// Vector kernels (grid-stride, fixed grid, deterministic partial sums).
// ---------------------------------------------------------------------------
__device__ inline double block_sum(double v, double *s) {
  s[threadIdx.x] = v;
  __syncthreads();
  for (int o = kVB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  double r = s[0];
  __syncthreads();
  return r;
}
// The conjugate gradient runs on A0 = the Hessian with row and column gi
// replaced by the identity (symmetric positive definite for a connected
// diagram); with b[gi] = 0 its solution has x[gi] = 0, the gauge of
// include/MA/optimal_transport.hpp:82-86.  Scalars live on the device:
// scal = [rz (of the iteration's parity, 2), rr, ended, bb, done, iterations,
// breakdown].  No launch of more than one workgroup writes a flag that it
// returns on: its waves would read it before or after that write, and some of
// a workgroup would miss the others' barriers.  So k_cg_spmv returns on done
// and sets ended, k_cg_update returns on ended and sets done.
//
// An iteration is k_cg_spmv, k_cg_update and the preconditioner.  Below a few
// hundred thousand rows its time is the number of launches (about 5 us each),
// so the direction p = z + beta p is formed inside the product (p of a
// neighbour on the fly from z and the last p; two buffers of p take turns),
// and what the preconditioner needs at each r is written where r is.  With
// the cycle's own fusions an iteration on 150k rows went from 17 launches to
// 11 and from 89 to 73 us (10.1 k_cg_spmv, 5.1 k_cg_update, 58 the cycle).

// The head of the preconditioner at unknown i: y = omega r / D, and its
// share of r.y
template <class TY>
struct Head {
  const TY *dinv;
  TY *y;  // null: no head
  double omega;
  __device__ inline double operator()(int64_t i, double r) const {
    if (!y) return 0.0;
    const TY v = (TY)(omega * r * (double)dinv[i]);
    y[i] = v;
    return r * (double)v;
  }
};

// x = 0, r = b (r[gi] = 0), partial sums of r.r and (part_rz) of r.y; clears
// the scalars
template <class TY>
__global__ void __launch_bounds__(kCgThreads)
    k_cg_begin(int64_t n, const double *b, int32_t gi, double *x, double *r, Head<TY> head,
               double *part_rr, double *part_rz, double *scal) {
  __shared__ double s[2 * kCgThreads / 64];
  double c[2] = {0.0, 0.0};
  int64_t first, last;
  cg_rows(n, first, last);
  for (int64_t i = first + threadIdx.x; i < last; i += kCgThreads) {
    const double ri = (i == gi) ? 0.0 : b[i];
    x[i] = 0.0;
    r[i] = ri;
    c[0] += ri * ri;
    c[1] += head(i, ri);
  }
  cg_block_sums(c, s);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = c[0];
    if (part_rz) part_rz[blockIdx.x] = c[1];
    if (blockIdx.x == 0)
      for (int k = 0; k < 8; k++) scal[k] = 0.0;
  }
}
// bb = r.r; done when it is 0
__global__ void __launch_bounds__(kCgThreads) k_cg_scal_init(const double *part_rr, int np,
                                                             double *scal) {
  __shared__ double s[kCgThreads / 64];
  const double rr = cg_block_sum(threadIdx.x < np ? part_rr[threadIdx.x] : 0.0, s);
  if (threadIdx.x == 0) {
    scal[2] = rr;
    scal[4] = rr;
    if (rr == 0.0) scal[3] = scal[5] = 1.0;
  }
}
static_assert(kCgGrid <= kCgThreads, "one partial sum per thread");
// Start of iteration: nrz partial sums of r.z give beta, those of r.r the
// stopping test; then p = z + beta p_old, Ap = A0 p and partial sums of p.Ap.
// gz >= 0: the matrix holds the Hessian's own values and row gz is the gauge
// row, Ap[gz] = 0 (every vector of the iteration has a zero there, so column
// gz contributes nothing either); gz < 0: the values are already gauge-fixed.
__global__ void __launch_bounds__(kCgThreads)
    k_cg_spmv(int64_t n, int parity, const int32_t *__restrict__ ptr,
              const int32_t *__restrict__ col, const double *__restrict__ val,
              const double *__restrict__ z, const double *__restrict__ p_old,
              double *__restrict__ p, double *__restrict__ Ap, const double *part_rz, int nrz,
              const double *part_rr, double *part_pap, double *scal, double tol2, int32_t gz) {
  __shared__ double s[2 * kCgThreads / 64];
  const int t = (int)threadIdx.x, lane = t % kRowLanes;
  double v[2] = {t < nrz ? part_rz[t] : 0.0, t < gridDim.x ? part_rr[t] : 0.0};
  int64_t i, last;
  cg_rows(n, i, last);
  i += t / kRowLanes;
  RowHead<double> row;
  row.load(ptr, col, val, i, i < last, lane);
  if (scal[5] != 0.0) return;
  cg_block_sums(v, s);
  const double rz = v[0], rr = v[1], rz_old = scal[1 - parity];
  const bool end = scal[7] != 0.0 || (scal[6] != 0.0 && rr <= tol2 * scal[4]);
  if (blockIdx.x == 0 && t == 0) {
    scal[parity] = rz;
    scal[2] = rr;
    if (end) scal[3] = 1.0;
  }
  if (end) return;
  const double beta = (rz_old > 0.0) ? rz / rz_old : 0.0;
  // (the first iteration has no p_old: what the buffer holds is not read)
  auto at = [&](int64_t j) { return beta != 0.0 ? fma(beta, p_old[j], z[j]) : z[j]; };
  double acc = 0.0;
  // the kRowLanes lanes of a group share i, so they iterate together
  while (i < last) {
    const double a = row.dot(col, val, at);
    if (lane == 0) {
      const double pi = at(i), ai = i == gz ? 0.0 : a;
      p[i] = pi;
      Ap[i] = ai;
      acc += pi * ai;
    }
    i += kCgGroups;
    row.load(ptr, col, val, i, i < last, lane);
  }
  acc = cg_block_sum(acc, s);
  if (t == 0) part_pap[blockIdx.x] = acc;
}
// x += alpha p, r -= alpha Ap; the preconditioner's head; partial sums of r.r
// and (part_rz) of r.y
template <class TY>
__global__ void __launch_bounds__(kCgThreads)
    k_cg_update(int64_t n, int parity, const double *part_pap, double *scal, double *x, double *r,
                const double *p, const double *Ap, Head<TY> head, double *part_rr,
                double *part_rz) {
  __shared__ double s[2 * kCgThreads / 64];
  const double part = threadIdx.x < gridDim.x ? part_pap[threadIdx.x] : 0.0;
  if (scal[3] != 0.0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) scal[5] = 1.0;
    return;
  }
  const double pap = cg_block_sum(part, s);
  const double alpha = (pap > 0.0) ? scal[parity] / pap : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (pap > 0.0) {
      scal[6] += 1.0;
    } else {
      // p.Ap <= 0 (or NaN) with a nonzero residual: the matrix is not
      // positive definite on the search space.  The breakdown flag ends the
      // iteration at the next stopping test (alpha = 0 leaves x and r
      // unchanged in every block).
      scal[7] = 1.0;
    }
  }
  double c[2] = {0.0, 0.0};
  int64_t first, last;
  cg_rows(n, first, last);
  for (int64_t i = first + threadIdx.x; i < last; i += kCgThreads) {
    x[i] += alpha * p[i];
    const double ri = r[i] - alpha * Ap[i];
    r[i] = ri;
    c[0] += ri * ri;
    c[1] += head(i, ri);
  }
  cg_block_sums(c, s);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = c[0];
    if (part_rz) part_rz[blockIdx.x] = c[1];
  }
}
// The stopping test after the last iteration of a batch (k_cg_spmv of the
// next one would make the same).
__global__ void __launch_bounds__(kCgThreads)
    k_cg_end(const double *part_rr, int np, double *scal, double tol2) {
  __shared__ double s[kCgThreads / 64];
  if (scal[5] != 0.0) return;
  const double rr = cg_block_sum(threadIdx.x < np ? part_rr[threadIdx.x] : 0.0, s);
  if (threadIdx.x == 0) {
    scal[2] = rr;
    if (scal[7] != 0.0 || rr <= tol2 * scal[4]) scal[3] = scal[5] = 1.0;
  }
}
__global__ void k_set_zero_at(double *x, int32_t i) { x[i] = 0.0; }

// Reductions for the Newton driver: min m, ||m - nu||^2, max |m-nu|/nu, nu.w,
// sum(m - nu).  g = m - nu is written.
__global__ void __launch_bounds__(kVB) k_newton_stats(int64_t n, const double *m,
                                                      const double *nu, const double *w,
                                                      double *g, double *part) {
  __shared__ double s[kVB];
  double mn = HUGE_VAL, ss = 0.0, mr = 0.0, dot = 0.0, sg = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kVB + threadIdx.x; i < n; i += (int64_t)kVGrid * kVB) {
    const double gi = m[i] - nu[i];
    g[i] = gi;
    sg += gi;
    mn = fmin(mn, m[i]);
    ss += gi * gi;
    mr = fmax(mr, fabs(gi) / nu[i]);
    dot += nu[i] * w[i];
  }
  // min / max via the same shared buffer
  s[threadIdx.x] = mn;
  __syncthreads();
  for (int o = kVB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] = fmin(s[threadIdx.x], s[threadIdx.x + o]);
    __syncthreads();
  }
  mn = s[0];
  __syncthreads();
  s[threadIdx.x] = mr;
  __syncthreads();
  for (int o = kVB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] = fmax(s[threadIdx.x], s[threadIdx.x + o]);
    __syncthreads();
  }
  mr = s[0];
  __syncthreads();
  ss = block_sum(ss, s);
  dot = block_sum(dot, s);
  sg = block_sum(sg, s);
  if (threadIdx.x == 0) {
    part[5 * blockIdx.x + 0] = mn;
    part[5 * blockIdx.x + 1] = ss;
    part[5 * blockIdx.x + 2] = mr;
    part[5 * blockIdx.x + 3] = dot;
    part[5 * blockIdx.x + 4] = sg;
  }
}
// y = x + a d; *moved = 1 if any entry of y differs from x
__global__ void k_axpy_to(int64_t n, const double *x, double a, const double *d, double *y,
                          int32_t *moved) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) {
    const double v = x[i] + a * d[i];
    y[i] = v;
    if (v != x[i]) *moved = 1;
  }
}
// Two-word weights (hi, lo): (yh, yl) = (xh, xl) + a d.  The step joins the
// high word by TwoSum, the low word is added to the exact error and the pair
// is renormalised (|yl| <= ulp(yh) / 2); *moved = 1 if either word changes.
__global__ void k_axpy_dd(int64_t n, const double *xh, const double *xl, double a,
                          const double *d, double *yh, double *yl, int32_t *moved) {
#pragma clang fp contract(off)
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) {
    const double h = xh[i], t = a * d[i];
    const double s = h + t, bb = s - h;
    const double lo = ((h - (s - bb)) + (t - bb)) + xl[i];
    const double nh = s + lo, nl = lo - (nh - s);
    yh[i] = nh;
    yl[i] = nl;
    if (nh != h || nl != xl[i]) *moved = 1;
  }
}
// Renormalises caller-given two-word weights: (h, l) <- TwoSum(h, l).
__global__ void k_dd_norm(int64_t n, double *h, double *l) {
#pragma clang fp contract(off)
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) {
    const double a = h[i], b = l[i];
    const double s = a + b, bb = s - a;
    h[i] = s;
    l[i] = (a - (s - bb)) + (b - bb);
  }
}
__global__ void k_neg(int64_t n, double *x) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = -x[i];
}
__global__ void k_add_const(int64_t n, double *x, double c) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] += c;
}

// rows of ncol components from Morton to the caller's order
__global__ void k_columns(const double *src, const int32_t *perm, int64_t n, int ncol,
                          double *out) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < ncol * n) out[(int64_t)perm[t / ncol] * ncol + t % ncol] = src[t];
}

struct NewtonStats {
  double minm, l2, maxrel, nuw, sumg;
};

static hipError_t newton_stats(ma_engine *e, const double *m, const double *nu, const double *w,
                               double *g, NewtonStats &st) {
  SolverBuffers &S = e->sb;
  MA_HIP_RET(S.red.ensure(5 * kVGrid + 16));
  hipLaunchKernelGGL(k_newton_stats, dim3(kVGrid), dim3(kVB), 0, e->stream, e->n, m, nu, w, g,
                     S.red.p);
  std::vector<double> h(5 * kVGrid);
  MA_HIP_RET(read_back(e, {{h.data(), S.red.p, sizeof(double) * 5 * kVGrid}}));
  st.minm = HUGE_VAL;
  st.maxrel = 0.0;
  double ss = 0.0, dot = 0.0, sg = 0.0;
  for (int b = 0; b < kVGrid; b++) {
    st.minm = std::min(st.minm, h[5 * b]);
    ss += h[5 * b + 1];
    st.maxrel = std::max(st.maxrel, h[5 * b + 2]);
    dot += h[5 * b + 3];
    sg += h[5 * b + 4];
  }
  st.l2 = std::sqrt(ss);
  st.nuw = dot;
  st.sumg = sg;
  return hipSuccess;
}

// Representability floor of FP64 weights: the largest relative mass change
// one ulp of a weight can make, max_i max_{j != i} |H_ij| ulp(w_i) / nu_i
// (kVGrid partial maxima).  Below it no FP64 step can lower the error.
__global__ void __launch_bounds__(kVB) k_weight_floor(int64_t n, const int32_t *ptr,
                                                      const int32_t *col, const double *val,
                                                      const double *w, const double *nu,
                                                      double *part) {
  __shared__ double sm[kVB];
  double f = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kVB + threadIdx.x; i < n; i += (int64_t)kVGrid * kVB) {
    double m = 0.0;
    for (int32_t q = ptr[i]; q < ptr[i + 1]; q++)
      if (col[q] != i) m = fmax(m, fabs(val[q]));
    const double a = fabs(w[i]);
    f = fmax(f, m * (nextafter(a, HUGE_VAL) - a) / nu[i]);
  }
  sm[threadIdx.x] = f;
  __syncthreads();
  for (int o = kVB / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sm[threadIdx.x] = fmax(sm[threadIdx.x], sm[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

// The floor at weights w (Morton order) from the Hessian of the last evaluation.
static ma_status weight_floor(ma_engine *e, const double *w, const double *nu, double *floor) {
  SolverBuffers &S = e->sb;
  MA_HIP_TRY(S.red.ensure(5 * kVGrid + 16));
  hipLaunchKernelGGL(k_weight_floor, dim3(kVGrid), dim3(kVB), 0, e->stream, e->n,
                     e->eb.csr_ptr.p, e->eb.csr_col.p, e->eb.csr_val.p, w, nu, S.red.p);
  std::vector<double> h(kVGrid);
  MA_HIP_TRY(read_back(e, {{h.data(), S.red.p, sizeof(double) * kVGrid}}));
  *floor = *std::max_element(h.begin(), h.end());
  return MA_OK;
}

// Work vectors and scalars of one conjugate-gradient solve (n entries each,
// p twice; part_*: up to kCgGrid partial sums; scal: 8 scalars).
struct CgWork {
  double *r, *z, *p[2], *Ap, *part_rz, *part_rr, *part_pap, *scal;
};

// The iterations of the preconditioned conjugate gradient on M0 (see
// k_cg_spmv for gz), from x = 0, on the engine's stream.  head: what the
// preconditioner takes from the kernels that write r; precondition() launches
// the rest of z = P r and leaves nrz partial sums of r.z (0: the head is the
// whole preconditioner).  Iterations run in batches; the scalars stay on the
// device and the host checks the converged flag once per batch.  With
// use_graph the batches of a long solve are recorded once into a HIP graph
// (kernel nodes only) and replayed.  Returns MA_SINGULAR on a breakdown (p.Ap <= 0) and
// MA_LINEAR_FAIL when maxiter iterations end above rel_tol (the residual
// check of include/MA/optimal_transport.hpp:67-79); x, *iters and *rel_res
// are set in every case.
template <class TY, class Precond>
static ma_status cg_iterate(ma_engine *e, int64_t n, const int32_t *ptr, const int32_t *col,
                            const double *val, int32_t gz, const double *b, int32_t gi,
                            double *x, const CgWork &W, Head<TY> head, int nrz,
                            Precond precondition, double rel_tol, int maxiter, int batch,
                            bool use_graph, int64_t *iters, double *rel_res) {
  *iters = 0;
  *rel_res = 0.0;
  double *scal = W.scal;
  const int np = cg_grid(n);
  const dim3 grid(np), block(kCgThreads);
  double *head_rz = nrz ? nullptr : W.part_rz;  // r.y is r.z
  if (!nrz) nrz = np;
  hipLaunchKernelGGL(k_cg_begin<TY>, grid, block, 0, e->stream, n, b, gi, x, W.r, head, W.part_rr,
                     head_rz, scal);
  hipLaunchKernelGGL(k_cg_scal_init, dim3(1), block, 0, e->stream, W.part_rr, np, scal);
  MA_HIP_TRY(precondition());
  const double tol2 = rel_tol * rel_tol;
  double sc[8];
  MA_HIP_TRY(read_back(e, {{sc, scal, sizeof sc}}));
  if (sc[4] == 0.0) return MA_OK;
  // iterations it0 .. it0 + count - 1 (batch is even: the parity pattern repeats)
  auto launch = [&](int it0, int count) -> hipError_t {
    for (int q = 0; q < count; q++) {
      const int parity = (it0 + q) & 1;
      hipLaunchKernelGGL(k_cg_spmv, grid, block, 0, e->stream, n, parity, ptr, col, val, W.z,
                         W.p[1 - parity], W.p[parity], W.Ap, W.part_rz, nrz, W.part_rr,
                         W.part_pap, scal, tol2, gz);
      hipLaunchKernelGGL(k_cg_update<TY>, grid, block, 0, e->stream, n, parity, W.part_pap, scal,
                         x, W.r, W.p[parity], W.Ap, head, W.part_rr, head_rz);
      MA_HIP_RET(precondition());
    }
    hipLaunchKernelGGL(k_cg_end, dim3(1), block, 0, e->stream, W.part_rr, np, scal, tol2);
    return hipGetLastError();
  };
  // Recording and instantiating a graph costs as much as some 20 replays of it
  // (60-90 launches each) save: with the graph from the first batch a Newton
  // solve of N = 1000 took 17.6 ms against 16.8 ms without, from the 8th of 18
  // batches on 150k rows 11.1 against 11.0 ms.  Solves that have run longer
  // than that replay the rest.
  constexpr int kGraphFrom = 32;  // batches launched one by one before
  hipGraphExec_t exec = nullptr;
  int it = 0;
  hipError_t err = hipSuccess;
  while (it < maxiter) {
    const int count = std::min(batch, maxiter - it);
    if (use_graph && !exec && it >= kGraphFrom * batch && count == batch) {
      hipGraph_t graph = nullptr;
      MA_HIP_TRY(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
      const hipError_t le = launch(0, batch);
      const hipError_t ce = hipStreamEndCapture(e->stream, &graph);
      MA_HIP_TRY(le);
      MA_HIP_TRY(ce);
      const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      MA_HIP_TRY(ie);
    }
    if (exec && count == batch)
      err = hipGraphLaunch(exec, e->stream);
    else
      err = launch(it, count);
    if (err != hipSuccess) break;
    it += count;
    err = read_back(e, {{sc, scal, sizeof sc}});
    if (err != hipSuccess || sc[5] != 0.0) break;
  }
  if (exec) (void)hipGraphExecDestroy(exec);
  MA_HIP_TRY(err);
  hipLaunchKernelGGL(k_set_zero_at, dim3(1), dim3(1), 0, e->stream, x, gi);
  MA_HIP_TRY(hipGetLastError());
  *iters = (int64_t)sc[6];
  *rel_res = std::sqrt(sc[2] / sc[4]);
  if (sc[7] != 0.0) {
    e->err = "conjugate gradient breakdown (p.Ap <= 0): the gauge-fixed Hessian is not "
             "positive definite (disconnected cells?)";
    return MA_SINGULAR;
  }
  if (sc[5] == 0.0 || !(*rel_res <= rel_tol)) {
    char msg[160];
    snprintf(msg, sizeof msg,
             "linear solve stopped after %lld iterations at relative residual %.3g "
             "(tolerance %.3g)", (long long)*iters, *rel_res, rel_tol);
    e->err = msg;
    return MA_LINEAR_FAIL;
  }
  return MA_OK;
}

// Solve M0 d = b by the conjugate gradient, M0 = M with row and column gi
// replaced by the identity (the gauge), preconditioned by the aggregation
// multigrid cycle (precond 0) or by Jacobi (precond 1), with the engine's
// work buffers.  Returns MA_SINGULAR for a zero diagonal outside the gauge
// row, otherwise as cg_iterate.
// Tolerance at or above which the multigrid hierarchy is built in FP32.
constexpr double kAmgF32Tol = 1e-7;

static ma_status pcg(ma_engine *e, const CsrView &M, int32_t gi, const double *b, double *x,
                     double rel_tol, int maxiter, int precond, int64_t *iters,
                     double *rel_res) {
  *iters = 0;
  *rel_res = 0.0;
  SolverBuffers &S = e->sb;
  const int64_t n = M.n;
  MA_HIP_TRY(S.r.ensure((size_t)n));
  MA_HIP_TRY(S.z.ensure((size_t)n));
  MA_HIP_TRY(S.p.ensure((size_t)n));
  MA_HIP_TRY(S.q.ensure((size_t)n));
  MA_HIP_TRY(S.Ap.ensure((size_t)n));
  MA_HIP_TRY(S.red.ensure(5 * kVGrid + 16));
  static_assert(3 * kCgGrid <= 5 * kVGrid, "partial sums");
  CgWork W{S.r.p, S.z.p, {S.p.p, S.q.p}, S.Ap.p, S.red.p, S.red.p + kCgGrid,
           S.red.p + 2 * kCgGrid, S.red.p + 5 * kVGrid};
  if (!e->amg) e->amg = amg_create();
  {
    const int levels = precond == 0 ? 0 : 1;  // Jacobi needs level 0 only
    // a loose solve (every inexact-Newton step) takes the FP32 hierarchy:
    // its rounding (~1e-7) stays below what such a solve resolves
    const bool fp32 = rel_tol >= kAmgF32Tol;
    ma_status st = amg_setup(e, *e->amg, M, gi, levels, fp32);
    if (st != MA_OK) return st;
  }
  const double *val = amg_level0_values(*e->amg), *dinv = amg_level0_dinv(*e->amg);
  if (precond != 0)
    return cg_iterate(e, n, M.ptr, M.col, val, -1, b, gi, x, W, Head<double>{dinv, W.z, 1.0}, 0,
                      [] { return hipGetLastError(); }, rel_tol, maxiter, 32, e->use_graphs != 0,
                      iters, rel_res);
  auto cycle = [&]() { return amg_apply(e, *e->amg, W.r, W.z, W.part_rz, W.scal + 5); };
  const AmgHead h = amg_head(e, *e->amg);
  if (h.fp32)
    return cg_iterate(e, n, M.ptr, M.col, val, -1, b, gi, x, W,
                      Head<float>{(const float *)h.dinv, (float *)h.y, h.omega}, h.partials, cycle,
                      rel_tol, maxiter, 8, e->use_graphs != 0, iters, rel_res);
  return cg_iterate(e, n, M.ptr, M.col, val, -1, b, gi, x, W,
                    Head<double>{(const double *)h.dinv, (double *)h.y, h.omega}, h.partials,
                    cycle, rel_tol, maxiter, 8, e->use_graphs != 0, iters, rel_res);
}

// ---------------------------------------------------------------------------
// ma_solve_laplacian_csr_noalloc: the work memory of its conjugate gradient
// is this fixed device array (one copy per GPU, held until the process
// ends), carved into the Jacobi diagonal, five vectors of MA_NOALLOC_MAX_N
// entries, the partial sums, the scalars and two status flags.  Host code
// never passes `scratch` itself to a kernel (in host code the name is a
// stand-in, not a device address): ma_create looks up its address on each
// device once (scratch_ptr) and every launch uses that address.
// ---------------------------------------------------------------------------
constexpr int64_t kNaN = MA_NOALLOC_MAX_N;
constexpr size_t kNaVec = 6 * (size_t)kNaN;                 // dinv, r, z, p (2), Ap
constexpr size_t kNaDoubles = kNaVec + 3 * kCgGrid + 16 + 2;
static __device__ __align__(256) double scratch[kNaDoubles];

constexpr int kMaxDevices = 64;
static std::mutex scratch_mu;
static double *scratch_addr[kMaxDevices] = {};
static hipError_t scratch_status[kMaxDevices] = {};
static bool scratch_done[kMaxDevices] = {};

// Looks up this device's copy of `scratch` (the device must be current);
// once per device.
static void scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (scratch_done[device]) return;
  void *ptr = nullptr;
  scratch_status[device] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  scratch_addr[device] = scratch_status[device] == hipSuccess ? static_cast<double *>(ptr) : nullptr;
  scratch_done[device] = true;
}

// flags = 0 (the two status words at the end of the scratch array)
__global__ void k_na_clear(int32_t *flags) {
  if (threadIdx.x < 2) flags[threadIdx.x] = 0;
}
// Checks a caller CSR matrix (rowptr n + 1 entries from 0 to nnz, columns in
// [0, n)) without reading outside it, and forms the Jacobi inverse diagonal
// of the gauge-fixed matrix (row gi: 1).  flags[0]: bad structure;
// flags[1]: a non-positive diagonal outside row gi.
__global__ void k_na_check(int64_t n, int64_t nnz, const int32_t *ptr, const int32_t *col,
                           const double *val, int32_t gi, double *dinv, int32_t *flags) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t a = ptr[i], b = ptr[i + 1];
  if ((i == 0 && a != 0) || (i == n - 1 && b != nnz) || a < 0 || b < a || b > nnz) {
    atomicOr(&flags[0], 1);
    dinv[i] = 0.0;
    return;
  }
  double d = 0.0;
  for (int64_t q = a; q < b; q++) {
    const int32_t j = col[q];
    if (j < 0 || j >= n) {
      atomicOr(&flags[0], 1);
      continue;
    }
    if (j == i) d += val[q];
  }
  if (i == gi) d = 1.0;
  dinv[i] = d > 0.0 ? 1.0 / d : 0.0;
  if (!(d > 0.0)) atomicOr(&flags[1], 1);
}

// The Hessian of the last evaluation (Morton order) and its gauge slot: the
// caller's last Dirac, whose weight is never moved
// (include/MA/optimal_transport.hpp:82-86).
// Connected components of the graph of a symmetric CSR matrix (an edge per
// nonzero off-diagonal entry) by minimum-label propagation: labels start as
// the row index and take the smallest label of their row until nothing
// changes; every row then holds the smallest index of its component.
__global__ void k_cc_init(int64_t n, int32_t *label) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) label[i] = (int32_t)i;
}
__global__ void k_cc_step(int64_t n, const int32_t *ptr, const int32_t *col, const double *val,
                          int32_t *label, int32_t *changed) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int32_t m = label[i];
  for (int32_t q = ptr[i]; q < ptr[i + 1]; q++)
    if (val[q] != 0.0) m = min(m, label[col[q]]);
  if (m < label[i]) {
    label[i] = m;
    *changed = 1;
  }
}
__global__ void k_cc_any_nonzero(int64_t n, const int32_t *label, int32_t *flag) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n && label[i] != 0) *flag = 1;
}

// Whether the diagram of the last evaluation is connected (its Hessian's
// graph has one component).  Used only after a solve has failed, to tell a
// disconnected diagram (a singular Newton system) from other failures.
static ma_status diagram_connected(ma_engine *e, bool *connected) {
  const int64_t n = e->n;
  SolverBuffers &S = e->sb;
  MA_HIP_TRY(S.cc.ensure((size_t)n));
  MA_HIP_TRY(S.moved.ensure(1));
  const unsigned nb = (unsigned)((n + 255) / 256);
  const int32_t *ptr = e->eb.csr_ptr.p, *col = e->eb.csr_col.p;
  const double *val = e->eb.csr_val.p;
  hipLaunchKernelGGL(k_cc_init, dim3(nb), dim3(256), 0, e->stream, n, S.cc.p);
  int32_t changed = 1;
  // in-place updates carry a label along many rows per sweep; the number
  // of sweeps is bounded by the graph's diameter
  for (int64_t sweep = 0; changed && sweep < n; sweep += 32) {
    MA_HIP_TRY(hipMemsetAsync(S.moved.p, 0, sizeof(int32_t), e->stream));
    for (int k = 0; k < 32; k++)
      hipLaunchKernelGGL(k_cc_step, dim3(nb), dim3(256), 0, e->stream, n, ptr, col, val, S.cc.p,
                         S.moved.p);
    MA_HIP_TRY(read_back(e, {{&changed, S.moved.p, sizeof(int32_t)}}));
  }
  int32_t other = 0;
  MA_HIP_TRY(hipMemsetAsync(S.moved.p, 0, sizeof(int32_t), e->stream));
  hipLaunchKernelGGL(k_cc_any_nonzero, dim3(nb), dim3(256), 0, e->stream, n, S.cc.p, S.moved.p);
  MA_HIP_TRY(read_back(e, {{&other, S.moved.p, sizeof(int32_t)}}));
  *connected = other == 0;
  return MA_OK;
}

static hipError_t eval_csr(ma_engine *e, CsrView &M, int32_t &gi) {
  M.n = e->n;
  M.nnz = e->nnz;
  M.ptr = e->eb.csr_ptr.p;
  M.col = e->eb.csr_col.p;
  M.val = e->eb.csr_val.p;
  return read_back(e, {{&gi, e->iperm.p + (e->n - 1), sizeof(int32_t)}});
}

}  // namespace ma

using namespace ma;

ma_status ma::need(ma_engine *e) {
  if (!e) return MA_BAD_INPUT;
  if (!e->have_mesh || !e->have_diracs) {
    e->err = "mesh and Diracs must be set first";
    return MA_NO_DATA;
  }
  if (!e->grid_valid) {
    hipError_t r = build_triangle_bins(e);
    if (r != hipSuccess) {
      e->err = std::string("triangle binning: ") + hipGetErrorString(r);
      return MA_HIP_ERROR;
    }
    e->grid_valid = true;
  }
  return MA_OK;
}

static void choose_grid(ma_engine *e, const double *X, int64_t n, int layout) {
  double x0 = e->dom[0], y0 = e->dom[1], x1 = e->dom[2], y1 = e->dom[3];
  if (!e->have_mesh) {
    x0 = y0 = HUGE_VAL;
    x1 = y1 = -HUGE_VAL;
  }
  for (int64_t i = 0; i < n; i++) {
    double x = layout == MA_XY_COLMAJOR ? X[i] : X[2 * i];
    double y = layout == MA_XY_COLMAJOR ? X[n + i] : X[2 * i + 1];
    x0 = std::min(x0, x);
    x1 = std::max(x1, x);
    y0 = std::min(y0, y);
    y1 = std::max(y1, y);
  }
  double side = std::max(x1 - x0, y1 - y0);
  if (!(side > 0)) side = 1.0;
  side *= 1.0 + 1e-6;
  const double cx = 0.5 * (x0 + x1), cy = 0.5 * (y0 + y1);
  // about 1.5 Diracs per bin; and, with a mesh already set, at most ~16
  // triangles per bin (the triangles share the grid: with few Diracs on a
  // fine mesh, bins of thousands of triangles made every scan of a cell's
  // triangles, and their sort at set-up, long serial loops)
  const double per4 = std::log(4.0);
  int L = (int)std::lround(std::log(std::max(1.0, (double)n / 1.5)) / per4);
  if (e->have_mesh)
    L = std::max(L, (int)std::lround(std::log(std::max(1.0, (double)e->nt / 16.0)) / per4));
  L = std::max(0, std::min(L, kMaxLevels));
  Grid g;
  g.L = L;
  g.G = 1 << L;
  g.nbins = (int64_t)g.G * g.G;
  g.h = side / g.G;
  g.x0 = cx - 0.5 * side;
  g.y0 = cy - 0.5 * side;
  e->grid = g;
}

extern "C" {

void ma_default_solve_opts(ma_solve_opts *o) {
  if (!o) return;
  o->precision = MA_FP64;
  o->stop_rule = MA_STOP_L2;
  o->eps_g = 1e-7;
  o->tol = 1e-8;
  o->maxiter = 100;
  o->alpha_min = std::ldexp(1.0, -30);
  o->cg_tol = 0.0;
  o->cg_maxiter = 20000;
  o->verbose = 0;
  o->preconditioner = 0;
}

ma_status ma_create(int device, ma_engine **out) {
  if (!out) return MA_BAD_INPUT;
  *out = nullptr;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= device || device < 0)
    return MA_HIP_ERROR;
  if (hipSetDevice(device) != hipSuccess) return MA_HIP_ERROR;
  scratch_init(device);  // address of this device's no-allocation work memory
  ma_engine *e = new ma_engine();
  e->device = device;
  if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess) {
    delete e;
    return MA_HIP_ERROR;
  }
  if (hipHostMalloc(reinterpret_cast<void **>(&e->pinned), kReadBytes, hipHostMallocDefault) !=
      hipSuccess) {
    hipStreamDestroy(e->stream);
    delete e;
    return MA_HIP_ERROR;
  }
  for (auto &ev : e->ev) hipEventCreate(&ev);
  *out = e;
  return MA_OK;
}

void ma_destroy(ma_engine *e) {
  if (!e) return;
  hipSetDevice(e->device);
  hipStreamSynchronize(e->stream);
  for (auto &ev : e->ev) hipEventDestroy(ev);
  hipStreamDestroy(e->stream);
  (void)hipHostFree(e->pinned);
  if (e->amg) amg_destroy(e->amg);
  // every device buffer is released by its owner's destructor
  delete e;
}

const char *ma_last_error(const ma_engine *e) { return e ? e->err.c_str() : "null engine"; }

ma_status ma_set_mesh(ma_engine *e, int64_t nv, const double *vxy, const double *vval,
                      int64_t nt, const int32_t *tri) {
  if (!e || nv < 3 || nt < 1 || !vxy || !vval || !tri) return MA_BAD_INPUT;
  if (nt > (int64_t)INT32_MAX / 4 || nv > (int64_t)INT32_MAX) return MA_BAD_INPUT;
  hipSetDevice(e->device);
  for (int64_t f = 0; f < 3 * nt; f++)
    if (tri[f] < 0 || tri[f] >= nv) {
      e->err = "triangle vertex index out of range";
      return MA_BAD_INPUT;
    }
  double x0 = HUGE_VAL, y0 = HUGE_VAL, x1 = -HUGE_VAL, y1 = -HUGE_VAL;
  for (int64_t i = 0; i < nv; i++) {
    if (!std::isfinite(vxy[2 * i]) || !std::isfinite(vxy[2 * i + 1]) || !std::isfinite(vval[i])) {
      e->err = "non-finite mesh data";
      return MA_BAD_INPUT;
    }
    x0 = std::min(x0, vxy[2 * i]);
    x1 = std::max(x1, vxy[2 * i]);
    y0 = std::min(y0, vxy[2 * i + 1]);
    y1 = std::max(y1, vxy[2 * i + 1]);
  }
  invalidate_mesh(e);
  MA_HIP_TRY(e->vxy.ensure((size_t)(2 * nv)));
  MA_HIP_TRY(e->vval.ensure((size_t)nv));
  DBuf<int32_t> dtri;
  MA_HIP_TRY(dtri.ensure((size_t)(3 * nt)));
  MA_HIP_TRY(hipMemcpyAsync(e->vxy.p, vxy, sizeof(double) * 2 * nv, hipMemcpyHostToDevice, e->stream));
  MA_HIP_TRY(hipMemcpyAsync(e->vval.p, vval, sizeof(double) * nv, hipMemcpyHostToDevice, e->stream));
  MA_HIP_TRY(hipMemcpyAsync(dtri.p, tri, sizeof(int32_t) * 3 * nt, hipMemcpyHostToDevice, e->stream));
  const double box[4] = {x0, y0, x1, y1};
  return finish_mesh(e, nv, nt, dtri.p, box);
}

}  // extern "C"

void ma::invalidate_mesh(ma_engine *e) {
  e->have_mesh = false;
  e->grid_valid = false;
  e->have_eval = false;
  e->have_hessian = false;
}

ma_status ma::finish_mesh(ma_engine *e, int64_t nv, int64_t nt, const int32_t *d_tri,
                          const double box[4]) {
  // every mesh buffer may be overwritten below: nothing may use the old mesh
  // if this fails half way
  invalidate_mesh(e);
  // a mesh vertex outside the current grid invalidates the Dirac binning
  if (e->have_diracs && (box[0] < e->grid.x0 || box[1] < e->grid.y0 ||
                         box[2] > e->grid.x0 + e->grid.G * e->grid.h ||
                         box[3] > e->grid.y0 + e->grid.G * e->grid.h)) {
    e->have_diracs = false;
  }
  for (int i = 0; i < 4; i++) e->dom[i] = box[i];
  MA_HIP_TRY(e->tri.ensure((size_t)nt));
  MA_HIP_TRY(e->triv.ensure((size_t)(3 * nt)));
  MA_HIP_TRY(e->tbox.ensure((size_t)nt));
  DBuf<int32_t> bad;
  MA_HIP_TRY(bad.ensure(1));
  MA_HIP_TRY(hipMemsetAsync(bad.p, 0, sizeof(int32_t), e->stream));
  hipLaunchKernelGGL(k_tri_prep, dim3((unsigned)((nt + 127) / 128)), dim3(128), 0, e->stream,
                     e->vxy.p, e->vval.p, d_tri, nt, e->tri.p, e->triv.p, e->tbox.p, bad.p);
  int32_t hb = 0;
  MA_HIP_TRY(hipMemcpyAsync(&hb, bad.p, sizeof(int32_t), hipMemcpyDeviceToHost, e->stream));
  MA_HIP_TRY(hipStreamSynchronize(e->stream));
  bad.release();
  if (hb) {
    e->err = "degenerate (zero-area) triangle";
    return MA_BAD_INPUT;
  }
  ma_status st = sort_triangles(e, nt);
  if (st != MA_OK) return st;
  e->nv = nv;
  e->nt = nt;
  e->have_mesh = true;
  return MA_OK;
}

extern "C" {

ma_status ma_set_diracs(ma_engine *e, int64_t n, const double *X, int layout) {
  if (!e || n < 1 || !X || (layout != MA_XY_INTERLEAVED && layout != MA_XY_COLMAJOR))
    return MA_BAD_INPUT;
  if (n > (int64_t)INT32_MAX / 8) return MA_BAD_INPUT;
  hipSetDevice(e->device);
  for (int64_t i = 0; i < 2 * n; i++)
    if (!std::isfinite(X[i])) {
      e->err = "non-finite Dirac position";
      return MA_BAD_INPUT;
    }
  // the Dirac buffers are overwritten below: nothing may use the old Diracs
  // if this fails half way
  e->have_diracs = false;
  e->grid_valid = false;
  e->have_eval = false;
  e->have_hessian = false;
  e->owner_init = false;
  e->far_valid = false;
  e->mask_ok = true;
  e->many_far = false;
  e->n = n;
  choose_grid(e, X, n, layout);
  DBuf<double> &dX = e->cb.xy;
  MA_HIP_TRY(dX.ensure((size_t)(2 * n)));
  MA_HIP_TRY(hipMemcpyAsync(dX.p, X, sizeof(double) * 2 * n, hipMemcpyHostToDevice, e->stream));
  MA_HIP_TRY(build_dirac_grid(e, dX.p, layout));
  e->have_diracs = true;
  return MA_OK;
}

static ma_status eval_morton(ma_engine *e, int precision, double *fval) {
  if (precision != MA_FP64 && precision != MA_MIXED) {
    e->err = "unknown precision";
    return MA_BAD_INPUT;
  }
  return evaluate(e, 0, fval, precision == MA_MIXED);
}

ma_status ma_kantorovich(ma_engine *e, const double *w, int precision, double *fval, double *g,
                         int64_t *nnz) {
  return ma_kantorovich_x(e, w, nullptr, precision, fval, g, nnz);
}

ma_status ma_kantorovich_x(ma_engine *e, const double *w, const double *w_lo, int precision,
                           double *fval, double *g, int64_t *nnz) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!w) return MA_BAD_INPUT;
  if (precision != MA_FP64 && precision != MA_MIXED) {
    e->err = "unknown precision";
    return MA_BAD_INPUT;  // rejected before anything is overwritten
  }
  EvalBuffers &B = e->eb;
  MA_HIP_TRY(B.w_s.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, w, B.w_s.p, false));
  if (w_lo) {
    MA_HIP_TRY(B.wlo_s.ensure((size_t)e->n));
    MA_HIP_TRY(to_morton(e, w_lo, B.wlo_s.p, false));
    hipLaunchKernelGGL(k_dd_norm, dim3((unsigned)((e->n + 255) / 256)), dim3(256), 0, e->stream,
                       e->n, B.w_s.p, B.wlo_s.p);
  }
  WloScope scope(B, w_lo != nullptr);
  double fv = 0.0;
  s = eval_morton(e, precision, &fv);
  if (s != MA_OK) return s;
  if (fval) *fval = fv;
  if (g) MA_HIP_TRY(from_morton(e, e->eb.mass_s.p, g, false));
  if (nnz) *nnz = e->nnz;
  return MA_OK;
}

ma_status ma_kantorovich_device(ma_engine *e, const double *d_w, int precision, double *fval,
                                double *d_g, int64_t *nnz) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!d_w) return MA_BAD_INPUT;
  if (precision != MA_FP64 && precision != MA_MIXED) {
    e->err = "unknown precision";
    return MA_BAD_INPUT;  // rejected before anything is overwritten
  }
  MA_HIP_TRY(e->eb.w_s.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, d_w, e->eb.w_s.p, true));
  double fv = 0.0;
  s = eval_morton(e, precision, &fv);
  if (s != MA_OK) return s;
  if (fval) *fval = fv;
  if (d_g) {
    MA_HIP_TRY(from_morton(e, e->eb.mass_s.p, d_g, true));
    MA_HIP_TRY(hipStreamSynchronize(e->stream));
  }
  if (nnz) *nnz = e->nnz;
  return MA_OK;
}

ma_status ma_hessian_copy(ma_engine *e, int32_t *rowptr, int32_t *col, double *val) {
  if (!e || !rowptr || !col || !val) return MA_BAD_INPUT;
  if (!e->have_hessian) {
    e->err = "no successful Kantorovich evaluation since the last change of inputs";
    return MA_NO_DATA;
  }
  MA_HIP_TRY(csr_to_caller(e, rowptr, col, val));
  return MA_OK;
}

ma_status ma_cell_costs(ma_engine *e, double *cost) {
  if (!e || !cost) return MA_BAD_INPUT;
  if (!e->have_hessian) {
    e->err = "no successful Kantorovich evaluation since the last change of inputs";
    return MA_NO_DATA;
  }
  MA_HIP_TRY(from_morton(e, e->eb.intg_s.p, cost, false));
  return MA_OK;
}

// Copies an interleaved per-Dirac array of `ncol` components from Morton
// order on the device to the caller's order on the host.
static hipError_t columns_to_host(ma_engine *e, const double *src, int ncol, double *dst) {
  DBuf<double> &out = e->cb.xy;
  MA_HIP_RET(out.ensure((size_t)(ncol * e->n)));
  hipLaunchKernelGGL(k_columns, dim3((unsigned)((ncol * e->n + 127) / 128)), dim3(128), 0,
                     e->stream, src, e->perm.p, e->n, ncol, out.p);
  MA_HIP_RET(hipGetLastError());
  MA_HIP_RET(hipMemcpyAsync(dst, out.p, sizeof(double) * ncol * e->n, hipMemcpyDeviceToHost,
                            e->stream));
  return hipStreamSynchronize(e->stream);
}

ma_status ma_first_moment(ma_engine *e, const double *w, double *mass, double *mom) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!w) return MA_BAD_INPUT;
  MA_HIP_TRY(e->eb.w_s.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, w, e->eb.w_s.p, false));
  s = evaluate(e, 1, nullptr);
  if (s != MA_OK) return s;
  if (mass) MA_HIP_TRY(from_morton(e, e->eb.mass_s.p, mass, false));
  if (mom) MA_HIP_TRY(columns_to_host(e, e->eb.mom_s.p, 2, mom));
  return MA_OK;
}

ma_status ma_second_moment(ma_engine *e, const double *w, double *mass, double *mom,
                           double *inertia) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!w) return MA_BAD_INPUT;
  MA_HIP_TRY(e->eb.w_s.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, w, e->eb.w_s.p, false));
  s = evaluate(e, 3, nullptr);
  if (s != MA_OK) return s;
  if (mass) MA_HIP_TRY(from_morton(e, e->eb.mass_s.p, mass, false));
  if (mom) MA_HIP_TRY(columns_to_host(e, e->eb.mom_s.p, 2, mom));
  if (inertia) MA_HIP_TRY(columns_to_host(e, e->eb.mom2_s.p, 3, inertia));
  return MA_OK;
}

ma_status ma_solve_laplacian(ma_engine *e, const double *g, double *d, double rel_tol,
                             int maxiter, double *res, int64_t *iters) {
  if (!e || !g || !d) return MA_BAD_INPUT;
  if (!e->have_hessian) {
    e->err = "no successful Kantorovich evaluation since the last change of inputs";
    return MA_NO_DATA;
  }
  SolverBuffers &S = e->sb;
  MA_HIP_TRY(S.g.ensure((size_t)e->n));
  MA_HIP_TRY(S.d.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, g, S.g.p, false));
  int64_t it = 0;
  double rr = 0.0;
  CsrView M;
  int32_t gi = 0;
  MA_HIP_TRY(eval_csr(e, M, gi));
  const ma_status ps = pcg(e, M, gi, S.g.p, S.d.p, rel_tol > 0 ? rel_tol : 1e-12,
                           maxiter > 0 ? maxiter : 100000, 0, &it, &rr);
  if (ps != MA_OK && ps != MA_LINEAR_FAIL) return ps;
  MA_HIP_TRY(from_morton(e, S.d.p, d, false));
  if (res) *res = rr;
  if (iters) *iters = it;
  return ps;
}

ma_status ma_solve_laplacian_csr(ma_engine *e, int64_t n, const int32_t *rowptr,
                                 const int32_t *col, const double *val, const double *g,
                                 double *d, double rel_tol, int maxiter, double *res,
                                 int64_t *iters) {
  if (!e || n < 1 || !rowptr || !col || !val || !g || !d) return MA_BAD_INPUT;
  if (n > INT32_MAX) return MA_BAD_INPUT;
  std::vector<int32_t> hp(rowptr, rowptr + n + 1);
  const int64_t nnz = hp[n];
  if (hp[0] != 0 || nnz < 0) {
    e->err = "row pointer must start at 0";
    return MA_BAD_INPUT;
  }
  for (int64_t i = 0; i < n; i++)
    if (hp[i + 1] < hp[i]) {
      e->err = "row pointer must be non-decreasing";
      return MA_BAD_INPUT;
    }
  for (int64_t q = 0; q < nnz; q++)
    if (col[q] < 0 || col[q] >= n) {
      e->err = "column index out of range";
      return MA_BAD_INPUT;
    }
  SolverBuffers &S = e->sb;
  MA_HIP_TRY(S.hptr.ensure((size_t)n + 1));
  MA_HIP_TRY(S.hcol.ensure((size_t)nnz + 1));
  MA_HIP_TRY(S.hval.ensure((size_t)nnz + 1));
  MA_HIP_TRY(S.hg.ensure((size_t)n));
  MA_HIP_TRY(S.hd.ensure((size_t)n));
  MA_HIP_TRY(hipMemcpyAsync(S.hptr.p, rowptr, sizeof(int32_t) * (n + 1), hipMemcpyHostToDevice,
                            e->stream));
  MA_HIP_TRY(hipMemcpyAsync(S.hcol.p, col, sizeof(int32_t) * nnz, hipMemcpyHostToDevice,
                            e->stream));
  MA_HIP_TRY(hipMemcpyAsync(S.hval.p, val, sizeof(double) * nnz, hipMemcpyHostToDevice,
                            e->stream));
  MA_HIP_TRY(hipMemcpyAsync(S.hg.p, g, sizeof(double) * n, hipMemcpyHostToDevice, e->stream));
  CsrView M;
  M.n = n;
  M.nnz = nnz;
  M.ptr = S.hptr.p;
  M.col = S.hcol.p;
  M.val = S.hval.p;
  M.own_col = S.hcol.p;
  M.own_val = S.hval.p;
  int64_t it = 0;
  double rr = 0.0;
  const ma_status ps = pcg(e, M, (int32_t)(n - 1), S.hg.p, S.hd.p,
                           rel_tol > 0 ? rel_tol : 1e-12, maxiter > 0 ? maxiter : 100000, 0,
                           &it, &rr);
  if (ps != MA_OK && ps != MA_LINEAR_FAIL) return ps;
  MA_HIP_TRY(hipMemcpyAsync(d, S.hd.p, sizeof(double) * n, hipMemcpyDeviceToHost, e->stream));
  MA_HIP_TRY(hipStreamSynchronize(e->stream));
  if (res) *res = rr;
  if (iters) *iters = it;
  return ps;
}

ma_status ma_solve_laplacian_csr_noalloc(ma_engine *e, int64_t n, int64_t nnz,
                                         const int32_t *d_rowptr, const int32_t *d_col,
                                         const double *d_val, const double *d_g, double *d_d,
                                         double rel_tol, int maxiter, double *res,
                                         int64_t *iters) {
  if (!e || !d_rowptr || !d_col || !d_val || !d_g || !d_d) return MA_BAD_INPUT;
  if (n < 1 || n > kNaN || nnz < 0 || nnz > INT32_MAX) {
    e->err = "ma_solve_laplacian_csr_noalloc: n must be in [1, MA_NOALLOC_MAX_N] and nnz in "
             "[0, 2^31)";
    return MA_BAD_INPUT;
  }
  if (hipSetDevice(e->device) != hipSuccess) return MA_HIP_ERROR;
  double *base = (e->device >= 0 && e->device < kMaxDevices) ? scratch_addr[e->device] : nullptr;
  if (!base) {
    e->err = std::string("no-allocation work memory unavailable on this device: ") +
             hipGetErrorString(e->device >= 0 && e->device < kMaxDevices
                                   ? scratch_status[e->device] : hipErrorInvalidDevice);
    return MA_HIP_ERROR;
  }
  double *dinv = base;
  double *sums = base + kNaVec;
  CgWork W{base + kNaN, base + 2 * kNaN, {base + 3 * kNaN, base + 4 * kNaN}, base + 5 * kNaN, sums,
           sums + kCgGrid, sums + 2 * kCgGrid, sums + 3 * kCgGrid};
  int32_t *flags = reinterpret_cast<int32_t *>(sums + 3 * kCgGrid + 16);
  const int32_t gi = (int32_t)(n - 1);  // gauge: the last unknown, as ma_solve_laplacian_csr
  hipLaunchKernelGGL(k_na_clear, dim3(1), dim3(64), 0, e->stream, flags);
  hipLaunchKernelGGL(k_na_check, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream, n,
                     nnz, d_rowptr, d_col, d_val, gi, dinv, flags);
  int32_t hf[2] = {0, 0};
  MA_HIP_TRY(read_back(e, {{hf, flags, sizeof hf}}));
  if (hf[0]) {
    e->err = "CSR matrix: row pointers must run from 0 to nnz without decreasing and columns "
             "must lie in [0, n)";
    return MA_BAD_INPUT;
  }
  if (hf[1]) {
    e->err = "singular matrix: a row other than the gauge row has no positive diagonal entry";
    return MA_SINGULAR;
  }
  int64_t it = 0;
  double rr = 0.0;
  const ma_status st = cg_iterate(e, n, d_rowptr, d_col, d_val, gi, d_g, gi, d_d, W,
                                  Head<double>{dinv, W.z, 1.0}, 0,
                                  [] { return hipGetLastError(); }, rel_tol > 0 ? rel_tol : 1e-12,
                                  maxiter > 0 ? maxiter : 100000, 32, false, &it, &rr);
  if (res) *res = rr;
  if (iters) *iters = it;
  if (st == MA_OK || st == MA_LINEAR_FAIL || st == MA_SINGULAR) {
    MA_HIP_TRY(hipStreamSynchronize(e->stream));  // d_d is complete on return
  }
  return st;
}

ma_status ma_ot_solve(ma_engine *e, const double *nu, double *w, int init_w,
                      const ma_solve_opts *opts, ma_stats *stats) {
  return ma_ot_solve_x(e, nu, w, nullptr, init_w, opts, stats);
}

// w_lo == nullptr: FP64 weights (ma_ot_solve); otherwise the iterate is
// carried in two words (S.w + S.wl) and every evaluation forms the bisector
// offsets from both.
ma_status ma_ot_solve_x(ma_engine *e, const double *nu, double *w, double *w_lo, int init_w,
                        const ma_solve_opts *opts, ma_stats *stats) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!nu || !w) return MA_BAD_INPUT;
  const bool dd = w_lo != nullptr;
  ma_solve_opts o;
  ma_default_solve_opts(&o);
  if (opts) o = *opts;
  const auto t_start = std::chrono::steady_clock::now();
  const int64_t n = e->n;
  SolverBuffers &S = e->sb;
  EvalBuffers &B = e->eb;
  for (DBuf<double> *b : {&S.w, &S.nu, &S.g, &S.d, &S.wtrial}) MA_HIP_TRY(b->ensure((size_t)n));
  MA_HIP_TRY(S.moved.ensure(1));
  MA_HIP_TRY(B.w_s.ensure((size_t)n));
  MA_HIP_TRY(to_morton(e, nu, S.nu.p, false));
  if (init_w) {
    MA_HIP_TRY(to_morton(e, w, S.w.p, false));
  } else {
    MA_HIP_TRY(hipMemsetAsync(S.w.p, 0, sizeof(double) * n, e->stream));
  }
  if (dd) {
    for (DBuf<double> *b : {&S.wl, &S.wtl, &B.wlo_s}) MA_HIP_TRY(b->ensure((size_t)n));
    if (init_w) {
      MA_HIP_TRY(to_morton(e, w_lo, S.wl.p, false));
      hipLaunchKernelGGL(k_dd_norm, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream,
                         n, S.w.p, S.wl.p);
    } else {
      MA_HIP_TRY(hipMemsetAsync(S.wl.p, 0, sizeof(double) * n, e->stream));
    }
  }
  WloScope scope(B, dd);
  ma_stats st{};
  double ms_eval = 0.0, ms_lin = 0.0;
  // Mixed precision: evaluations run with FP32 geometry while the max
  // relative mass error is above kSwitch (FP32 masses are good to about
  // 1e-6 relative), then in FP64.  The damping test, the CG scalars and the
  // stopping test are FP64 throughout, and the solve never stops on an FP32
  // evaluation: the final check is always an FP64 evaluation.
  constexpr double kSwitch = 1e-4, kStall = 0.05;
  // FP32 masses scatter by ~1e-6 of ||nu||_2 (l2 over the cells); a gradient
  // within kNoiseRatio of that scatter is reduced no further by an FP32 step
  constexpr double kF32Noise = 1e-6, kNoiseRatio = 100.0;
  // a failed full step is checked against the weights' representability
  // floor once the max relative error is below kFloorCheck
  constexpr double kFloorCheck = 1e-6, kFloorMargin = 4.0;
  double noise_l2 = 0.0;
  {
    long double q = 0.0L;
    for (int64_t i = 0; i < n; i++) q += (long double)nu[i] * nu[i];
    noise_l2 = kF32Noise * std::sqrt((double)q);
  }
  bool fp32_phase = o.precision == MA_MIXED;
  // the first FP64 direction after FP32 steps starts from their scatter,
  // spread over every cell (an FP64 iterate's error sits in a few): it is
  // solved ten times tighter so that one step clears the stopping test
  bool after_fp32 = false;
  bool last_fp64 = false;
  auto eval_at = [&](const double *wm, const double *wml, double &fval,
                     NewtonStats &ns) -> ma_status {
    auto t0 = std::chrono::steady_clock::now();
    hipMemcpyAsync(B.w_s.p, wm, sizeof(double) * n, hipMemcpyDeviceToDevice, e->stream);
    if (dd)
      hipMemcpyAsync(B.wlo_s.p, wml, sizeof(double) * n, hipMemcpyDeviceToDevice, e->stream);
    ma_status r = eval_morton(e, fp32_phase ? MA_MIXED : MA_FP64, &fval);
    last_fp64 = !fp32_phase;
    st.neval++;
    if (fp32_phase) st.neval_fp32++;
    if (r != MA_OK) return r;
    hipError_t he = newton_stats(e, B.mass_s.p, S.nu.p, wm, S.g.p, ns);
    if (he != hipSuccess) {
      e->err = hipGetErrorString(he);
      return MA_HIP_ERROR;
    }
    ms_eval += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return MA_OK;
  };
  double fval = 0.0;
  NewtonStats ns{};
  s = eval_at(S.w.p, S.wl.p, fval, ns);
  if (s != MA_OK) return s;
  double numin = 0.0;
  {
    std::vector<double> hnu(nu, nu + n);
    numin = *std::min_element(hnu.begin(), hnu.end());
  }
  const double eps0 = std::min(ns.minm, numin) / 2.0;
  ma_status result = MA_OK;
  if (eps0 <= 0) {
    // include/MA/optimal_transport.hpp:137-148 (empty initial cell)
    std::vector<double> m(n);
    from_morton(e, B.mass_s.p, m.data(), false);
    st.bad_index = std::min_element(m.begin(), m.end()) - m.begin();
    e->err = "Laguerre cell of Dirac " + std::to_string(st.bad_index) + " is empty";
    result = MA_EMPTY_CELL;
  }
  auto keep_going = [&](const NewtonStats &q) {
    return o.stop_rule == MA_STOP_L2 ? (q.l2 >= o.eps_g) : (q.maxrel > o.tol);
  };
  int64_t niter = 0;
  const double l2_0 = ns.l2;
  while (result == MA_OK) {
    if (!keep_going(ns)) {
      if (last_fp64) break;
      // converged on an FP32 evaluation: confirm (or continue) in FP64
      fp32_phase = false;
      after_fp32 = true;
      s = eval_at(S.w.p, S.wl.p, fval, ns);
      if (s != MA_OK) return s;
      continue;
    }
    if (niter++ > o.maxiter) {  // `niter++ <= maxiter` (optimal_transport.hpp:151)
      result = MA_NOT_CONVERGED;
      break;
    }
    // Newton direction d = -H^-1 g (gauge fixed)
    auto t0 = std::chrono::steady_clock::now();
    double rel = o.cg_tol;
    if (rel <= 0) {
      // inexact Newton forcing term: tightened as the residual shrinks, but
      // no tighter than the stopping test needs (a tenth of the remaining
      // reduction; the quadratic term takes care of the rest)
      const double need = o.stop_rule == MA_STOP_L2 ? o.eps_g / std::max(ns.l2, 1e-300)
                                                    : o.tol / std::max(ns.maxrel, 1e-300);
      rel = std::min(1e-2 * ns.l2 / std::max(l2_0, 1e-300), 1e-3);
      const bool first64 = after_fp32 && !fp32_phase;
      rel = std::max(rel, std::min((first64 ? 0.01 : 0.1) * need, 1e-3));
      if (first64) after_fp32 = false;
      rel = std::max(rel, 1e-12);
      // an FP32 gradient is known to its scatter only: solving much further
      // than that buys nothing (a tenth of it, so that the last FP32 step
      // still lands near the scatter in the max-relative norm too)
      if (fp32_phase) rel = std::max(rel, std::min(0.5, 0.1 * noise_l2 / std::max(ns.l2, 1e-300)));
    }
    int64_t it = 0;
    double rr = 0.0;
    CsrView M;
    int32_t gi = 0;
    MA_HIP_TRY(eval_csr(e, M, gi));
    // H is singular along the constant vector: the part of g along it (the
    // rounding-level difference between the computed total mass and sum(nu))
    // cannot be corrected by any step.  Removing it spreads that difference
    // over all cells instead of leaving it in the gauge cell, where it would
    // set a floor of |sum g| / nu_gauge on the max relative error.
    hipLaunchKernelGGL(k_add_const, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream,
                       n, S.g.p, -ns.sumg / (double)n);
    const ma_status ps = pcg(e, M, gi, S.g.p, S.d.p, rel, o.cg_maxiter, o.preconditioner, &it,
                             &rr);
    st.cg_iter += it;
    if (ps != MA_OK) {
      // no usable Newton direction: stop at the last accepted weights
      // (include/MA/optimal_transport.hpp:48-58,67-79 reports the same two
      // failures)
      if (ps != MA_SINGULAR && ps != MA_LINEAR_FAIL) return ps;
      result = ps;
      break;
    }
    hipLaunchKernelGGL(k_neg, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream, n, S.d.p);
    MA_HIP_TRY(hipStreamSynchronize(e->stream));
    ms_lin += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    // close to the FP32 scatter the step lands at about that scatter: its
    // trial points are evaluated in FP64 (the step itself was taken from the
    // FP32 evaluation), which spares an FP64 re-evaluation at the same point
    if (fp32_phase && ns.l2 <= kNoiseRatio * noise_l2) {
      fp32_phase = false;
      after_fp32 = true;
    }
    // backtracking (optimal_transport.hpp:158-176)
    double alpha = 1.0;
    const double n0 = ns.l2;
    const NewtonStats ns0 = ns;
    while (true) {
      MA_HIP_TRY(hipMemsetAsync(S.moved.p, 0, sizeof(int32_t), e->stream));
      if (dd)
        hipLaunchKernelGGL(k_axpy_dd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream,
                           n, S.w.p, S.wl.p, alpha, S.d.p, S.wtrial.p, S.wtl.p, S.moved.p);
      else
        hipLaunchKernelGGL(k_axpy_to, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                           e->stream, n, S.w.p, alpha, S.d.p, S.wtrial.p, S.moved.p);
      int32_t moved = 0;
      MA_HIP_TRY(read_back(e, {{&moved, S.moved.p, sizeof(int32_t)}}));
      if (!moved) {
        // alpha d is below half an ulp of every weight: the trial point is
        // the iterate itself, and so is every shorter step (the weights'
        // resolution, not the step length, ends the search)
        result = MA_LINESEARCH_FAIL;
        e->err = "step below the resolution of the weights";
        ns = ns0;
        break;
      }
      s = eval_at(S.wtrial.p, S.wtl.p, fval, ns);
      if (s != MA_OK) return s;
      if (ns.minm >= eps0 && ns.l2 <= (1.0 - alpha / 2.0) * n0) break;
      if (!dd && alpha == 1.0 && !fp32_phase && ns0.maxrel < kFloorCheck && e->have_hessian) {
        // a full step that does not lower the error this close to the
        // solution: if the error is already at the weights' representability
        // floor, no shorter step can help either (each would only be
        // evaluated to find that out)
        double floor = 0.0;
        const ma_status fs = weight_floor(e, S.w.p, S.nu.p, &floor);
        if (fs != MA_OK) return fs;
        if (ns0.maxrel <= kFloorMargin * floor) {
          // (the norm of the error is rounding here and need not halve while
          // the last cells above the tolerance come below it)
          if (ns.minm >= eps0 && !keep_going(ns)) break;
          result = MA_LINESEARCH_FAIL;
          char msg[160];
          snprintf(msg, sizeof msg,
                   "max relative mass error %.3g is at the representability floor of the FP64 "
                   "weights (%.3g)", ns0.maxrel, floor);
          e->err = msg;
          ns = ns0;
          break;
        }
      }
      alpha *= 0.5;
      if (alpha < o.alpha_min) {
        result = MA_LINESEARCH_FAIL;
        e->err = "step length below alpha_min";
        ns = ns0;
        break;
      }
    }
    if (result != MA_OK) break;
    S.w.swap(S.wtrial);
    if (dd) S.wl.swap(S.wtl);
    // leave the FP32 phase at kSwitch, or earlier when FP32 progress stalls
    // close to its accuracy floor (a damped step, or less than a halving of
    // the error, once below kStall)
    if (fp32_phase && (ns.maxrel <= kSwitch ||
                       (ns0.maxrel < kStall && (alpha < 1.0 || ns.maxrel > 0.5 * ns0.maxrel)))) {
      // near the FP32 accuracy floor the FP32 residual is mostly rounding:
      // take the next direction from an FP64 evaluation at the same point
      fp32_phase = false;
      after_fp32 = true;
      s = eval_at(S.w.p, S.wl.p, fval, ns);
      if (s != MA_OK) return s;
    }
    if (o.verbose)
      fprintf(stderr, "it %lld: f=%.17g |df|=%.6g maxrel=%.3g tau=%g eval=%lld cg=%lld\n",
              (long long)niter, fval - ns.nuw, ns.l2, ns.maxrel, alpha, (long long)st.neval,
              (long long)it);
  }
  if ((result == MA_LINESEARCH_FAIL || result == MA_LINEAR_FAIL) && e->have_hessian) {
    // a diagram in several pieces (a domain with separate components) has a
    // singular Newton system: the gauge fixes one piece only, and targets
    // that do not match each piece's mass cannot be met.  After a failed
    // line search the last evaluation is a rejected trial point, whose empty
    // cells would show as isolated rows: the graph is taken at the weights
    // kept, evaluated again (FP64), which also leaves the engine's last
    // evaluation at the weights returned.
    if (result == MA_LINESEARCH_FAIL) {
      const std::string why = e->err;
      fp32_phase = false;
      s = eval_at(S.w.p, S.wl.p, fval, ns);
      if (s != MA_OK) return s;
      e->err = why;
    }
    bool connected = true;
    const ma_status cs = diagram_connected(e, &connected);
    if (cs != MA_OK) return cs;
    if (!connected) {
      result = MA_SINGULAR;
      e->err = "singular Newton system: the Laguerre diagram is disconnected (the density's "
               "support has separate components), so the gauge fixes only one of them";
    }
  }
  st.niter = niter;
  st.max_rel_err = ns.maxrel;
  st.l2_err = ns.l2;
  st.fval = fval - ns.nuw;
  st.ms_eval = ms_eval;
  st.ms_linear = ms_lin;
  MA_HIP_TRY(from_morton(e, S.w.p, w, false));
  if (dd) MA_HIP_TRY(from_morton(e, S.wl.p, w_lo, false));
  st.ms_total =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
  if (stats) *stats = st;
  return result;
}

ma_status ma_adjoint(ma_engine *e, const double *w, double *dY, double *dval) {
  ma_status s = need(e);
  if (s != MA_OK) return s;
  if (!w) return MA_BAD_INPUT;
  MA_HIP_TRY(e->eb.w_s.ensure((size_t)e->n));
  MA_HIP_TRY(to_morton(e, w, e->eb.w_s.p, false));
  return adjoint(e, dY, dval);
}

ma_status ma_set_option(ma_engine *e, int option, int64_t value) {
  if (!e) return MA_BAD_INPUT;
  switch (option) {
    case MA_OPT_FORCE_GENERAL:
      if (value < 0 || value > 2) return MA_BAD_INPUT;
      e->force_general = (int)value;
      return MA_OK;
    case MA_OPT_CAP_CAND:
      if (value < 4 || value > 4096) return MA_BAD_INPUT;
      e->cap_cand = (int)value;
      return MA_OK;
    case MA_OPT_GRAPHS:
      e->use_graphs = value != 0;
      return MA_OK;
    case MA_OPT_LOCAL_RINGS:
      if (value < 0 || value > 64) return MA_BAD_INPUT;
      e->local_rings = (int)value;
      return MA_OK;
    case MA_OPT_WALK_BUDGET:
      if (value < 0 || value > (1 << 20)) return MA_BAD_INPUT;
      e->walk_budget = (int)value;
      return MA_OK;
    case MA_OPT_AMG_OMEGA:
      if (value < 100 || value > 1000) return MA_BAD_INPUT;
      e->amg_omega = value * 1e-3;
      return MA_OK;
    case MA_OPT_AMG_CORR:
      if (value < 500 || value > 3000) return MA_BAD_INPUT;
      e->amg_corr = value * 1e-3;
      return MA_OK;
    case MA_OPT_AMG_SWEEPS:
      if (value != 1 && value != 2) return MA_BAD_INPUT;
      e->amg_sweeps = (int)value;
      return MA_OK;
    case MA_OPT_FAR_CELLS:
      if (value != 0 && value != 1) return MA_BAD_INPUT;
      e->far_cells = (int)value;
      return MA_OK;
    default:
      return MA_BAD_INPUT;
  }
}

ma_status ma_get_eval_info(const ma_engine *e, ma_eval_info *info) {
  if (!e || !info) return MA_BAD_INPUT;
  *info = e->info;
  return MA_OK;
}

ma_status ma_cell_paths(ma_engine *e, int64_t count, const int64_t *ids, int32_t *out) {
  if (!e || count < 0 || (count > 0 && (!ids || !out))) return MA_BAD_INPUT;
  if (!e->have_eval) {
    e->err = "no evaluation yet";
    return MA_NO_DATA;
  }
  std::vector<int32_t> pn(e->n), iperm(e->n);
  MA_HIP_TRY(hipMemcpyAsync(pn.data(), e->eb.pn.p, sizeof(int32_t) * e->n, hipMemcpyDeviceToHost,
                            e->stream));
  MA_HIP_TRY(hipMemcpyAsync(iperm.data(), e->iperm.p, sizeof(int32_t) * e->n,
                            hipMemcpyDeviceToHost, e->stream));
  MA_HIP_TRY(hipStreamSynchronize(e->stream));
  for (int64_t i = 0; i < count; i++) {
    if (ids[i] < 0 || ids[i] >= e->n) return MA_BAD_INPUT;
    out[i] = std::max(pn[iperm[ids[i]]], -1);
  }
  return MA_OK;
}

}  // extern "C"

namespace ma {

// dPhi/dy_k = int_{Lag_k} rho 2 (y_k - x) dx = -2 (first moment about y_k),
// written in the caller's order (interleaved x, y).
__global__ void k_adjoint_dy(int64_t n, const int32_t *perm, const double *mom_local,
                             double *dy) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int64_t i = perm[k];
  dy[2 * i] = -2.0 * mom_local[2 * k];
  dy[2 * i + 1] = -2.0 * mom_local[2 * k + 1];
}

// Partial derivatives of the dual value Phi(Y, w, rho) = int rho(x) min_i
// (|x - y_i|^2 - w_i) dx at fixed weights.  At the optimal weights they are
// the derivatives of W2^2 (envelope theorem): the centroid form 2 m_i (y_i -
// b_i) of include/MA/lloyd.hpp:126-144 for the positions, and
// sum_i int_{Lag_i} (|x - y_i|^2 - w_i) phi_v(x) dx for the vertex values.
ma_status adjoint(ma_engine *e, double *dY, double *dval) {
  EvalBuffers &B = e->eb;
  MA_HIP_TRY(B.dval.ensure((size_t)e->nv));
  MA_HIP_TRY(hipMemsetAsync(B.dval.p, 0, sizeof(double) * e->nv, e->stream));
  ma_status s = evaluate(e, 2, nullptr);
  if (s != MA_OK) return s;
  if (dY) {
    DBuf<double> &tmp = e->cb.xy;
    MA_HIP_TRY(tmp.ensure((size_t)(2 * e->n)));
    hipLaunchKernelGGL(k_adjoint_dy, dim3((unsigned)((e->n + 127) / 128)), dim3(128), 0,
                       e->stream, e->n, e->perm.p, B.mom_s.p, tmp.p);
    MA_HIP_TRY(hipMemcpyAsync(dY, tmp.p, sizeof(double) * 2 * e->n, hipMemcpyDeviceToHost,
                              e->stream));
    MA_HIP_TRY(hipStreamSynchronize(e->stream));
  }
  if (dval) {
    MA_HIP_TRY(hipMemcpyAsync(dval, B.dval.p, sizeof(double) * e->nv, hipMemcpyDeviceToHost,
                              e->stream));
    MA_HIP_TRY(hipStreamSynchronize(e->stream));
  }
  return MA_OK;
}
}  // namespace ma
