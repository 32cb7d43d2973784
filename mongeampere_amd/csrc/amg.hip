// Aggregation multigrid preconditioner for the gauge-fixed Hessian (a
// weighted graph Laplacian of the power diagram) and the conjugate gradient
// that uses it.  Replaces the sparse direct factorisation of
// solve_laplacian_matrix (include/MA/optimal_transport.hpp:41-87).
//
// Hierarchy: aggregates are runs of kAgg consecutive unknowns in Morton
// order (spatially compact groups of Diracs), prolongation is piecewise
// constant, coarse operators are Galerkin products P^T A P.  Because the
// aggregate map i -> i / kAgg is monotone, a coarse row is the merge of
// kAgg sorted fine rows.  Cycle: V(1,1) (or V(2,2)) with damped Jacobi
// (omega, default 0.85), coarse correction scaled by corr (default 1.5:
// over-correction for piecewise-constant prolongation), dense inverse at the
// coarsest level.  The defaults minimise the linear-solve time of the
// N = 1M Newton solve over a sweep of omega in [0.6, 1], corr in [1, 2] and
// both cycles: V(1,1) takes ~55 % more CG iterations than V(2,2) (~440
// against ~285) at ~60 % of the cost per iteration (120 against 128 ms per
// solve); omega 2/3 or 1, or corr 1 or 2, cost 10-200 % more.
//
// The hierarchy's values, diagonals and work vectors are FP64 or FP32 (T);
// row products accumulate in FP64 either way.  The conjugate gradient's own
// operator is the FP64 gauge-fixed level-0 matrix (val0), kept apart, so an
// FP32 hierarchy changes only the preconditioner's rounding: the residuals
// and the stopping test stay FP64.  FP32 halves the bytes of the values and
// vectors the fine-level sweeps move.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <type_traits>

#include "geom_common.h"
#include "lanes.h"

namespace ma {

constexpr int kAgg = 4;
constexpr int kCoarsest = 192;   // dense solve at or below this size
constexpr int kVB2 = 256;

// ---------------------------------------------------------------------------
// Setup
// ---------------------------------------------------------------------------

// Level 0: the Hessian with row and column gi removed (identity there), so
// the system is SPD and the solution keeps x[gi] = 0.  A row other than gi
// without a positive diagonal (a cell sharing no edge, or a NaN) sets bit 0 of
// *bad, one that is not in column order bit 1.
// With outf, also an FP32 copy of the values and inverse diagonal.
__global__ void k_amg_level0(int64_t n, const int32_t *ptr, const int32_t *col,
                             const double *val, int32_t gi, double *out, double *dinv,
                             float *outf, float *dinvf, int32_t *bad) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  double d = 0.0;
  int32_t last = 0;
  bool descends = false;
  for (int32_t q = ptr[i]; q < ptr[i + 1]; q++) {
    const int32_t j = col[q];
    descends |= j < last;
    last = j;
    double v = val[q];
    if (i == gi || j == gi) v = (i == j) ? 1.0 : 0.0;
    out[q] = v;
    if (outf) outf[q] = (float)v;
    if (j == i) d = v;
  }
  if (i == gi) d = 1.0;
  dinv[i] = d > 0.0 ? 1.0 / d : 0.0;
  if (dinvf) dinvf[i] = (float)dinv[i];
  if (!(d > 0.0)) atomicOr(bad, 1);
  if (descends) atomicOr(bad, 2);
}

// Brings the rows of M into column order, on the host (a caller's matrix may
// come in any order; the engine's rows never take this).  Coarse rows are
// merges of rows in that order: of others they would hold columns twice, more
// entries than amg_build has room for.
static hipError_t sort_rows(ma_engine *e, const CsrView &M) {
  std::vector<int32_t> ptr((size_t)M.n + 1), col((size_t)M.nnz);
  std::vector<double> val((size_t)M.nnz);
  MA_HIP_RET(hipMemcpyAsync(ptr.data(), M.ptr, sizeof(int32_t) * ptr.size(),
                            hipMemcpyDeviceToHost, e->stream));
  MA_HIP_RET(hipMemcpyAsync(col.data(), M.col, sizeof(int32_t) * col.size(),
                            hipMemcpyDeviceToHost, e->stream));
  MA_HIP_RET(hipMemcpyAsync(val.data(), M.val, sizeof(double) * val.size(),
                            hipMemcpyDeviceToHost, e->stream));
  MA_HIP_RET(hipStreamSynchronize(e->stream));
  std::vector<std::pair<int32_t, double>> row;
  for (int64_t i = 0; i < M.n; i++) {
    row.clear();
    for (int32_t q = ptr[i]; q < ptr[i + 1]; q++) row.emplace_back(col[q], val[q]);
    std::stable_sort(row.begin(), row.end(),
                     [](const auto &a, const auto &b) { return a.first < b.first; });
    for (size_t q = 0; q < row.size(); q++) {
      col[ptr[i] + q] = row[q].first;
      val[ptr[i] + q] = row[q].second;
    }
  }
  MA_HIP_RET(hipMemcpyAsync(M.own_col, col.data(), sizeof(int32_t) * col.size(),
                            hipMemcpyHostToDevice, e->stream));
  MA_HIP_RET(hipMemcpyAsync(M.own_val, val.data(), sizeof(double) * val.size(),
                            hipMemcpyHostToDevice, e->stream));
  return hipStreamSynchronize(e->stream);
}

// Merge of the kAgg sorted fine rows of coarse row I (columns mapped j/kAgg).
template <bool FILL, class T>
__device__ inline void coarse_row(int64_t I, int64_t n, const int32_t *ptr, const int32_t *col,
                                  const T *val, int32_t *cnt_or_ptr, int32_t *ccol, T *cval,
                                  T *cdinv) {
  int32_t pos[kAgg], end[kAgg];
#pragma unroll
  for (int r = 0; r < kAgg; r++) {
    const int64_t i = I * kAgg + r;
    pos[r] = (i < n) ? ptr[i] : 0;
    end[r] = (i < n) ? ptr[i + 1] : 0;
  }
  int32_t o = FILL ? cnt_or_ptr[I] : 0;
  int32_t cnt = 0;
  double diag = 0.0;
  while (true) {
    int32_t cmin = INT32_MAX;
#pragma unroll
    for (int r = 0; r < kAgg; r++)
      if (pos[r] < end[r]) cmin = min(cmin, col[pos[r]] / kAgg);
    if (cmin == INT32_MAX) break;
    double s = 0.0;
#pragma unroll
    for (int r = 0; r < kAgg; r++)
      while (pos[r] < end[r] && col[pos[r]] / kAgg == cmin) {
        s += (double)val[pos[r]];
        pos[r]++;
      }
    if (FILL) {
      ccol[o + cnt] = cmin;
      cval[o + cnt] = (T)s;
      if (cmin == I) diag = s;
    }
    cnt++;
  }
  if (FILL)
    cdinv[I] = (T)(diag > 0.0 ? 1.0 / diag : 0.0);
  else
    cnt_or_ptr[I] = cnt;
}

template <bool FILL, class T>
__global__ void k_amg_coarse(int64_t nc, int64_t n, const int32_t *ptr, const int32_t *col,
                             const T *val, int32_t *cnt_or_ptr, int32_t *ccol, T *cval,
                             T *cdinv) {
  const int64_t I = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (I < nc) coarse_row<FILL, T>(I, n, ptr, col, val, cnt_or_ptr, ccol, cval, cdinv);
}
// The same with one wave per coarse row: the kAgg fine rows are consecutive, so
// lane e takes their e-th entry, sums the entries of its column (in the order
// of the merge) and, if it is the first of them, writes the column at its rank.
// A thread's merge is a chain of dependent loads: on levels with few rows it
// took 35 (count) and 53 us (fill) against 7 and 12 us here; with many rows its
// fewer instructions win (250k coarse rows: 43 and 73 us, against about 90
// each), hence kWaveRows.  Rows of more than 64 entries are merged by lane 0.
constexpr int64_t kWaveRows = 65536;
template <bool FILL, class T>
__global__ void __launch_bounds__(kVB2) k_amg_coarse_wave(int64_t nc, int64_t n,
                                                          const int32_t *ptr, const int32_t *col,
                                                          const T *val, int32_t *cnt_or_ptr,
                                                          int32_t *ccol, T *cval, T *cdinv) {
  const int64_t I = (blockIdx.x * (int64_t)kVB2 + threadIdx.x) >> 6;
  if (I >= nc) return;
  const int lane = (int)threadIdx.x & 63;
  const int32_t p0 = ptr[I * kAgg], p1 = ptr[min(I * kAgg + kAgg, n)];
  const int tot = __builtin_amdgcn_readfirstlane(p1 - p0);
  if (tot > 64) {
    if (lane == 0)
      coarse_row<FILL, T>(I, n, ptr, col, val, cnt_or_ptr, ccol, cval, cdinv);
    return;
  }
  const int key = lane < tot ? col[p0 + lane] / kAgg : INT32_MAX;
  const double v = FILL && lane < tot ? (double)val[p0 + lane] : 0.0;
  const int vhi = __double2hiint(v), vlo = __double2loint(v);
  bool first = lane < tot;
  double s = 0.0;
  for (int e = 0; e < tot; e++) {
    const bool eq = __builtin_amdgcn_readlane(key, e) == key;
    if (eq && e < lane) first = false;
    if (FILL) {
      const double ve = __hiloint2double(__builtin_amdgcn_readlane(vhi, e),
                                         __builtin_amdgcn_readlane(vlo, e));
      if (eq) s += ve;
    }
  }
  const unsigned long long heads = __ballot(first);
  if (!FILL) {
    if (lane == 0) cnt_or_ptr[I] = __popcll(heads);
    return;
  }
  int rank = 0;
  for (unsigned long long m = heads; m; m &= m - 1)
    rank += __builtin_amdgcn_readlane(key, __ffsll((long long)m) - 1) < key;
  if (first) {
    const int32_t o = cnt_or_ptr[I] + rank;
    ccol[o] = key;
    cval[o] = (T)s;
  }
  const unsigned long long dg = __ballot(first && key == (int)I);
  if (dg ? first && key == (int)I : lane == 0)
    cdinv[I] = (T)(dg && s > 0.0 ? 1.0 / s : 0.0);
}

// Inverse of the coarsest matrix (symmetric positive definite) by in-place
// Gauss-Jordan elimination without pivoting, one workgroup: thread (tx, ty) of
// 32 x 32 keeps elements (ty + 32 a, tx + 32 b) in registers, and a step
// passes its pivot row and column through LDS (double buffered: one barrier a
// step).  A non-positive pivot (a disconnected piece) counts as 1.  Bound by
// the FP64 rate of its one compute unit; at 157 unknowns 175 us, against 1.7
// ms for a Cholesky factor in global memory and 2.8 ms for its inverse with
// one thread per column (serial chains of global loads).
constexpr int kDenseSide = 32;
template <int TILES, class T>
__global__ void __launch_bounds__(kDenseSide *kDenseSide) k_amg_dense_inv(
    int n, const int32_t *ptr, const int32_t *col, const T *val, double *inv) {
  __shared__ double srow[2][kDenseSide * TILES], scol[2][kDenseSide * TILES];
  const int tid = (int)threadIdx.x, tx = tid % kDenseSide, ty = tid / kDenseSide;
  for (int q = tid; q < n * n; q += kDenseSide * kDenseSide) inv[q] = 0.0;
  __syncthreads();
  for (int i = tid; i < n; i += kDenseSide * kDenseSide)
    for (int32_t q = ptr[i]; q < ptr[i + 1]; q++) inv[i * n + col[q]] = (double)val[q];
  __syncthreads();
  double A[TILES][TILES];
#pragma unroll
  for (int a = 0; a < TILES; a++)
#pragma unroll
    for (int b = 0; b < TILES; b++) {
      const int i = ty + kDenseSide * a, j = tx + kDenseSide * b;
      A[a][b] = i < n && j < n ? inv[i * n + j] : 0.0;
    }
  // row and column k to LDS
  auto publish = [&](int k) {
    const int t = k / kDenseSide, r = k % kDenseSide;
#pragma unroll
    for (int c = 0; c < TILES; c++)
      if (c == t) {
        if (ty == r) {
#pragma unroll
          for (int b = 0; b < TILES; b++) srow[k & 1][tx + kDenseSide * b] = A[c][b];
        }
        if (tx == r) {
#pragma unroll
          for (int a = 0; a < TILES; a++) scol[k & 1][ty + kDenseSide * a] = A[a][c];
        }
      }
  };
  publish(0);
  for (int k = 0; k < n; k++) {
    __syncthreads();
    const double d = srow[k & 1][k];
    const double ip = 1.0 / (d > 0.0 ? d : 1.0);
    double r[TILES], c[TILES];
#pragma unroll
    for (int b = 0; b < TILES; b++) r[b] = srow[k & 1][tx + kDenseSide * b] * ip;
#pragma unroll
    for (int a = 0; a < TILES; a++) c[a] = scol[k & 1][ty + kDenseSide * a];
#pragma unroll
    for (int a = 0; a < TILES; a++)
#pragma unroll
      for (int b = 0; b < TILES; b++) A[a][b] -= c[a] * r[b];
    const int t = k / kDenseSide, q = k % kDenseSide;
#pragma unroll
    for (int e = 0; e < TILES; e++)
      if (e == t) {
        if (ty == q) {
#pragma unroll
          for (int b = 0; b < TILES; b++) A[e][b] = r[b];
        }
        if (tx == q) {
#pragma unroll
          for (int a = 0; a < TILES; a++) A[a][e] = -c[a] * ip;
          if (ty == q) A[e][e] = ip;
        }
      }
    if (k + 1 < n) publish(k + 1);
  }
#pragma unroll
  for (int a = 0; a < TILES; a++)
#pragma unroll
    for (int b = 0; b < TILES; b++) {
      const int i = ty + kDenseSide * a, j = tx + kDenseSide * b;
      if (i < n && j < n) inv[i * n + j] = A[a][b];
    }
}

// ---------------------------------------------------------------------------
// Cycle kernels (all return at once when the conjugate gradient has
// converged: done[0] != 0).  T: values, diagonals and coarse vectors; TB,
// TX, TY: right-hand side, iterate and output (FP64 at level 0, where they
// are the conjugate gradient's r and z).
//
// Up to a few hundred thousand rows a cycle is bound by the number of its
// launches (3-5 us each on the coarse levels, most of it the chain row pointer
// -> entry -> gather and the gap to the next launch), so that what fits into a
// neighbour is part of it: level 0's first sweep comes from the residual update of the
// conjugate gradient, a coarse level's from the restriction above it, r.z
// from level 0's last sweep, and the levels of at most kTailRows rows with
// the dense solve are one workgroup's work.
// ---------------------------------------------------------------------------
// y = x + omega (b - A x) / D; rows are read by groups of kRowLanes lanes
// (consecutive entries of consecutive rows: coalesced).  With xc the first
// sweep after the coarse correction: x' = x + corr xc[. / kAgg], formed on
// the fly, takes the place of x.  DOT: cg_grid(n) workgroups of
// kCgThreads threads, and the partial sums of b.y go to part.
template <bool DOT, bool CORR, class T, class TB, class TX, class TY>
__global__ void __launch_bounds__(DOT ? kCgThreads : kVB2)
    k_amg_smooth(int64_t n, const int32_t *ptr, const int32_t *col, const T *val, const T *dinv,
                 const TB *b, const TX *x, const T *xc, TY *y, double *part, const double *done,
                 double kOmega, double kCorr) {
  const int lane = (int)threadIdx.x % kRowLanes;
  auto at = [&](int64_t j) {
    return CORR ? (double)x[j] + kCorr * (double)xc[j / kAgg] : (double)x[j];
  };
  int64_t i = xcd_share(blockIdx.x, gridDim.x) * (kVB2 / kRowLanes), last = n;
  if (DOT) cg_rows(n, i, last);
  i += threadIdx.x / kRowLanes;
  RowHead<T> row;
  row.load(ptr, col, val, i, i < last, lane);
  if (*done != 0.0) return;
  double acc = 0.0;
  while (i < last) {  // a group's lanes go together
    const double ax = row.dot(col, val, at);
    if (lane == 0) {
      const double bi = (double)b[i];
      const TY v = (TY)(at(i) + kOmega * (bi - ax) * (double)dinv[i]);
      y[i] = v;
      acc += bi * (double)v;
    }
    if (!DOT) return;
    i += kCgGroups;
    row.load(ptr, col, val, i, i < last, lane);
  }
  if (DOT) {
    __shared__ double s[kCgThreads / 64];
    acc = cg_block_sum(acc, s);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
  }
}
// bc[I] = sum over the aggregate of (b - A x): kAgg rows x kRowLanes lanes;
// with dinv_c, also the coarse level's first smoothing sweep from zero,
// yc = omega bc / Dc (saves that level a launch)
template <class T, class TB, class TX>
__global__ void __launch_bounds__(kVB2)
    k_amg_restrict(int64_t nc, int64_t n, const int32_t *ptr, const int32_t *col, const T *val,
                   const TB *b, const TX *x, T *bc, const T *dinv_c, T *yc, const double *done,
                   double kOmega) {
  constexpr int kLanes = kAgg * kRowLanes;
  const int64_t t = xcd_share(blockIdx.x, gridDim.x) * kVB2 + threadIdx.x;
  const int64_t I = t / kLanes;
  const int lane = (int)(t % kLanes);
  const int64_t i = I * kAgg + lane / kRowLanes;
  const bool valid = I < nc && i < n;
  RowHead<T> row;
  row.load(ptr, col, val, i, valid, lane % kRowLanes);
  if (*done != 0.0) return;
  const double ax = row.dot(col, val, [&](int64_t j) { return (double)x[j]; });
  double s = (valid && lane % kRowLanes == 0) ? (double)b[i] - ax : 0.0;
  for (int o = kRowLanes; o < kLanes; o <<= 1) s += __shfl_xor(s, o, kLanes);
  if (I < nc && lane == 0) {
    bc[I] = (T)s;
    if (dinv_c) yc[I] = (T)(kOmega * s * (double)dinv_c[I]);
  }
}

// The last levels of a cycle, one workgroup: the smoothed levels lv[0 .. nlev)
// (at most kTailRows rows, each level a kAgg-th of the one before) and the
// dense solve below them, with the vectors in LDS.  b, y: the first level's
// right-hand side and first sweep (nlev = 0: the dense solve's right-hand
// side); x: its result.  With part the one partial sum of b.x goes there
// (nlev = 0).  Bound by the chain of its steps (load, residual, restriction,
// dense solve, correction): 8.7 us for 250 + 63 rows in FP32, 13.8 us for
// 586 + 147 in FP64, against the three or five launches it replaces.  More
// rows would not fit the registers of one pass and take a second one of about
// the length of a launch.
constexpr int kTailRows = 1024, kTailLevels = 2, kTailThreads = 1024;
static_assert(kTailRows <= kCoarsest * kAgg * kAgg, "smoothed levels of the tail");
template <class T>
struct TailLevel {
  int n;
  const int32_t *ptr, *col;
  const T *val, *dinv;
};
template <class T>
struct Tail {
  TailLevel<T> lv[kTailLevels];
  int nlev, nd;          // smoothed levels; rows of the dense level
  const double *inv;
  double omega, corr;
  int two;               // V(2,2)
};
// A level's rows, all of them at once and kept in registers: groups of
// kRowLanes lanes, N rows each, two entries of a row per lane (rows of more
// entries, few, are read on from memory).
constexpr int kTailGroups = kTailThreads / kRowLanes;
template <int N, class T>
struct TailRows {
  int32_t c[N][2];
  T v[N][2];
  unsigned lng = 0;  // bit r: row r goes on
  __device__ inline void load(const TailLevel<T> &L, int lane) {
    const int i0 = (int)threadIdx.x / kRowLanes;
    int32_t q[N], e[N];
#pragma unroll
    for (int r = 0; r < N; r++) {
      const int i = min(i0 + r * kTailGroups, L.n - 1);
      q[r] = L.ptr[i] + lane;
      e[r] = L.ptr[i + 1];
    }
#pragma unroll
    for (int r = 0; r < N; r++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        // (an empty slot: 0 times the row's own unknown)
        c[r][k] = min(i0 + r * kTailGroups, L.n - 1);
        v[r][k] = (T)0;
        if (q[r] + k * kRowLanes < e[r]) {
          c[r][k] = L.col[q[r] + k * kRowLanes];
          v[r][k] = L.val[q[r] + k * kRowLanes];
        }
        if (q[r] + 2 * kRowLanes < e[r]) lng |= 1u << r;
      }
  }
  // f(i, A x at row i) on lane 0 of row i's group
  template <class X, class F>
  __device__ inline void each(const TailLevel<T> &L, X &&x, F &&f) const {
    const int i0 = (int)threadIdx.x / kRowLanes, lane = (int)threadIdx.x % kRowLanes;
    double s[N];
#pragma unroll
    for (int r = 0; r < N; r++) {
      s[r] = (double)v[r][0] * x(c[r][0]);
      s[r] += (double)v[r][1] * x(c[r][1]);
    }
    if (lng)
#pragma unroll
      for (int r = 0; r < N; r++)
        if (lng >> r & 1) {
          const int i = min(i0 + r * kTailGroups, L.n - 1);
          for (int32_t k = L.ptr[i] + lane + 2 * kRowLanes; k < L.ptr[i + 1]; k += kRowLanes)
            s[r] += (double)L.val[k] * x(L.col[k]);
        }
#pragma unroll
    for (int r = 0; r < N; r++) {
      s[r] = oct_sum(s[r]);
      if (lane == 0 && i0 + r * kTailGroups < L.n) f(i0 + r * kTailGroups, s[r]);
    }
  }
};
template <class T, class TB, class TX>
__global__ void __launch_bounds__(kTailThreads)
    k_amg_tail(Tail<T> t, const TB *b, const T *y, TX *x, double *part, const double *done) {
  // every level's vectors after those of the one before
  constexpr int kAll = kTailRows + kTailRows / kAgg + kCoarsest;
  __shared__ T sy[kAll], sx[kAll], sd[kTailRows + kTailRows / kAgg];
  __shared__ double sb[kAll], res[kTailRows];
  const int tid = (int)threadIdx.x, lane = tid % kRowLanes;
  const int n0 = t.nlev ? t.lv[0].n : t.nd, n1 = t.nlev > 1 ? t.lv[1].n : 0;
  const double om = t.omega, co = t.corr;
  // the levels' first entries, loaded with the vectors and kept for the way up
  TailRows<kTailRows / kTailGroups, T> rows0;
  TailRows<kTailRows / kTailGroups / kAgg, T> rows1;
  if (t.nlev) rows0.load(t.lv[0], lane);
  if (t.nlev > 1) rows1.load(t.lv[1], lane);
  for (int i = tid; i < n0; i += kTailThreads) {
    sb[i] = (double)b[i];
    if (t.nlev) {
      sy[i] = y[i];
      sd[i] = t.lv[0].dinv[i];
    }
  }
  for (int i = tid; i < n1; i += kTailThreads) sd[n0 + i] = t.lv[1].dinv[i];
  if (*done != 0.0) return;
  __syncthreads();
  // down from a level at off: smooth (V(2,2)), residual, restriction
  auto down = [&](const TailLevel<T> &L, const auto &rows, int off, int nc, bool smoothed) {
    const T *v = sy + off;
    if (t.two) {
      rows.each(L, [&](int j) { return (double)sy[off + j]; }, [&](int i, double ax) {
        sx[off + i] = (T)((double)sy[off + i] + om * (sb[off + i] - ax) * (double)sd[off + i]);
      });
      __syncthreads();
      v = sx + off;
    }
    rows.each(L, [&](int j) { return (double)v[j]; },
              [&](int i, double ax) { res[i] = sb[off + i] - ax; });
    __syncthreads();
    const int oc = off + L.n;
    for (int I = tid; I < nc; I += kTailThreads) {
      double a[kAgg];
#pragma unroll
      for (int k = 0; k < kAgg; k++) a[k] = I * kAgg + k < L.n ? res[I * kAgg + k] : 0.0;
      static_assert(kAgg == 4, "sum of an aggregate in the order of k_amg_restrict");
      const double s = (a[0] + a[1]) + (a[2] + a[3]);
      sb[oc + I] = (double)(T)s;
      if (smoothed) sy[oc + I] = (T)(om * s * (double)sd[oc + I]);
    }
    __syncthreads();
  };
  // up to a level at off: correction from the level after it, smooth; the
  // first level's result goes to x
  auto up = [&](const TailLevel<T> &L, const auto &rows, int off, bool out) {
    __syncthreads();
    const T *xc = sx + off + L.n, *v = t.two ? sx + off : sy + off;
    auto at = [&](int j) { return (double)v[j] + co * (double)xc[j / kAgg]; };
    rows.each(L, at, [&](int i, double ax) {
      const T u = (T)(at(i) + om * (sb[off + i] - ax) * (double)sd[off + i]);
      if (t.two)
        sy[off + i] = u;
      else if (out)
        x[i] = (TX)u;
      else
        sx[off + i] = u;
    });
    if (!t.two) return;
    __syncthreads();
    rows.each(L, [&](int j) { return (double)sy[off + j]; }, [&](int i, double ax) {
      const T u = (T)((double)sy[off + i] + om * (sb[off + i] - ax) * (double)sd[off + i]);
      if (out)
        x[i] = (TX)u;
      else
        sx[off + i] = u;
    });
  };
  if (t.nlev) down(t.lv[0], rows0, 0, t.nlev > 1 ? n1 : t.nd, t.nlev > 1);
  if (t.nlev > 1) down(t.lv[1], rows1, n0, t.nd, false);
  {
    // coarsest: x = A^-1 b, 16 lanes per row, a group's rows together
    constexpr int kGroups = kTailThreads / kGroup, kRows = kCoarsest / kGroups;
    static_assert(kCoarsest % kGroups == 0, "rows of the dense solve");
    const int l = tid & (kGroup - 1), i0 = tid / kGroup, N = t.nd;
    const int off = t.nlev ? n0 + n1 : 0;
    const double *row[kRows];
    double s[kRows], dot = 0.0;
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      row[r] = t.inv + min(i0 + r * kGroups, N - 1) * N;
      s[r] = 0.0;
    }
#pragma unroll 6
    for (int k = l; k < N; k += kGroup)
#pragma unroll
      for (int r = 0; r < kRows; r++) s[r] += row[r][k] * sb[off + k];
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      const double v = row_sum(s[r]);
      const int i = i0 + r * kGroups;
      if (l == 0 && i < N) {
        if (t.nlev)
          sx[off + i] = (T)v;
        else
          x[i] = (TX)v;
        dot += sb[off + i] * v;
      }
    }
    if (part) {
      dot = cg_block_sum(dot, res);
      if (tid == 0) part[0] = dot;
    }
  }
  if (t.nlev > 1) up(t.lv[1], rows1, n0, false);
  if (t.nlev) up(t.lv[0], rows0, 0, true);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
template <class T>
struct AmgLevel {
  int64_t n = 0;
  DBuf<int32_t> ptr, col;
  DBuf<T> val, dinv, x, y, b;  // level 0 of the FP64 hierarchy: val, dinv unused (val0, dinv0)
};

struct Amg {
  DBuf<double> val0, dinv0;          // gauge-fixed level-0 matrix (CG operator, Jacobi)
  std::vector<AmgLevel<double>> lv;  // FP64 hierarchy
  std::vector<AmgLevel<float>> lvf;  // FP32 hierarchy
  bool fp32 = false;                 // which one the last setup built
  DBuf<int32_t> bad;                 // zero-diagonal flag of the level-0 matrix
  DBuf<double> dense_inv;            // inverse of the coarsest matrix (one matrix-vector product)
  int nlev = 0;
  const int32_t *ptr0 = nullptr, *col0 = nullptr;  // level-0 pattern (the caller's CSR)
};

static inline unsigned nb2(int64_t n) { return (unsigned)((n + kVB2 - 1) / kVB2); }

Amg *amg_create() { return new Amg(); }
void amg_destroy(Amg *a) { delete a; }
const double *amg_level0_values(const Amg &a) { return a.val0.p; }
const double *amg_level0_dinv(const Amg &a) { return a.dinv0.p; }

static std::vector<AmgLevel<double>> &levels_of(Amg &A, double *) { return A.lv; }
static std::vector<AmgLevel<float>> &levels_of(Amg &A, float *) { return A.lvf; }
// values and inverse diagonal of level l in precision T
template <class T>
static const T *val_of(Amg &A, int l) {
  if (std::is_same<T, double>::value && l == 0) return reinterpret_cast<const T *>(A.val0.p);
  return levels_of(A, (T *)nullptr)[l].val.p;
}
template <class T>
static const T *dinv_of(Amg &A, int l) {
  if (std::is_same<T, double>::value && l == 0) return reinterpret_cast<const T *>(A.dinv0.p);
  return levels_of(A, (T *)nullptr)[l].dinv.p;
}

// Coarse levels and the coarsest dense inverse of the hierarchy in T.
template <class T>
static ma_status amg_build(ma_engine *e, Amg &A, const CsrView &M) {
  std::vector<AmgLevel<T>> &lv = levels_of(A, (T *)nullptr);
  const int64_t n = M.n;
  if (lv.empty()) lv.emplace_back();
  lv.reserve(32);
  size_t used = 1;
  lv[0].n = n;
  MA_HIP_TRY(lv[0].y.ensure((size_t)n));
  int64_t room = M.nnz;  // bound of the entries of the level being built
  while (lv[used - 1].n > kCoarsest && used < 32) {
    const size_t l = used - 1;
    const int64_t nf = lv[l].n, nc = (nf + kAgg - 1) / kAgg;
    const int32_t *fptr = (l == 0) ? M.ptr : lv[l].ptr.p;
    const int32_t *fcol = (l == 0) ? M.col : lv[l].col.p;
    const T *fval = val_of<T>(A, (int)l);
    if (lv.size() <= used) lv.emplace_back();
    AmgLevel<T> &C = lv[used++];
    C.n = nc;
    MA_HIP_TRY(C.ptr.ensure((size_t)nc + 1));
    MA_HIP_TRY(C.dinv.ensure((size_t)nc));
    MA_HIP_TRY(C.x.ensure((size_t)nc));
    MA_HIP_TRY(C.y.ensure((size_t)nc));
    MA_HIP_TRY(C.b.ensure((size_t)nc));
    const bool wave = nc <= kWaveRows;
    const dim3 grid(nb2(wave ? 64 * nc : nc));
    hipLaunchKernelGGL((wave ? k_amg_coarse_wave<false, T> : k_amg_coarse<false, T>), grid,
                       dim3(kVB2), 0, e->stream, nc, nf, fptr, fcol, fval, C.ptr.p, nullptr,
                       nullptr, nullptr);
    MA_HIP_TRY(exclusive_scan(e, C.ptr.p, C.ptr.p, nc));
    // small levels take room for as many entries as the level above has (or a
    // full matrix: rows in column order give every column once), instead of
    // waiting for their count
    if (!wave) {
      int32_t nnzc = 0;
      MA_HIP_TRY(read_back(e, {{&nnzc, C.ptr.p + nc, sizeof(int32_t)}}));
      room = nnzc;
    }
    room = std::min(room, nc * nc);
    MA_HIP_TRY(C.col.ensure((size_t)room + 1));
    MA_HIP_TRY(C.val.ensure((size_t)room + 1));
    hipLaunchKernelGGL((wave ? k_amg_coarse_wave<true, T> : k_amg_coarse<true, T>), grid,
                       dim3(kVB2), 0, e->stream, nc, nf, fptr, fcol, fval, C.ptr.p, C.col.p,
                       C.val.p, C.dinv.p);
  }
  const AmgLevel<T> &Lc = lv[used - 1];
  const int32_t *cptr = (used == 1) ? M.ptr : Lc.ptr.p;
  const int32_t *ccol = (used == 1) ? M.col : Lc.col.p;
  MA_HIP_TRY(A.dense_inv.ensure((size_t)(Lc.n * Lc.n)));
  auto dense = Lc.n <= 2 * kDenseSide ? k_amg_dense_inv<2, T>
               : Lc.n <= 4 * kDenseSide ? k_amg_dense_inv<4, T> : k_amg_dense_inv<6, T>;
  static_assert(kCoarsest <= 6 * kDenseSide, "coarsest matrix in registers");
  hipLaunchKernelGGL(dense, dim3(1), dim3(kDenseSide * kDenseSide), 0, e->stream, (int)Lc.n, cptr,
                     ccol, val_of<T>(A, (int)used - 1), A.dense_inv.p);
  A.nlev = (int)used;
  return MA_OK;
}

// Builds the hierarchy from the CSR matrix M (max_levels = 1: the
// gauge-fixed level-0 matrix only), in FP32 when fp32 is set.  Aggregation
// follows the index order, so a spatially coherent order (Morton) gives
// compact aggregates.
ma_status amg_setup(ma_engine *e, Amg &A, const CsrView &M, int32_t gi, int max_levels,
                    bool fp32) {
  const int64_t n = M.n;
  A.ptr0 = M.ptr;
  A.col0 = M.col;
  A.fp32 = fp32 && max_levels != 1;
  MA_HIP_TRY(A.val0.ensure((size_t)M.nnz + 1));
  MA_HIP_TRY(A.dinv0.ensure((size_t)n));
  float *valf = nullptr, *dinvf = nullptr;
  if (A.fp32) {
    if (A.lvf.empty()) A.lvf.emplace_back();
    MA_HIP_TRY(A.lvf[0].val.ensure((size_t)M.nnz + 1));
    MA_HIP_TRY(A.lvf[0].dinv.ensure((size_t)n));
    valf = A.lvf[0].val.p;
    dinvf = A.lvf[0].dinv.p;
  }
  MA_HIP_TRY(A.bad.ensure(1));
  int32_t bad = 0;
  for (int pass = 0; pass < 2; pass++) {
    MA_HIP_TRY(hipMemsetAsync(A.bad.p, 0, sizeof(int32_t), e->stream));
    hipLaunchKernelGGL(k_amg_level0, dim3(nb2(n)), dim3(kVB2), 0, e->stream, n, M.ptr, M.col,
                       M.val, gi, A.val0.p, A.dinv0.p, valf, dinvf, A.bad.p);
    MA_HIP_TRY(read_back(e, {{&bad, A.bad.p, sizeof(int32_t)}}));
    if (!(bad & 2) || !M.own_col) break;
    MA_HIP_TRY(sort_rows(e, M));
  }
  if (bad & 1) {
    // include/MA/optimal_transport.hpp:48-58 reports zero diagonal entries
    // of the gauge-fixed matrix the same way (its Cholesky cannot proceed)
    e->err = "singular Hessian: a cell other than the gauge cell has no positive diagonal "
             "entry (it shares no edge with another cell)";
    return MA_SINGULAR;
  }
  if (max_levels == 1) {
    A.nlev = 1;
    MA_HIP_TRY(hipGetLastError());
    return MA_OK;
  }
  const ma_status st = A.fp32 ? amg_build<float>(e, A, M) : amg_build<double>(e, A, M);
  if (st != MA_OK) return st;
  MA_HIP_TRY(hipGetLastError());
  return MA_OK;
}

// First level of the tail: the first one below level 0 with at most kTailRows
// rows (the coarsest level at the latest).
template <class T>
static int tail_start(Amg &A) {
  std::vector<AmgLevel<T>> &lv = levels_of(A, (T *)nullptr);
  int l = 1;
  while (l < A.nlev - 1 && lv[l].n > kTailRows) l++;
  return l;
}

// z = M^-1 r (one V-cycle) with the hierarchy in T; level 0 reads r and its
// first sweep (amg_head, written with r), and writes z (FP64).  V(2,2) keeps
// level 0's iterate in z.
template <class T>
static hipError_t amg_cycle(ma_engine *e, Amg &A, const double *r, double *z, double *part,
                            const double *done) {
  std::vector<AmgLevel<T>> &lv = levels_of(A, (T *)nullptr);
  const int nl = A.nlev;
  const double om = e->amg_omega, co = e->amg_corr;  // Jacobi damping, coarse over-correction
  const bool two = e->amg_sweeps != 1;                 // V(2,2), else V(1,1)
  Tail<T> t{};
  t.inv = A.dense_inv.p;
  t.omega = om;
  t.corr = co;
  t.two = two;
  t.nd = (int)lv[nl - 1].n;
  if (nl == 1) {
    hipLaunchKernelGGL((k_amg_tail<T, double, double>), dim3(1), dim3(kTailThreads), 0, e->stream,
                       t, r, (const T *)nullptr, z, part, done);
    return hipGetLastError();
  }
  auto ptr_of = [&](int l) { return l == 0 ? A.ptr0 : lv[l].ptr.p; };
  auto col_of = [&](int l) { return l == 0 ? A.col0 : lv[l].col.p; };
  const T *none = nullptr;
  double *no_part = nullptr;
  const int lt = tail_start<T>(A);
  // downward (the first sweep of a coarse level comes from the restriction)
  for (int l = 0; l < lt; l++) {
    AmgLevel<T> &L = lv[l];
    AmgLevel<T> &Ln = lv[l + 1];
    const bool seed = l + 1 < nl - 1;  // the coarsest level is solved directly
    const T *dc = seed ? Ln.dinv.p : none;
    T *yc = seed ? Ln.y.p : nullptr;
    const unsigned gr = nb2(Ln.n * kAgg * kRowLanes), gs = nb2(L.n * kRowLanes);
    const T *x = L.y.p;
    if (l == 0) {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<false, false, T, double, T, double>), dim3(gs),
                           dim3(kVB2), 0, e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, x, none, z, no_part, done, om, co);
        hipLaunchKernelGGL((k_amg_restrict<T, double, double>), dim3(gr), dim3(kVB2), 0,
                           e->stream, Ln.n, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0), r,
                           (const double *)z, Ln.b.p, dc, yc, done, om);
      } else {  // V(1,1): the one downward sweep is the iterate
        hipLaunchKernelGGL((k_amg_restrict<T, double, T>), dim3(gr), dim3(kVB2), 0, e->stream,
                           Ln.n, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0), r, x, Ln.b.p, dc,
                           yc, done, om);
      }
    } else {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<false, false, T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, x, none, L.x.p, no_part, done, om,
                           co);
        x = L.x.p;
      }
      hipLaunchKernelGGL((k_amg_restrict<T, T, T>), dim3(gr), dim3(kVB2), 0, e->stream, Ln.n,
                         L.n, ptr_of(l), col_of(l), val_of<T>(A, l), (const T *)L.b.p, x,
                         Ln.b.p, dc, yc, done, om);
    }
  }
  for (int l = lt; l < nl - 1; l++)
    t.lv[t.nlev++] = {(int)lv[l].n, ptr_of(l), col_of(l), val_of<T>(A, l), dinv_of<T>(A, l)};
  hipLaunchKernelGGL((k_amg_tail<T, T, T>), dim3(1), dim3(kTailThreads), 0, e->stream, t,
                     (const T *)lv[lt].b.p, (const T *)lv[lt].y.p, lv[lt].x.p, no_part, done);
  // upward
  for (int l = lt - 1; l >= 0; l--) {
    AmgLevel<T> &L = lv[l];
    const T *xc = lv[l + 1].x.p;
    const unsigned gs = nb2(L.n * kRowLanes);
    const dim3 gd(cg_grid(L.n)), bd(kCgThreads);
    if (l == 0) {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<false, true, T, double, double, T>), dim3(gs),
                           dim3(kVB2), 0, e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const double *)z, xc, L.y.p, no_part, done, om,
                           co);
        hipLaunchKernelGGL((k_amg_smooth<true, false, T, double, T, double>), gd, bd, 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const T *)L.y.p, none, z, part, done, om, co);
      } else {
        hipLaunchKernelGGL((k_amg_smooth<true, true, T, double, T, double>), gd, bd, 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const T *)L.y.p, xc, z, part, done, om, co);
      }
    } else {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<false, true, T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, (const T *)L.x.p, xc, L.y.p,
                           no_part, done, om, co);
        hipLaunchKernelGGL((k_amg_smooth<false, false, T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, (const T *)L.y.p, none, L.x.p,
                           no_part, done, om, co);
      } else {
        hipLaunchKernelGGL((k_amg_smooth<false, true, T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, (const T *)L.y.p, xc, L.x.p,
                           no_part, done, om, co);
      }
    }
  }
  return hipGetLastError();
}

AmgHead amg_head(ma_engine *e, Amg &A) {
  AmgHead h;
  h.fp32 = A.fp32;
  h.omega = e->amg_omega;
  h.partials = 1;  // the tail's own sum
  if (A.nlev > 1) {
    h.partials = cg_grid(A.fp32 ? A.lvf[0].n : A.lv[0].n);
    h.dinv = A.fp32 ? (const void *)dinv_of<float>(A, 0) : (const void *)dinv_of<double>(A, 0);
    h.y = A.fp32 ? (void *)A.lvf[0].y.p : (void *)A.lv[0].y.p;
  }
  return h;
}

// z = M^-1 r (one V-cycle) and the partial sums of r.z; done: device flag,
// cycles are skipped once set.
hipError_t amg_apply(ma_engine *e, Amg &A, const double *r, double *z, double *part,
                     const double *done) {
  return A.fp32 ? amg_cycle<float>(e, A, r, z, part, done)
                : amg_cycle<double>(e, A, r, z, part, done);
}

}  // namespace ma
