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
// without a positive diagonal (a cell sharing no edge, or a NaN) sets *bad.
// With outf, also an FP32 copy of the values and inverse diagonal.
__global__ void k_amg_level0(int64_t n, const int32_t *ptr, const int32_t *col,
                             const double *val, int32_t gi, double *out, double *dinv,
                             float *outf, float *dinvf, int32_t *bad) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  double d = 0.0;
  for (int32_t q = ptr[i]; q < ptr[i + 1]; q++) {
    const int32_t j = col[q];
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
// ---------------------------------------------------------------------------
// Sparse row times vector by a group of kRowLanes lanes, FP64 accumulation.
template <class T, class TX>
__device__ inline double row_dot_t(const int32_t *__restrict__ ptr,
                                   const int32_t *__restrict__ col, const T *__restrict__ val,
                                   const TX *__restrict__ x, int64_t i, bool valid, int lane) {
  double s = 0.0;
  if (valid)
    for (int32_t q = ptr[i] + lane; q < ptr[i + 1]; q += kRowLanes)
      s += (double)val[q] * (double)x[col[q]];
  for (int o = 1; o < kRowLanes; o <<= 1) s += __shfl_xor(s, o, kRowLanes);
  return s;
}
// x = omega * b / D   (first sweep from x = 0)
template <class T, class TB>
__global__ void k_amg_smooth0(int64_t n, const T *dinv, const TB *b, T *x, const double *done,
                              double kOmega) {
  if (*done != 0.0) return;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = (T)(kOmega * (double)b[i] * (double)dinv[i]);
}
// y = x + omega (b - A x) / D; rows are read by groups of kRowLanes lanes
// (consecutive entries of consecutive rows: coalesced)
template <class T, class TB, class TX, class TY>
__global__ void k_amg_smooth(int64_t n, const int32_t *ptr, const int32_t *col, const T *val,
                             const T *dinv, const TB *b, const TX *x, TY *y, const double *done,
                             double kOmega) {
  if (*done != 0.0) return;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = t / kRowLanes;
  const int lane = (int)(t % kRowLanes);
  const double ax = row_dot_t(ptr, col, val, x, i, i < n, lane);
  if (i < n && lane == 0)
    y[i] = (TY)((double)x[i] + kOmega * ((double)b[i] - ax) * (double)dinv[i]);
}
// bc[I] = sum over the aggregate of (b - A x): kAgg rows x kRowLanes lanes;
// with dinv_c, also the coarse level's first smoothing sweep from zero,
// yc = omega bc / Dc (saves that level a launch)
template <class T, class TB, class TX>
__global__ void k_amg_restrict(int64_t nc, int64_t n, const int32_t *ptr, const int32_t *col,
                               const T *val, const TB *b, const TX *x, T *bc, const T *dinv_c,
                               T *yc, const double *done, double kOmega) {
  if (*done != 0.0) return;
  constexpr int kGroup = kAgg * kRowLanes;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t I = t / kGroup;
  const int lane = (int)(t % kGroup);
  const int64_t i = I * kAgg + lane / kRowLanes;
  const bool valid = I < nc && i < n;
  const double ax = row_dot_t(ptr, col, val, x, i, valid, lane % kRowLanes);
  double s = (valid && lane % kRowLanes == 0) ? (double)b[i] - ax : 0.0;
  for (int o = kRowLanes; o < kGroup; o <<= 1) s += __shfl_xor(s, o, kGroup);
  if (I < nc && lane == 0) {
    bc[I] = (T)s;
    if (dinv_c) yc[I] = (T)(kOmega * s * (double)dinv_c[I]);
  }
}
// First post-smoothing sweep fused with the prolongation: with
// x' = x + corr * xc[. / kAgg] (the corrected iterate, formed on the fly),
// y = x' + omega (b - A x') / D
template <class T, class TB, class TX, class TY>
__global__ void k_amg_smooth_prolong(int64_t n, const int32_t *ptr, const int32_t *col,
                                     const T *val, const T *dinv, const TB *b, const TX *x,
                                     const T *xc, TY *y, const double *done, double kOmega,
                                     double kCorr) {
  if (*done != 0.0) return;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = t / kRowLanes;
  const int lane = (int)(t % kRowLanes);
  double ax = 0.0;
  if (i < n)
    for (int32_t q = ptr[i] + lane; q < ptr[i + 1]; q += kRowLanes) {
      const int32_t j = col[q];
      ax += (double)val[q] * ((double)x[j] + kCorr * (double)xc[j / kAgg]);
    }
  for (int o = 1; o < kRowLanes; o <<= 1) ax += __shfl_xor(ax, o, kRowLanes);
  if (i < n && lane == 0) {
    const double xi = (double)x[i] + kCorr * (double)xc[i / kAgg];
    y[i] = (TY)(xi + kOmega * ((double)b[i] - ax) * (double)dinv[i]);
  }
}
// coarsest: x = A^-1 b, one workgroup, 16 lanes per row
constexpr int kDenseThreads = 1024;
template <class TB, class TX>
__global__ void __launch_bounds__(kDenseThreads) k_amg_dense_solve(int64_t n, const double *inv,
                                                                   const TB *b, TX *x,
                                                                   const double *done) {
  if (*done != 0.0) return;
  __shared__ double sb[kCoarsest];
  for (int i = threadIdx.x; i < n; i += kDenseThreads) sb[i] = (double)b[i];
  __syncthreads();
  // a group's rows together, so that their loads overlap
  constexpr int kRows = kCoarsest / (kDenseThreads / kGroup);
  const int l = (int)threadIdx.x & (kGroup - 1), i0 = (int)threadIdx.x / kGroup;
  const int N = (int)n;
  const double *row[kRows];
  double s[kRows];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    row[r] = inv + min(i0 + r * (kDenseThreads / kGroup), N - 1) * N;
    s[r] = 0.0;
  }
#pragma unroll 4
  for (int k = l; k < N; k += kGroup)
#pragma unroll
    for (int r = 0; r < kRows; r++) s[r] += row[r][k] * sb[k];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    const double t = row_sum(s[r]);
    const int i = i0 + r * (kDenseThreads / kGroup);
    if (l == 0 && i < N) x[i] = (TX)t;
  }
}
static_assert(kCoarsest % (kDenseThreads / kGroup) == 0, "rows of k_amg_dense_solve");

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
  MA_HIP_TRY(lv[0].x.ensure((size_t)n));
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
    const int32_t zero = 0;
    MA_HIP_TRY(hipMemcpyAsync(C.ptr.p + nc, &zero, sizeof(int32_t), hipMemcpyHostToDevice,
                              e->stream));
    MA_HIP_TRY(exclusive_scan(e, C.ptr.p, C.ptr.p, nc + 1));
    // small levels take room for as many entries as the level above has,
    // instead of waiting for their count
    if (!wave) {
      int32_t nnzc = 0;
      MA_HIP_TRY(hipMemcpyAsync(&nnzc, C.ptr.p + nc, sizeof(int32_t), hipMemcpyDeviceToHost,
                                e->stream));
      MA_HIP_TRY(hipStreamSynchronize(e->stream));
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
  MA_HIP_TRY(hipMemsetAsync(A.bad.p, 0, sizeof(int32_t), e->stream));
  hipLaunchKernelGGL(k_amg_level0, dim3(nb2(n)), dim3(kVB2), 0, e->stream, n, M.ptr, M.col,
                     M.val, gi, A.val0.p, A.dinv0.p, valf, dinvf, A.bad.p);
  int32_t bad = 0;
  MA_HIP_TRY(hipMemcpyAsync(&bad, A.bad.p, sizeof(int32_t), hipMemcpyDeviceToHost, e->stream));
  MA_HIP_TRY(hipStreamSynchronize(e->stream));
  if (bad) {
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

// z = M^-1 r (one V-cycle) with the hierarchy in T; level 0 reads r and
// keeps its iterate in z (FP64), its smoother output in lv[0].y (T).
template <class T>
static hipError_t amg_cycle(ma_engine *e, Amg &A, const double *r, double *z, const double *done) {
  std::vector<AmgLevel<T>> &lv = levels_of(A, (T *)nullptr);
  const int nl = A.nlev;
  const double om = e->amg_omega, co = e->amg_corr;  // Jacobi damping, coarse over-correction
  const bool two = e->amg_sweeps != 1;                 // V(2,2), else V(1,1)
  auto ptr_of = [&](int l) { return l == 0 ? A.ptr0 : lv[l].ptr.p; };
  auto col_of = [&](int l) { return l == 0 ? A.col0 : lv[l].col.p; };
  if (nl == 1) {
    hipLaunchKernelGGL((k_amg_dense_solve<double, double>), dim3(1), dim3(kDenseThreads), 0,
                       e->stream, lv[0].n, A.dense_inv.p, r, z, done);
    return hipGetLastError();
  }
  // downward (the first sweep of a coarse level comes from the restriction)
  for (int l = 0; l < nl - 1; l++) {
    AmgLevel<T> &L = lv[l];
    AmgLevel<T> &Ln = lv[l + 1];
    const bool seed = l + 1 < nl - 1;  // the coarsest level is solved directly
    const T *dc = seed ? Ln.dinv.p : (const T *)nullptr;
    T *yc = seed ? Ln.y.p : nullptr;
    const unsigned gr = nb2(Ln.n * kAgg * kRowLanes), gs = nb2(L.n * kRowLanes);
    if (l == 0) {
      hipLaunchKernelGGL((k_amg_smooth0<T, double>), dim3(nb2(L.n)), dim3(kVB2), 0, e->stream,
                         L.n, dinv_of<T>(A, 0), r, L.y.p, done, om);
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<T, double, T, double>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const T *)L.y.p, z, done, om);
        hipLaunchKernelGGL((k_amg_restrict<T, double, double>), dim3(gr), dim3(kVB2), 0,
                           e->stream, Ln.n, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0), r,
                           (const double *)z, Ln.b.p, dc, yc, done, om);
      } else {  // V(1,1): the one downward sweep is the iterate
        hipLaunchKernelGGL((k_amg_restrict<T, double, T>), dim3(gr), dim3(kVB2), 0, e->stream,
                           Ln.n, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0), r,
                           (const T *)L.y.p, Ln.b.p, dc, yc, done, om);
      }
    } else {
      const T *x = L.y.p;
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth<T, T, T, T>), dim3(gs), dim3(kVB2), 0, e->stream, L.n,
                           ptr_of(l), col_of(l), val_of<T>(A, l), dinv_of<T>(A, l),
                           (const T *)L.b.p, (const T *)L.y.p, L.x.p, done, om);
        x = L.x.p;
      }
      hipLaunchKernelGGL((k_amg_restrict<T, T, T>), dim3(gr), dim3(kVB2), 0, e->stream, Ln.n,
                         L.n, ptr_of(l), col_of(l), val_of<T>(A, l), (const T *)L.b.p, x,
                         Ln.b.p, dc, yc, done, om);
    }
  }
  {
    AmgLevel<T> &Lc = lv[nl - 1];
    hipLaunchKernelGGL((k_amg_dense_solve<T, T>), dim3(1), dim3(kDenseThreads), 0, e->stream,
                       Lc.n, A.dense_inv.p, (const T *)Lc.b.p, Lc.x.p, done);
  }
  // upward
  for (int l = nl - 2; l >= 0; l--) {
    AmgLevel<T> &L = lv[l];
    const T *xc = lv[l + 1].x.p;
    const unsigned gs = nb2(L.n * kRowLanes);
    if (l == 0) {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth_prolong<T, double, double, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const double *)z, xc, L.y.p, done, om, co);
        hipLaunchKernelGGL((k_amg_smooth<T, double, T, double>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const T *)L.y.p, z, done, om);
      } else {
        hipLaunchKernelGGL((k_amg_smooth_prolong<T, double, T, double>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(0), col_of(0), val_of<T>(A, 0),
                           dinv_of<T>(A, 0), r, (const T *)L.y.p, xc, z, done, om, co);
      }
    } else {
      if (two) {
        hipLaunchKernelGGL((k_amg_smooth_prolong<T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, (const T *)L.x.p, xc, L.y.p,
                           done, om, co);
        hipLaunchKernelGGL((k_amg_smooth<T, T, T, T>), dim3(gs), dim3(kVB2), 0, e->stream, L.n,
                           ptr_of(l), col_of(l), val_of<T>(A, l), dinv_of<T>(A, l),
                           (const T *)L.b.p, (const T *)L.y.p, L.x.p, done, om);
      } else {
        hipLaunchKernelGGL((k_amg_smooth_prolong<T, T, T, T>), dim3(gs), dim3(kVB2), 0,
                           e->stream, L.n, ptr_of(l), col_of(l), val_of<T>(A, l),
                           dinv_of<T>(A, l), (const T *)L.b.p, (const T *)L.y.p, xc, L.x.p,
                           done, om, co);
      }
    }
  }
  return hipGetLastError();
}

// z = M^-1 r (one V-cycle); done: device flag, cycles are skipped once set.
hipError_t amg_apply(ma_engine *e, Amg &A, const double *r, double *z, const double *done) {
  return A.fp32 ? amg_cycle<float>(e, A, r, z, done) : amg_cycle<double>(e, A, r, z, done);
}

}  // namespace ma
