// Internal declarations shared by the engine's HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <initializer_list>
#include <string>
#include <vector>

#include "../../include/ma/ma.h"

namespace ma {

struct Amg;  // multigrid hierarchy (amg.hip)

// ---------------------------------------------------------------------------
// Device buffer (owned, grows on demand, never shrinks until destroyed).
// ---------------------------------------------------------------------------
template <class T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  DBuf(DBuf &&o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  ~DBuf() { release(); }
  hipError_t ensure(size_t count) {
    if (count <= n) return hipSuccess;
    if (p) {
      hipError_t e = hipFree(p);
      p = nullptr;
      n = 0;
      if (e != hipSuccess) return e;
    }
    size_t c = count > 0 ? count : 1;
    hipError_t e = hipMalloc(reinterpret_cast<void **>(&p), c * sizeof(T));
    if (e == hipSuccess) n = c;
    return e;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  // exchanges the allocations (pointer and capacity together)
  void swap(DBuf &o) noexcept {
    T *tp = p;
    p = o.p;
    o.p = tp;
    size_t tn = n;
    n = o.n;
    o.n = tn;
  }
};

// Uniform square grid of 2^L x 2^L bins over a square region; bins are indexed
// by the Morton (Z-order) code of their integer coordinates.
struct Grid {
  double x0, y0;  // lower-left corner
  double h;       // bin side
  int L;          // levels: G = 2^L bins per side
  int G;
  int64_t nbins;  // G * G
};

// Per-triangle data, counter-clockwise vertices, density a x + b y + c.
struct TriData {
  double x[3], y[3];
  double a, b, c;
};

// Capacity of the general kernel's per-thread polygons, and of the staging
// of one Hessian row (neighbours + diagonal).
constexpr int kMaxPoly = 64;
constexpr int kMaxRow = 65;
// Capacity of the one-workgroup-per-cell kernel for larger cells (polygon in
// LDS), its workgroup size and the staging of one of its rows.
constexpr int kHugePoly = 1024;
constexpr int kHugeBlock = 256;
constexpr int kHugeRow = kHugePoly + 1;
// Cells whose bin rectangle spans more bins than this skip the one-thread-
// per-cell kernels (their candidate loops are sequential) for the
// one-workgroup-per-cell kernel.
constexpr int kBigRect = 64;
// Up to this many cells left by the fast path go straight to the
// one-workgroup-per-cell kernel.
constexpr int kHugeRoute = 32768;
constexpr int kLongRows = 1024;  // pool of staged rows longer than kMaxRow
// Site-centric cell search: rings of bins visited before the pyramid walk,
// and pyramid nodes a cell may visit before it is left to the bin path
// (defaults; MA_OPT_LOCAL_RINGS / MA_OPT_WALK_BUDGET).
constexpr int kLocalRings = 8;
constexpr int kWalkBudget = 1024;
// Candidate triangles per cell kept by the cell kernels for the pair list
// (cells with more are scanned again).
constexpr int kPadTri = 24;
// Polygon capacity of the register/LDS fast path (vertices per cell).
constexpr int kMaxFast = 16;
constexpr int kMaxLevels = 12;  // levels of the bin grid above the bins

// Event counts that every workgroup adds to are striped over 16 cache lines
// (one address takes an atomic every 8 ns or so): stripe `b` mod 16 of count
// `which` (0: fragments, 1: vertices) behind the plain counters.
constexpr int kPlainCounters = 16, kCounterStripes = 16;
constexpr int kCounters = kPlainCounters + 2 * kCounterStripes * 16;
__host__ __device__ inline unsigned long long *counter_stripe(unsigned long long *counters,
                                                              int which, unsigned b) {
  return counters + kPlainCounters + (which * kCounterStripes + (b % kCounterStripes)) * 16;
}

// Fragment polygons written out by the first-moment kernels while `count` is
// set (ma_fragments).  Each fragment of positive area reserves one record and
// its vertices; nothing is written past the capacities, but the counts keep
// advancing, so a pass that ran out learns the sizes it needs.
struct FragOut {
  unsigned long long *count = nullptr;  // [0] fragments, [1] vertices
  int32_t *cell = nullptr;  // caller index of the Dirac
  int32_t *tri = nullptr;   // triangle index (engine order, see ma_engine::tperm)
  int32_t *nv = nullptr;    // vertex count
  int64_t *start = nullptr; // first vertex
  double *xy = nullptr;     // absolute coordinates, interleaved, counter-clockwise
  int64_t cap_frag = 0, cap_vert = 0;
};

// Buffers of the output entry points (fragment polygons, rasterisation).
struct OutBuffers {
  DBuf<unsigned long long> fcount;
  DBuf<int32_t> fcell, ftri, fnv;
  DBuf<int64_t> fstart;
  DBuf<double> fxy;
  DBuf<uint64_t> key, key2;   // radix sort by (Dirac, triangle)
  DBuf<int32_t> idx, idx2;
  DBuf<unsigned char> sort_tmp;
  DBuf<int64_t> scnt, sstart; // vertex counts and offsets in sorted order
  DBuf<double> sxy;           // sorted vertices
  DBuf<int32_t> scell, stri;
  DBuf<double> colors, img;   // rasterisation
  DBuf<double> pix;           // image pixels (mesh from an image)
  DBuf<int64_t> vbeg, vend;   // per Dirac: its fragments' vertices in sorted order
  DBuf<int64_t> hcnt, hoff;   // per Dirac: cell polygon vertex count and offset
  DBuf<double> hxy;           // cell polygons
};

struct EvalBuffers {
  DBuf<double> w_s;          // weights in Morton order
  // low words of two-word weights (w = w_s + wlo_s) for the evaluation in
  // progress when use_wlo is set; plain FP64 weights otherwise
  DBuf<double> wlo_s;
  bool use_wlo = false;
  const double *wlo() const { return use_wlo ? wlo_s.p : nullptr; }
  DBuf<double> pyr;          // max-weight pyramid (all levels)
  DBuf<double> pyr3;         // per level: max over the 3 x 3 neighbouring nodes
  DBuf<int32_t> cand_cnt;    // CSR offsets of the per-bin candidate lists (nbins + 1)
  DBuf<int32_t> cand;        // candidate owners, bin after bin
  DBuf<int32_t> cbin;        // bin of each candidate entry (before refinement)
  DBuf<int32_t> ckeep;       // keep flags of the entries, then their prefix sums
  DBuf<int32_t> cand2, cstart2;  // refined lists (swapped with cand / cand_cnt)
  DBuf<double> plane;        // plane pyramid (4 per node) and its sums
  DBuf<double> node_sums;
  DBuf<int32_t> owner;       // per bin, best competitor of the last evaluation
  DBuf<int32_t> rect;        // per Dirac: bin rectangle (x0, y0, x1, y1)
  DBuf<double> mass_s, intg_s, fval_part;
  DBuf<double> mom_s;        // first moments (2 per Dirac)
  DBuf<double> mom2_s;       // second moments (3 per Dirac, mode 3)
  DBuf<double> dval;         // adjoint w.r.t. vertex density values (nv)
  DBuf<int32_t> row_cnt;     // per Dirac, entries incl. diagonal
  DBuf<int32_t> row_col;     // n x cap_row (rows of the general kernels)
  DBuf<double> row_val;      // n x cap_row
  DBuf<int32_t> csr_ptr, csr_col;   // Morton-order CSR
  DBuf<double> csr_val;
  DBuf<int32_t> flags;       // [0] overflow poly,
                             // [3] cells for the general kernels
  DBuf<unsigned long long> counters;  // [0] fragments, [1] candidates, [2] max poly, [3] empty,
                                      // [4] vertices, [5] FP64 re-decisions, [6] bin-path cells,
                                      // [7] failing cell (k_cell_huge), [8] long rows;
                                      // more fragments and vertices in the stripes
                                      // (counter_stripe)
  // per-wave event counts of the cell kernel, striped over 16 cache lines
  // (kStripes counters of 16 words each) so that no single address takes
  // an atomic from every wave: [0..15] cells that walked the pyramid,
  // [16..31] cells left to the bin path, [32..47] cells left to the general
  // kernels (word 0 of each line used)
  DBuf<unsigned long long> stripes;
  DBuf<int32_t> scan_tmp;
  DBuf<double> red_tmp;
  // register/LDS fast path
  DBuf<double> px, py, eacc, bbox;
  DBuf<float> pxf, pyf;          // FP32 polygons (mixed mode)
  DBuf<int32_t> plab, pn, tcount, poff, pair_cell, pair_tri, glist;
  DBuf<int32_t> cstage;  // the first candidates of every bin, kept by the counting walk
  DBuf<int32_t> ptri;         // kPadTri candidate triangles per cell, [k * kPadTri + c]
  DBuf<int32_t> ovf;          // pairs for k_frag_wide (+ count)
  // cells beyond the general kernel (list + count at [n]) and their long rows
  DBuf<int32_t> hlist, hrow_col;
  DBuf<double> hrow_val;
  DBuf<unsigned char> far;    // per Dirac: its cell took the bin path last time (FP64)
  DBuf<unsigned char> binmask;  // bins whose candidate owners are built (few cells left over)
};

// What the calls that copy Diracs in and results out work in.
struct CopyBuffers {
  DBuf<double> xy;            // positions (2 n) in the caller's layout, column (n) or results
  DBuf<double> xi;            // positions, interleaved
  DBuf<int32_t> bin, cnt;     // bin of a Dirac; entries per bin
  DBuf<int32_t> ptr, col;     // the Hessian in the caller's order
  DBuf<double> val;
};

struct SolverBuffers {
  DBuf<double> w, m, nu, g, d, x, r, z, p, q, Ap, wtrial, red;
  DBuf<double> stage;         // host <-> device staging of per-Dirac arrays
  DBuf<int32_t> hptr, hcol;   // caller-supplied CSR (ma_solve_laplacian_csr)
  DBuf<double> hval, hg, hd;
  DBuf<int32_t> moved;        // set when a trial point differs from the iterate
  DBuf<int32_t> cc;           // component labels of the Hessian's graph
  DBuf<double> wl, wtl;       // low words of the iterate and trial point (two-word weights)
};

// Sets EvalBuffers::use_wlo for the evaluations of one entry point and
// clears it on every way out, so that no other entry point sees low words.
struct WloScope {
  EvalBuffers &B;
  WloScope(EvalBuffers &b, bool on) : B(b) { B.use_wlo = on; }
  ~WloScope() { B.use_wlo = false; }
  WloScope(const WloScope &) = delete;
  WloScope &operator=(const WloScope &) = delete;
};

}  // namespace ma

struct ma_engine {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev[12] = {};  // [10], [11]: around the site-centric cell kernel
  std::string err;

  // mesh
  int64_t nv = 0, nt = 0;
  double dom[4] = {0, 0, 0, 0};  // domain bounding box
  // triangles in Morton order of their centroids (tperm: that order -> the
  // caller's triangle index), so that the triangles a wave of pairs reads
  // share cache lines
  ma::DBuf<ma::TriData> tri;
  ma::DBuf<int32_t> triv;  // ccw vertex ids (nt x 3)
  ma::DBuf<float4> tbox;   // FP32 bounding boxes, rounded outwards
  ma::DBuf<int32_t> tperm;
  ma::DBuf<double> vxy, vval;
  bool have_mesh = false;

  // Diracs and grid
  int64_t n = 0;
  bool have_diracs = false;
  ma::Grid grid{};
  ma::DBuf<double> pos;        // Morton-ordered positions (2 n)
  ma::DBuf<int32_t> perm;      // Morton slot -> caller index
  ma::DBuf<int32_t> iperm;     // caller index -> Morton slot
  ma::DBuf<int32_t> bin_start; // Diracs of bin b: [bin_start[b], bin_start[b+1])
  ma::DBuf<int32_t> tbin_start, tbin_items;
  bool grid_valid = false;     // triangle bins built for the current grid

  ma::Amg *amg = nullptr;
  int cap_cand = 48;
  int force_general = 0;  // MA_OPT_FORCE_GENERAL
  int use_graphs = 1;     // MA_OPT_GRAPHS: replay CG batches from a HIP graph
  int local_rings = ma::kLocalRings;  // MA_OPT_LOCAL_RINGS
  int walk_budget = ma::kWalkBudget;  // MA_OPT_WALK_BUDGET
  double amg_omega = 0.85;  // MA_OPT_AMG_OMEGA: Jacobi damping of the multigrid smoother
  double amg_corr = 1.5;         // MA_OPT_AMG_CORR: coarse-correction scaling
  int amg_sweeps = 1;            // MA_OPT_AMG_SWEEPS: smoothing sweeps each way (1 or 2)
  int far_cells = 1;             // MA_OPT_FAR_CELLS
  bool ran_candidates = false;  // the last evaluation built per-bin candidate lists
  int cap_row = ma::kMaxRow;

  ma::EvalBuffers eb;
  ma::CopyBuffers cb;
  uint32_t *pinned = nullptr;  // kReadBytes of host memory (read_back)
  ma::SolverBuffers sb;
  ma::OutBuffers ob;
  ma::FragOut fo;  // set only while ma_fragments / ma_draw_laguerre run
  ma_eval_info info{};
  // have_eval: the last evaluation (any mode) succeeded, so per-cell outputs
  // (vertex counts, masses) describe the current mesh, Diracs and weights;
  // have_hessian: it was a Kantorovich evaluation, so the CSR Hessian and
  // the per-cell costs are current.  Both are cleared when an evaluation
  // starts and when the mesh or the Diracs change.
  bool have_eval = false;
  bool have_hessian = false;
  // per-bin owners hold -1 or a Dirac of the current grid (warm start of the
  // candidate search)
  bool owner_init = false;
  // eb.far describes the current Diracs (set by an FP64 evaluation, cleared
  // when the Diracs change)
  bool far_valid = false;
  // candidate lists: built only around the few left-over cells until such an
  // attempt falls through (reset with the Diracs); refined to exact owners
  // when many cells take the bin path (set per evaluation)
  bool mask_ok = true;
  bool refine = true;
  bool many_far = false;  // the last FP64 evaluation sent >= n/16 cells to the bin path
  int64_t nnz = 0;

  // host scratch
  std::vector<int64_t> pyr_off;
};

namespace ma {

// Checks that mesh and Diracs are set and builds the triangle bins if needed
// (engine.hip).
ma_status need(ma_engine *e);
// Marks the mesh (and everything computed from it) unusable; called before
// any mesh buffer is overwritten.
void invalidate_mesh(ma_engine *e);
// Completes a mesh whose vertices (e->vxy, e->vval) are on the device: triangle
// records and bounding boxes from the device triangle list d_tri (nt x 3),
// domain box `box` (x0, y0, x1, y1).
ma_status finish_mesh(ma_engine *e, int64_t nv, int64_t nt, const int32_t *d_tri,
                      const double box[4]);

// Reorders e->tri / triv / tbox (caller order on entry) by the Morton code of
// the triangle centroids and sets e->tperm (output.hip).
ma_status sort_triangles(ma_engine *e, int64_t nt);

// Geometry (geometry.hip)
hipError_t build_dirac_grid(ma_engine *e, const double *d_X, int layout);
hipError_t build_triangle_bins(ma_engine *e);
// Evaluates masses / value / Hessian (CSR in Morton order) at Morton-ordered
// weights e->eb.w_s.  mode 0: Kantorovich, mode 1: first moments, mode 2:
// first moments and the density-value adjoint (into eb.dval, which the caller
// zeroes).  fp32: FP32 cell geometry and quadrature (mixed precision, mode 0).
ma_status evaluate(ma_engine *e, int mode, double *fval_out, bool fp32 = false);
// Copy helpers between caller order and Morton order.
hipError_t to_morton(ma_engine *e, const double *src_caller, double *dst_morton, bool src_on_device);
hipError_t from_morton(ma_engine *e, const double *src_morton, double *dst_caller, bool dst_on_device);
// out[i] = in[0] + ... + in[i - 1] for i = 0 .. n (out may be in).
hipError_t exclusive_scan(ma_engine *e, const int32_t *in, int32_t *out, int64_t n);
hipError_t csr_to_caller(ma_engine *e, int32_t *rowptr, int32_t *col, double *val);
ma_status adjoint(ma_engine *e, double *dY_caller, double *dval);
// Words of device memory to the host, up to kReadBytes together: one kernel
// writes them into the engine's pinned page and the stream is waited for.  (A
// copy into pageable memory takes a launch, a wait and a host copy each, about
// 10 us; an evaluation of N = 1000 reads eleven such values.)
struct ReadPart {
  void *dst;
  const void *src;
  size_t bytes;  // a multiple of 4
};
constexpr int kReadParts = 4;
constexpr size_t kReadBytes = 32768;
hipError_t read_back(ma_engine *e, std::initializer_list<ReadPart> parts);

// A square CSR matrix on the device.
struct CsrView {
  int64_t n = 0, nnz = 0;
  const int32_t *ptr = nullptr, *col = nullptr;
  const double *val = nullptr;
  // col and val once more where amg_setup may bring the rows into column order
  int32_t *own_col = nullptr;
  double *own_val = nullptr;
};
// Multigrid preconditioner (amg.hip)
Amg *amg_create();
void amg_destroy(Amg *a);
// Returns MA_SINGULAR when a row other than gi has a non-positive diagonal.
ma_status amg_setup(ma_engine *e, Amg &A, const CsrView &M, int32_t gi, int max_levels,
                    bool fp32);
// What the conjugate gradient does for the cycle where it writes r: level 0's
// first sweep y = omega r / D (in the hierarchy's precision; y = null: the
// cycle has none).  partials: partial sums of r.z that amg_apply leaves.
struct AmgHead {
  bool fp32 = false;
  const void *dinv = nullptr;
  void *y = nullptr;
  double omega = 1.0;
  int partials = 0;
};
AmgHead amg_head(ma_engine *e, Amg &A);
hipError_t amg_apply(ma_engine *e, Amg &A, const double *r, double *z, double *part,
                     const double *done);
const double *amg_level0_values(const Amg &a);
const double *amg_level0_dinv(const Amg &a);

}  // namespace ma

#define MA_HIP_TRY(expr)                                                   \
  do {                                                                     \
    hipError_t _e = (expr);                                                \
    if (_e != hipSuccess) {                                                \
      e->err = std::string(#expr) + ": " + hipGetErrorString(_e);          \
      return _e == hipErrorOutOfMemory ? MA_OUT_OF_MEMORY : MA_HIP_ERROR;  \
    }                                                                      \
  } while (0)

#define MA_HIP_RET(expr)               \
  do {                                 \
    hipError_t _e = (expr);            \
    if (_e != hipSuccess) return _e;   \
  } while (0)
