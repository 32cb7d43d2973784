/*
 * ma.h -- C ABI of the MI355X (gfx950) semi-discrete optimal transport engine.
 *
 * This is the drop-in boundary for the hot path of MongeAmpere++
 * (power diagram x triangulation -> Kantorovich value / masses / Hessian ->
 * damped Newton).  No templates, no CGAL/Eigen types: plain pointers and sizes.
 *
 * Conventions shared with the reference:
 *   - power distance pi_i(x) = |x - y_i|^2 - w_i; a point tied between two
 *     Diracs belongs to neither (include/MA/predicates.hpp:85-86);
 *   - the density is P1 on a triangulation (values at vertices; per face a
 *     linear function, include/MA/functions.hpp:55-80);
 *   - Hessian entries H_ij = -int_{edge ij} rho ds / (2 |y_i - y_j|),
 *     H_ii = -sum_j H_ij (include/MA/kantorovich.hpp:109-122).
 *
 * All arrays are in the caller's Dirac order (index i = row i of X).
 * One engine = one device + one HIP stream; calls on one engine must not
 * overlap; distinct engines are independent.
 */
#ifndef MA_H
#define MA_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ma_engine ma_engine;

typedef enum {
  MA_OK = 0,
  MA_BAD_INPUT = 1,       /* wrong sizes, NaNs, non-triangles ...            */
  MA_EMPTY_CELL = 2,      /* a Laguerre cell is empty (ma_stats.bad_index)    */
  MA_SINGULAR = 3,        /* zero Hessian diagonal (a cell sharing no edge),
                             or the conjugate gradient met p.Ap <= 0        */
  MA_NOT_CONVERGED = 4,   /* Newton reached maxiter                           */
  MA_LINESEARCH_FAIL = 5, /* step length fell below alpha_min                 */
  MA_OUT_OF_MEMORY = 6,
  MA_HIP_ERROR = 7,
  MA_CAPACITY = 8,        /* a fixed-size per-cell buffer overflowed          */
  MA_NO_DATA = 9,         /* mesh or Diracs not set yet, or no (successful)
                             evaluation to read a Hessian from              */
  MA_LINEAR_FAIL = 10     /* the sparse linear solve stopped at its iteration
                             cap above its residual tolerance               */
} ma_status;

typedef enum { MA_FP64 = 0, MA_MIXED = 1 } ma_precision;
typedef enum { MA_XY_INTERLEAVED = 0, MA_XY_COLMAJOR = 1 } ma_layout;
typedef enum { MA_STOP_L2 = 0, MA_STOP_MAXREL = 1 } ma_stop_rule;

typedef struct {
  int precision;      /* ma_precision                                         */
  int stop_rule;      /* MA_STOP_L2: ||m - nu||_2 < eps_g (reference rule,
                         include/MA/optimal_transport.hpp:150);
                         MA_STOP_MAXREL: max_i |m_i - nu_i| / nu_i <= tol     */
  double eps_g;       /* default 1e-7                                          */
  double tol;         /* max-relative tolerance for MA_STOP_MAXREL            */
  int maxiter;        /* default 100; like the reference, up to maxiter + 1
                         Newton steps run (optimal_transport.hpp:151)         */
  double alpha_min;   /* backtracking floor (default 2^-30)                   */
  double cg_tol;      /* relative residual of the linear solves (0 = auto)   */
  int cg_maxiter;     /* default 20000                                        */
  int verbose;        /* print one line per Newton step to stderr             */
  int preconditioner; /* 0: aggregation multigrid (default), 1: Jacobi        */
} ma_solve_opts;

typedef struct {
  int64_t niter;        /* Newton steps  (reference Statistics::niter)        */
  int64_t neval;        /* Kantorovich evaluations (Statistics::neval)        */
  int64_t cg_iter;      /* total linear-solver iterations                     */
  int64_t bad_index;    /* Dirac index for MA_EMPTY_CELL                      */
  double max_rel_err;   /* final max_i |m_i - nu_i| / nu_i (FP64)             */
  double l2_err;        /* final ||m - nu||_2                                 */
  double fval;          /* final value of F(w) = fval(w) - <nu, w>            */
  double ms_total;      /* wall time of the solve                             */
  double ms_eval;       /* time in evaluations                                */
  double ms_linear;     /* time in linear solves                              */
  int64_t neval_fp32;   /* evaluations with FP32 geometry (mixed precision)   */
} ma_stats;

/* Per-phase timing (ms, HIP events on the engine's stream) and counters of
 * the last evaluation. */
typedef struct {
  double ms_total, ms_weights, ms_candidates, ms_cells, ms_assemble;
                        /* ms_candidates: per-bin candidate lists, built only
                           for cells that overflow the fast path            */
  double ms_cell_build, ms_pairs, ms_frag; /* parts of ms_cells             */
  int64_t nnz;          /* Hessian nonzeros (incl. diagonal)                  */
  int64_t nfrag;        /* non-empty (cell, triangle) fragments              */
  int64_t ncand;        /* sum over bins of candidate owners                  */
  int64_t max_poly;     /* largest cell polygon seen                          */
  int64_t empty_cells;  /* Diracs with zero mass                              */
  int64_t npairs;       /* (cell, triangle) pairs clipped                     */
  int64_t ngeneral;     /* cells evaluated by the general (overflow) kernel   */
  int64_t nbinpath;     /* cells not certified by the ring search, finished
                           by the max-weight pyramid walk                     */
  int64_t nvert;        /* sum of fast-path cell polygon vertex counts        */
  int64_t nredecide;    /* mixed mode: FP32 clip tests re-decided in FP64     */
  int64_t nbincand;     /* cells rebuilt from per-bin candidate owners (walk
                           over budget)                                       */
  int64_t nhuge;        /* cells beyond the general kernel's 60 vertices,
                           evaluated one workgroup per cell                   */
  double ms_cell_kernel; /* the site-centric cell kernel alone (inside
                           ms_cell_build)                                     */
} ma_eval_info;

ma_status ma_create(int device, ma_engine **out);
void ma_destroy(ma_engine *e);
const char *ma_last_error(const ma_engine *e);

/* Triangulated domain with P1 density values at the vertices.  Replaces the
 * (T, Functions) pair of include/MA/kantorovich.hpp:37-38.  Triangles may be
 * given in either orientation.  Data are copied. */
ma_status ma_set_mesh(ma_engine *e, int64_t nv, const double *vxy, const double *vval,
                      int64_t nt, const int32_t *tri);

/* Dirac positions X (n x 2), replaces `const Matrix &X`
 * (include/MA/kantorovich.hpp:39).  layout MA_XY_COLMAJOR matches Eigen's
 * MatrixXd storage (all x, then all y).  Data are copied. */
ma_status ma_set_diracs(ma_engine *e, int64_t n, const double *X, int layout);

/* One evaluation of the Kantorovich functional at weights w (host array, n).
 * Replaces MA::kantorovich (include/MA/kantorovich.hpp:35-141): *fval gets the
 * value, g (host, n, may be NULL) the cell masses, *nnz the number of stored
 * Hessian entries.  The Hessian stays on the device until ma_hessian_copy. */
ma_status ma_kantorovich(ma_engine *e, const double *w, int precision, double *fval,
                         double *g, int64_t *nnz);

/* Same with device-resident weights and masses (d_g may be NULL).  The
 * engine reads d_w on its own stream with no ordering against the stream
 * that wrote it: the caller makes sure d_w is complete before the call
 * (e.g. synchronises its stream).  d_g is complete when the call returns. */
ma_status ma_kantorovich_device(ma_engine *e, const double *d_w, int precision,
                                double *fval, double *d_g, int64_t *nnz);

/* Copies the last Hessian as CSR in the caller's Dirac order (rowptr n+1,
 * col/val nnz; columns sorted; duplicates summed like setFromTriplets,
 * include/MA/kantorovich.hpp:137-139). */
ma_status ma_hessian_copy(ma_engine *e, int32_t *rowptr, int32_t *col, double *val);

/* Per-cell transport cost of the last Kantorovich evaluation (caller order,
 * n entries): cost[i] = int_{Lag_i} rho(x) |x - y_i|^2 dx, the integrals
 * include/MA/kantorovich.hpp:124-131 sums into its value, which is
 * fval = sum_i (w_i m_i - cost[i]).  At the optimal weights the sum of the
 * costs is W2^2; formed cell by cell, a difference of two such sums keeps
 * the precision of the cells instead of that of the totals.  MA_NO_DATA if
 * the last evaluation failed or was not a Kantorovich evaluation. */
ma_status ma_cell_costs(ma_engine *e, double *cost);

/* Damped Newton solve; replaces MA::ot_solve
 * (include/MA/optimal_transport.hpp:89-193).  nu: target masses (n);
 * w: in = initial guess (used when init_w != 0, otherwise zeros),
 *    out = weights.  opts may be NULL (defaults). */
ma_status ma_ot_solve(ma_engine *e, const double *nu, double *w, int init_w,
                      const ma_solve_opts *opts, ma_stats *stats);

/* Two-word weights: the weights are w + w_lo (host arrays, n each; the pair
 * is renormalised so that |w_lo| <= ulp(w) / 2), and every bisector offset
 * w_k - w_j is formed from both words.  No counterpart in the reference,
 * whose weights are FP64: it serves callers whose targets are finer than
 * what FP64 weights can resolve.  Two Diracs 2e-6 apart exchange ~250 units
 * of mass per unit of weight difference, so one ulp of a weight near 0.07
 * moves 3.5e-15 of mass, which caps the max relative mass error near 1e-9 at
 * 200k cells; with the low word that cap is ~1e-25.
 * ma_kantorovich_x: ma_kantorovich at w + w_lo (w_lo NULL: exactly
 * ma_kantorovich).
 * ma_ot_solve_x: ma_ot_solve carrying the iterate in two words; w_lo is
 * in (with init_w) and out like w.  w alone (the high words) is the
 * solution rounded to FP64, whose own error is back at the FP64 cap. */
ma_status ma_kantorovich_x(ma_engine *e, const double *w, const double *w_lo, int precision,
                           double *fval, double *g, int64_t *nnz);
ma_status ma_ot_solve_x(ma_engine *e, const double *nu, double *w, double *w_lo, int init_w,
                        const ma_solve_opts *opts, ma_stats *stats);

/* Gauge-fixed Newton direction: solves H[:n-1,:n-1] d = g[:n-1], d[n-1] = 0
 * for the Hessian of the last evaluation.  Replaces solve_laplacian_matrix
 * (include/MA/optimal_transport.hpp:41-87).  *res gets ||H d - g|| over the
 * first n-1 rows, relative to ||g||. */
ma_status ma_solve_laplacian(ma_engine *e, const double *g, double *d, double rel_tol,
                             int maxiter, double *res, int64_t *iters);

/* Same gauge-fixed solve for a caller-supplied symmetric CSR matrix (n x n,
 * 0-based rowptr/col, the columns of a row in any order; e.g. a Hessian copied
 * out earlier or assembled by the caller), the solve_laplacian_matrix(h, g) call shape of
 * include/MA/optimal_transport.hpp:41-44.  Needs no mesh or Diracs.  The
 * multigrid aggregates follow the index order, so a spatially coherent
 * numbering converges fastest. */
ma_status ma_solve_laplacian_csr(ma_engine *e, int64_t n, const int32_t *rowptr,
                                 const int32_t *col, const double *val, const double *g,
                                 double *d, double rel_tol, int maxiter, double *res,
                                 int64_t *iters);

/* No counterpart in the reference.  For callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc): the gauge-fixed solve of ma_solve_laplacian_csr
 * (H[:n-1,:n-1] d = g[:n-1], d[n-1] = 0) for a symmetric CSR matrix already
 * in device memory (d_rowptr n + 1 entries from 0 to nnz, d_col and d_val
 * nnz entries), right-hand side d_g and solution d_d (n entries each, device
 * memory), by Jacobi-preconditioned conjugate gradients.  It allocates
 * nothing: its work memory is one fixed array per GPU (about 6 x 8 bytes x
 * MA_NOALLOC_MAX_N, held until the process ends) whose address ma_create
 * looks up, so n may not exceed MA_NOALLOC_MAX_N (MA_BAD_INPUT otherwise).
 * Every call on a GPU uses that GPU's one array: calls that overlap on one
 * GPU (from any engines) race and must be serialised by the caller.  Inputs
 * must be complete when the call starts (they are read on the engine's
 * stream); d_d is complete when it returns.  Returns MA_OK, MA_LINEAR_FAIL
 * (maxiter iterations ended above rel_tol; d_d holds the last iterate),
 * MA_SINGULAR (a zero diagonal outside row n-1, or p.Ap <= 0) or
 * MA_BAD_INPUT (sizes or CSR structure). */
#define MA_NOALLOC_MAX_N 262144
ma_status ma_solve_laplacian_csr_noalloc(ma_engine *e, int64_t n, int64_t nnz,
                                         const int32_t *d_rowptr, const int32_t *d_col,
                                         const double *d_val, const double *d_g, double *d_d,
                                         double rel_tol, int maxiter, double *res,
                                         int64_t *iters);

/* Cell masses and first moments (int rho x, int rho y), replaces
 * MA::first_moment (include/MA/lloyd.hpp:30-69).  mom is n x 2 interleaved. */
ma_status ma_first_moment(ma_engine *e, const double *w, double *mass, double *mom);

/* Cell masses, first moments (int rho x, int rho y; n x 2 interleaved) and
 * second moments (int rho x^2, int rho y^2, int rho x y; n x 3 interleaved),
 * replaces MA::second_moment (include/MA/lloyd.hpp:71-123), whose outputs
 * (masses, centroids, inertia) carry these raw integrals.  Any output may be
 * NULL. */
ma_status ma_second_moment(ma_engine *e, const double *w, double *mass, double *mom,
                           double *inertia);

/* Polygons of every fragment (Laguerre cell of Dirac i cut by triangle t) of
 * positive area at weights w, in FP64; replaces the traversal
 * MA::voronoi_triangulation_intersection
 * (include/MA/voronoi_triangulation_intersection.hpp:315-343), which hands
 * each fragment to a callback out(polygon, face, vertex).  Fragments come
 * sorted by (Dirac, triangle): fragment f is Dirac cell[f] (caller index)
 * cut by triangle tri[f] (index into the mesh's triangle list), with
 * vertices xy[2*start[f] .. 2*start[f+1]) (x, y interleaved, absolute
 * coordinates, counter-clockwise); start has nfrag + 1 entries.  *nfrag and
 * *nvert always receive the sizes; if cap_frag < *nfrag or cap_vert < *nvert
 * nothing is copied and MA_CAPACITY is returned (query with 0 and NULL
 * arrays).  Fragments of zero area (a cell touching a triangle along an edge
 * or at a point) are not listed. */
ma_status ma_fragments(ma_engine *e, const double *w, int64_t cap_frag, int64_t cap_vert,
                       int64_t *nfrag, int64_t *nvert, int32_t *cell, int32_t *tri,
                       int64_t *start, double *xy);

/* The Laguerre diagram rasterised, replacing MA::draw_laguerre_diagram
 * (include/MA/rasterization.hpp:491-547) with a put_pixel that sums: the box
 * [x0,x1] x [y0,y1] maps to a width x height pixel grid (pixel (i, j) =
 * [i, i+1] x [j, j+1] in pixel units, row j counted from the box's lower
 * edge), and every fragment adds, to each pixel it covers,
 *   cover x (mean of the density over the fragment's vertices) x colors[cell]
 * with cover = area of fragment cap pixel in pixel units (exact coverage, as
 * rasterize_convex_polygon, :403-470); pixels outside the grid are dropped.
 * colors: n x nc (caller order); img: width x height x nc, written
 * img[(j * width + i) * nc + c] (overwritten).  device_ptrs = 1: w, colors
 * and img are device pointers; w and colors must be complete when the call
 * starts (they are read on the engine's stream, unordered with the caller's
 * streams), and img is complete when it returns. */
ma_status ma_draw_laguerre(ma_engine *e, const double *w, const double *colors, int nc,
                           double x0, double y0, double x1, double y1, int width, int height,
                           double *img, int device_ptrs);

/* Uniform density `density` on a strictly convex polygon (m vertices,
 * interleaved x, y, either orientation), triangulated as a fan from its first
 * vertex: the domain of MA::voronoi_polygon_intersection
 * (include/MA/voronoi_polygon_intersection.hpp:153-188). */
ma_status ma_set_mesh_polygon(ma_engine *e, int m, const double *pxy, double density);

/* Every Dirac's Laguerre cell clipped to the mesh domain, replacing
 * MA::voronoi_polygon_intersection(P, dt, v)
 * (include/MA/voronoi_polygon_intersection.hpp:153-188, itself
 * polygon_halfplane_intersection of include/MA/polygon_intersection.hpp:46-73
 * over the neighbours of v) for all v at once: cell i has vertices
 * xy[2*start[i] .. 2*start[i+1]) (counter-clockwise, no collinear or repeated
 * vertices; none for an empty cell); start has n + 1 entries.  Exact for a
 * convex domain (ma_set_mesh_polygon, grid meshes): the cell polygon is the
 * convex hull of the cell's fragments.  *nvert always receives the total; if
 * cap_vert < *nvert nothing is copied and MA_CAPACITY is returned. */
ma_status ma_cell_polygons(ma_engine *e, const double *w, int64_t cap_vert, int64_t *nvert,
                           int64_t *start, double *xy);

/* Mesh and density from a grey-level image, replacing MA::image_to_pl_function
 * (include/MA/functions.hpp:82-120): pixels is width x height, row-major with
 * the first row at the top (pixel (x, y) at pixels[y * width + x], the layout
 * of CImg's image(x, y)); vertex (i, j) = (-1 + 2i/(width-1), -1 + 2j/(height-1)),
 * index i * height + j, density value pixels(i, height-1-j)/255 + 1e-3; each
 * grid square is split along its (i,j)-(i+1,j+1) diagonal (the reference's
 * Delaunay triangulation picks a diagonal of its own on these cocircular
 * squares), triangles 2 (i (height-1) + j) + {0, 1}.  *total (may be NULL)
 * receives the integral of the density, the reference's return value. */
ma_status ma_set_mesh_image(ma_engine *e, int width, int height, const double *pixels,
                            double *total);

/* Adjoint of the transport cost.  With the dual value
 *   Phi(Y, w, rho) = int rho(x) min_i (|x - y_i|^2 - w_i) dx,
 * W2^2(rho, sum_i nu_i delta_{y_i}) = max_w Phi + <nu, w>, so at the optimal
 * weights (pass the converged w) the envelope theorem gives
 *   dY   (n x 2 interleaved, may be NULL)  dW2^2/dy_i = 2 m_i (y_i - b_i)
 *        (b_i the density centroid of cell i: the Lloyd form of
 *        include/MA/lloyd.hpp:126-144),
 *   dval (nv, may be NULL)  dW2^2/drho_v = sum_i int_{Lag_i} (|x - y_i|^2 - w_i)
 *        phi_v(x) dx, phi_v the P1 hat function of mesh vertex v.
 * At other weights these are the partial derivatives of Phi at fixed w.  The
 * diagram is recomputed (one evaluation); nothing is kept from earlier calls.
 * No counterpart in the reference (it has no derivatives w.r.t. Y or rho). */
ma_status ma_adjoint(ma_engine *e, const double *w, double *dY, double *dval);

ma_status ma_get_eval_info(const ma_engine *e, ma_eval_info *info);

/* Per-cell outcome of the last evaluation, for the Diracs ids[0..count-1]
 * (caller indices): out[i] = number of vertices of the cell polygon built by
 * the register/LDS path (0: empty cell), or -1 if the cell was evaluated by
 * the general kernel. */
ma_status ma_cell_paths(ma_engine *e, int64_t count, const int64_t *ids, int32_t *out);

/* Engine options.  MA_OPT_FORCE_GENERAL (0/1/2): evaluate every cell with the
 * general kernel instead of the register/LDS fast path (1), or with the
 * one-workgroup-per-cell kernel for large cells (2) (for testing the overflow
 * paths); MA_OPT_CAP_CAND: initial capacity of the per-bin candidate
 * lists (grows automatically on overflow); MA_OPT_GRAPHS (0/1, default 1):
 * replay the batches of a long conjugate-gradient solve from a HIP graph. */
typedef enum {
  MA_OPT_FORCE_GENERAL = 1,
  MA_OPT_CAP_CAND = 2,
  MA_OPT_GRAPHS = 3,
  MA_OPT_LOCAL_RINGS = 4, /* rings of bins searched around each Dirac (0..64, default 8) */
  MA_OPT_WALK_BUDGET = 5, /* pyramid nodes per cell before the bin path (default 1024) */
  MA_OPT_AMG_OMEGA = 6,   /* multigrid Jacobi damping in 1/1000 (100..1000, default 850) */
  MA_OPT_AMG_CORR = 7,    /* coarse-correction scaling in 1/1000 (500..3000, default 1500) */
  MA_OPT_AMG_SWEEPS = 8,  /* Jacobi sweeps before and after the coarse correction (1 or 2, default 1) */
  MA_OPT_FAR_CELLS = 10   /* cells whose FP64 construction took the bin path at the previous
                             weights (far from their Diracs), when at least n/16 did: 1 sent to
                             the bin path at once (default), 0 searched from their Diracs
                             first like the others */
} ma_option;
ma_status ma_set_option(ma_engine *e, int option, int64_t value);
void ma_default_solve_opts(ma_solve_opts *o);

#ifdef __cplusplus
}
#endif
#endif /* MA_H */
