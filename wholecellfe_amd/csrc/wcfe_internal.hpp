// Host-side launcher declarations shared by the HIP translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "band_plan.hpp"
#include "wcfe_device.hpp"

namespace wcfe {

// Work list of one launch: map[item] = (cell << 20) | (item index within the
// cell), for item in [0, total).
struct WorkList {
  const int *map;
  int total;
};

// ---- assembly and vector kernels (k_assemble.hip) ----
enum AsmMode : int { ASM_FULL = 0, ASM_RESIDUAL = 1, ASM_STRAIN = 2 };

template <class T>
void launch_fill_systems(hipStream_t s, const CellParams *cp, const int *cells, int ncell, int max_npad, T *K,
                         const int *rank, int lower_only = 0);
void launch_fill(hipStream_t s, double *p, long long n, double value);
void launch_copy(hipStream_t s, const void *src, void *dst, long long bytes);
// K: dense systems; Kb: block-CSR values of sparse cells (View::el_bpos)
template <class T>
void launch_assemble(hipStream_t s, const View &v, int e_begin, int e_end, int mode, T *K, T *Kb, double *G,
                     double *Ke64, double *Rea, double *MM);
// whole-batch assembly: element pass over [e_begin, e_end) (all colours),
// then a node gather over [n0, n1) (ASM_FULL or ASM_RESIDUAL)
struct GatherPlan {
  const int *start;   // per node: groups [start[n], start[n+1])
  const int *col;     // per group: column node
  const int *bpos;    // per group: block-CSR position (sparse cells), else -1
  const int *cstart;  // per group: contributions [cstart[g], cstart[g+1])
  const int *ke;      // per contribution: offset of the 2 x 2 block in Ke64
  const int *node;    // per group: its row node
  int g0, g1;         // groups of the node range [n0, n1)
};
template <class T>
void launch_assemble_gather(hipStream_t s, const View &v, int e_begin, int e_end, int mode, const int *node_cell,
                            const int *adj_start, const int *adj, const GatherPlan &gp, int n0, int n1, double *Ge,
                            double *Ke64, double *G, T *K, T *Kb, int lower_only);
// UL strain increments and lumped masses: every node of the range over its
// elements in element order (node_cell null: cell 0; else converged UL cells)
void launch_node_strain(hipStream_t s, const View &v, const int *node_cell, const int *adj_start, const int *adj,
                        int n0, int n1, double *Rea, double *MM);
void launch_element_dump(hipStream_t s, const View &v, int e_begin, int e_end, double *Ge, double *Ke);
// per-cell norms of cells above NORM_CHUNK entries: partial sums per chunk
// (stride per cell = the batch's largest chunk count) and an arrival counter
// per cell (zero between launches).  At most 16 chunks: each chunk's release
// of its partial sum writes back an L2 (500000 unknowns in 123 chunks 23 us,
// in 16 11; 20600 unknowns in 1 chunk 12, in 3 or 6 7).
constexpr int NORM_CHUNK = 8192;
__host__ __device__ inline int norm_chunks(int ndof) {
  const int n = (ndof + NORM_CHUNK - 1) / NORM_CHUNK;
  return n < 1 ? 1 : n > 16 ? 16 : n;
}
struct NormWork {
  double *part = nullptr;
  unsigned *cnt = nullptr;
  int stride = 1;
};
// which 0 also starts a new linear solve (the refinement state), and with K
// takes the dense cells' pivot thresholds from its diagonal (64 units of
// roundoff of T times the largest entry); which 1 with lin_rtol >= 0 applies
// the refinement control to each refining cell
template <class T>
void launch_cell_norm(hipStream_t s, const CellParams *cp, CellState *cs, const int *cells, int ncell,
                      const double *vec, int which, int only_active, double lin_rtol = -1.0,
                      const NormWork &nw = NormWork(), const T *K = nullptr);
void launch_neg_copy(hipStream_t s, const double *src, double *dst, long long n);
void launch_matvec_ir(hipStream_t s, const View &v, const int *node_cell, const int *adj_start, const int *adj,
                      const double *Ke64, const double *G, const double *delta, double *r, int node_begin,
                      int node_end, const CellState *cs, const BndView &bv);
void launch_perm_gather(hipStream_t s, const int *node_cell, const CellParams *cp, const int *kpos, const double *r,
                        double *rp, int n0, int n1);
void launch_perm_scatter(hipStream_t s, const int *node_cell, const CellParams *cp, const CellState *cs,
                         const int *kpos, const double *dp, double *delta, int n0, int n1, int accumulate);
void launch_update_x(hipStream_t s, double2 *x, const double *delta, int node_begin, int node_end);
void launch_newton_control(hipStream_t s, CellState *cs, const int *cells, int ncell, double rtol, double atol);
void launch_commit_nodes(hipStream_t s, const View &v, const int *node_cell, double2 *X, double2 *x, double *ea,
                         double *cC, double2 *fau, const double *Rea, const double *MM, int node_begin, int node_end,
                         double dt);
// Bell kinetics of the springs (k_commit_springs)
struct BellArgs {
  double dt, k_on, k_off0, f_b;
  unsigned key_lo, key_hi;
  const int *replica;  // per cell: its Philox stream
  int *transitions;
};
void launch_commit_springs(hipStream_t s, const View &v, const int *sp_cell, const int *sp_elem, const int *sp_local,
                           double *state, double *anchor, int s_begin, int s_end, const BellArgs &bell);
void launch_commit_cells(hipStream_t s, CellState *cs, const int *cells, int ncell, double dt);
void launch_remap_nodes(hipStream_t s, int n_new, const int *src0, const int *src1, const double *w, int old_off,
                        const double2 *X, const double2 *x, const double *ea, const double *cC, const double2 *fau,
                        double2 *Xn, double2 *xn, double *ean, double *cCn, double2 *faun);

// ---- boundary and body forces (k_boundary.hip) ----
enum : int { REF_BEND = 0, REF_AREA = 1, REF_AP = 2 };
struct RefBoundaryArgs {
  double k_bend, tot_area, k_area, area_0, dt, rate, quantum, density;
  unsigned key_lo, key_hi, draw;
};
// cst: N+1 candidate offsets (empty range = interior vertex), cand: (nj, nint)
void launch_ref_boundary(hipStream_t s, int which, int n_nodes, const int *cst, const int2 *cand, const double *x,
                         const RefBoundaryArgs &a, const double *u, double *F, int *n_open);
void launch_ref_area_tot(hipStream_t s, int n_tris, const int *tris, const double *x, double *out);
void launch_bnd_frames(hipStream_t s, const BndView &bv, const double2 *x, int b0, int b1);
void launch_cell_area(hipStream_t s, const CellParams *cp, const int *cells, int ncell, const int *crange, int ncolor,
                      const int *el_tri, const double2 *x, double *area);
void launch_cell_gdot(hipStream_t s, const CellParams *cp, const int *cells, int ncell, const BndView &bv,
                      const double *delta);
template <class T>
void launch_node_terms(hipStream_t s, bool full, const View &v, const BndView &bv, const int *node_cell, int n0, int n1,
                       T *K, T *Kb, const int *row_ptr, const int *bcol, const int *diag_pos, double *G);
// the end of a Newton step with one workgroup per cell: x += delta, the FP64
// residual and its norm, the Newton test and the commit of a converged cell
// most elements of a cell: larger ones keep one workgroup longer than the
// batch-wide launches take (us per Newton step, one workgroup per cell /
// launches: one cell of 1000 elements 188 / 192, 1300 216 / 218, 1700 278 / 277,
// 2700 328 / 317, 11500 727 / 646; 12 UL cells of 1300 295 / 308, of 3000
// 497 / 492; FP64 alike)
constexpr int FINISH_ELEMS = 1700;
struct FinishArgs {
  double2 *X, *x, *fau;
  double *ea, *cC, *Ge, *G, *Rea, *MM, *sp_state, *sp_anchor;
  const double *delta;
  const int *celem;  // every cell's elements (elem_off), in element order
  const int *adj_start, *adj, *sp_elem, *sp_local;
  BndView bv;
  BellArgs bell;
  double rtol, atol, dt;
};
void launch_cell_finish(hipStream_t s, const View &v, const FinishArgs &f, const int *cells, int ncell);

// ---- dense LU and triangular solves (k_lu.hip) ----
// Dinv holds, per cell and diagonal block, the inverses of the block's unit
// lower and upper triangles (2 x 64 x 64 per block, npad * 128 per cell).
template <class T>
void launch_lu_diag_inv(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K, T *Dinv);
template <class T>
void launch_lu_panel_pp(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K,
                        int *ipiv, T *Dinv, int rows);
template <class T>
void launch_lu_laswp(hipStream_t s, const CellParams *cp, const WorkList &wl, int k, T *K, const int *ipiv);
template <class T>
void launch_lu_trsm(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K,
                    const T *Dinv);
template <class T>
void launch_lu_gemm(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K, T *Dinv,
                    int next_diag, int npanel, int strip, hipEvent_t ev_start = nullptr, hipEvent_t ev_stop = nullptr);
template <class T>
void launch_lu_solve(hipStream_t s, const CellParams *cp, const CellState *cs, const int *cells, int ncell,
                     const T *K, const T *Dinv, const int *ipiv, int pivoting, const double *r, double *delta,
                     int max_npad, int accumulate);
// static pivoting: forward and backward sweeps with one workgroup per block
// row (fwd: items (cell << 20 | block) by cell, block ascending; bwd: block
// descending) over the cells `cells` (for the any-refining test); yw: the
// exchange buffer, lu_solve_exchange_bytes(system rows) bytes, zeroed once;
// sync: SOLVE_SYNC_INTS ints, zeroed once
constexpr int SOLVE_SYNC_INTS = 4;
template <class T>
void launch_lu_solve_mw(hipStream_t s, const CellParams *cp, CellState *cs, const int *cells, int ncell,
                        const WorkList &fwd, const WorkList &bwd, const T *K, const T *Dinv, const double *r,
                        double *delta, void *yw, int *sync, int accumulate);
size_t lu_solve_exchange_bytes(long long rows, int elem_size);
size_t lu_solve_lds_bytes(int npad, int elem_size);
size_t lu_solve_max_dynamic(size_t max_lds);
// block bandwidth up to which one workgroup per cell runs the triangular sweeps
constexpr int SOLVE_WG_MAX_BW = 8;
// concurrent cell groups of the dense LU chosen automatically for wide bands
constexpr int AUTO_GROUPS_MAX = 4;
hipError_t lu_prepare_attributes(size_t max_lds);

// ---- band LU over the plans of band_plan.hpp (k_band.hip) ----
// the forward substitution of the first solve inside the fused block steps:
// y (band numbering, per cell at sys_off) = L^-1 P (-G); kinv: per band row
// its batch dof (-1: padding); slot: the plans' slots; y null: none
template <class T> struct StepFwd {
  T *y = nullptr, *slot = nullptr;
  const int *kinv = nullptr;
  const double *G = nullptr;
  int store_id = 0;  // also store the identity half of each diagonal pair (the spread-out solve reads it)
};
// one launch of n items (one level of the cells' plans)
template <class T>
void launch_lu_step(hipStream_t s, const CellParams *cp, CellState *cs, const StepItem *items, int n,
                    const BlockRef *refs, const FwdOp *fops, T *K, T *Dinv, StepFwd<T> fwd,
                    hipEvent_t ev_start = nullptr, hipEvent_t ev_stop = nullptr);
// every level of every listed cell in one launch, one workgroup per cell
void launch_lu_cell(hipStream_t s, const CellParams *cp, CellState *cs, const int2 *ranges, int ncell,
                    const StepItem *items, const BlockRef *refs, const FwdOp *fops, float *K, float *Dinv,
                    StepFwd<float> fwd, hipEvent_t ev_start = nullptr, hipEvent_t ev_stop = nullptr);
// one workgroup of a triangular sweep
struct SweepWG {
  int cell;
  SweepPart part;
};
// its vectors (band numbering, per cell at sys_off, but rhs and delta): SL_RHS
// blocks from rhs (from_y: from y), SL_Y from y, SL_X from x; SL_OUT_Y to x,
// SL_OUT_D to delta
template <class T> struct SweepVec {
  const double *rhs;
  const T *y;
  T *x, *slot;
  double *delta;
  int from_y;
};
// max_loc: the most LDS vector blocks of a workgroup in the launch
template <class T>
void launch_band_sweep(hipStream_t s, const CellParams *cp, const CellState *cs, const SweepWG *wgs, int nwg,
                       int max_loc, const SweepOp *ops, const SweepLoc *locs, const int *accs, const T *K,
                       const T *Dinv, const int *kinv, const SweepVec<T> &sv, int accumulate);
// refinement sweeps it0 .. max_refine - 1 of a cell by one workgroup (solve,
// FP64 residual, norm and control); parts: the cell's whole sweep and its
// backward half (the first solve after the fused block steps); z, inc: batch
// vectors for cells with smw; dirs: theirs too, 2 REFINE_DIRS vectors of a cell
// from its dirs on
constexpr int REFINE_DIRS = 12, REFINE_MORE = 8;
struct RefineWG {
  int cell;
  SweepPart whole, bwd;
  long long dirs;
};
struct RefineArgs {
  const int *el_tri, *adj_start, *adj;
  const double *Ke64, *G;
  double *r, *delta, *z, *inc, *dirs;
  BndView bv;
  double lin_rtol;
  int it0, max_refine, fwd_done;
  const RefineArgs *mem;  // the same pointers in device memory, for the path that seldom runs (cells with smw)
};
size_t refine_max_dynamic(size_t max_lds);
template <class T>
void launch_band_refine(hipStream_t s, const CellParams *cp, CellState *cs, const RefineWG *wgs, int nwg, int max_loc,
                        const SweepOp *ops, const SweepLoc *locs, const int *accs, const T *K, const T *Dinv,
                        const int *kinv, const SweepVec<T> &sv, const RefineArgs &ra);
hipError_t band_prepare_attributes(size_t max_lds);

// ---- sparse path: block-CSR systems and batched PCG (k_csr.hip) ----
constexpr int CG_ROWS = 1024;  // nodes per chunk (one thread per node)
enum CgMode : int { CG_INIT = 0, CG_STEP = 1 };
// per-cell conjugate-gradient state (one entry per cell; used by sparse cells)
struct CgState {
  double rz, rr, rr0, pq, alpha, beta;
  double tol;             // this solve's relative tolerance (set at its start)
  int iters, done, breakdown, total_iters;
  int chunk_off, nchunk;  // the cell's chunks in the chunk list / partials
  int pad_[2];
};
template <class T> struct CgVectors {
  T *x, *r, *z, *p, *q, *s, *dinv;  // 2 N each (dinv: 4 N); z = M^-1 r, q = K z, s = K p
  long long pstride;                // partial sums: three arrays of pstride (one per chunk of the batch)
};
template <class T> void launch_zero(hipStream_t s, T *p, long long n);
template <class T>
void launch_bsr_diag_inv(hipStream_t s, const int4 *chunks, int nchunk, const int *diag_pos, const T *val, T *dinv);
// chunks [cbase, cbase + nchunk) of the batch's chunk list
// lanes: 4, 8 or 16 lanes per block row in the SpMV
// rtol: cg_rtol; lin_rtol: the refinement's target (a later sweep's solve
// stops at max(cg_rtol, 0.1 lin_rtol / the cell's relative residual so far))
template <class T>
void launch_pcg_init(hipStream_t s, const int4 *chunks, int cbase, int nchunk, const int *cells, int ncell,
                     const CellState *cs, CgState *cg, const int *row_ptr, const int *col, const T *val,
                     const double *rhs, const CgVectors<T> &v, double *partials, double rtol, double lin_rtol,
                     int max_iter, int lanes);
// one iteration: the update (step: with the scalars formed from the last
// SpMV's partials, gin -> gout; else with gin's), then the SpMV
template <class T>
void launch_pcg_iteration(hipStream_t s, const int4 *chunks, int cbase, int nchunk, const CgState *gin,
                          CgState *gout, int step, const int *row_ptr, const int *col, const T *val,
                          const CgVectors<T> &v, double *partials, double rtol, int max_iter, int lanes);
// the scalars of the last SpMV by one workgroup per cell, gin -> gout
void launch_pcg_check(hipStream_t s, const int *cells, int ncell, const CellState *cs, const CgState *gin,
                      CgState *gout, const double *partials, long long pstride, double rtol, int max_iter);

template <class T>
void launch_pcg_finish(hipStream_t s, const int4 *chunks, int nchunk, const CellState *cs, const T *x, double *delta,
                       int accumulate);

// ---- calculateForce_FA on device pointers with no allocation (wcfe_noalloc.hip) ----
hipError_t noalloc_init(int device);
int noalloc_force_fa(int device, hipStream_t s, int n_nodes, int n_tris, const int *d_tris, const double *d_x,
                     const double *d_cC, const double *d_fau, int law, double kint, double *d_F, int *d_n_bad,
                     std::string &err);

// ---- reference-shaped stateless kernels (k_reference.hip) ----
void launch_eval_exp(hipStream_t s, long long n, const double *x, double *y);
void launch_ref_force_fa(hipStream_t s, int n_nodes, const int *ring_start, const int *ring, const int *tris,
                         const double *x, const double *cC, const double *fau, int law, double kint, double *F);
// uniform grid over substrate triangles (point location); list[start[c] ..
// start[c+1]) = triangles whose widened bounding box meets cell c, ascending
struct PointGrid {
  double ox, oy, inv_h;
  int gx, gy;
  const int *start, *list;
};
constexpr int SUBS_MAX_HITS = 16;  // containing substrate triangles per cell node (shared vertices)
void launch_ref_update_fa(hipStream_t s, int n_nodes, const double *X, const double *x, double *cA, double *cC,
                          double *fau, double dt, const PointGrid &grid, const int *stris, const double *SX,
                          const double *Sx, int law, double kint, int *n_unlocated);
// substrate hits: hit k of node i at k n_nodes + i, the first SUBS_FIRST_HITS
// planes apart from the others; 9 values per hit
constexpr int SUBS_FIRST_HITS = 2;
struct SubsHits {
  int *n, *overflow, *tri, *tri_more;
  double *val, *val_more;
};
void launch_ref_force_fa_subs(hipStream_t s, int n_nodes, const int *ring_start, const int *ring, const int *tris,
                              const double *x_cell, const double *cC, const double *fau, const PointGrid &grid,
                              const int *stris, const double *Sx, int law, double kint, const SubsHits &hits);
// K from the caller's dense matrices (FP64, packed), identity in the padding
template <class T>
void launch_dense_load(hipStream_t s, const CellParams *cp, int n_sys, int max_npad, const double *A64,
                       const long long *a_off, T *K);
void launch_dense_residual(hipStream_t s, const CellParams *cp, const CellState *cs, const int *cells, int ncell,
                           int max_ndof, const double *A64, const long long *a_off, const double *b, const double *x,
                           double *r);

// Host-side VTK frame writer (wcfe_vtk.hip): one cell or substrate, the
// reference's file layout.  Positions and fa_u with 2 (z = 0) or 3 components
// per node; strain 3 (planar [xx,yy,xy]) or 6 (Voigt) per node.
struct VtkInput {
  const char *path = nullptr;
  int style = 0, n_nodes = 0, n_tris = 0;
  const int32_t *tris = nullptr;
  const double *x = nullptr, *fau = nullptr, *ea = nullptr, *cA = nullptr, *cC = nullptr;
  int x_stride = 3, fau_stride = 3, ea_kind = 6;
  double cA_default = 100.0;  // the reference's initial c_A (main.cpp:674-677)
  int law = 1;
  double kint = 0.0, time = 0.0;
};
int write_vtk_file(const VtkInput &in, std::string &err);

}  // namespace wcfe
