// Host-side launchers of the MsFEM kernels (implemented in the .hip files).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "msfem_device.hpp"

namespace msfem {

// local2d.hip
int local2d_variants(int nf);
// whether a class (resolution, storage mode, launch-shape id) runs the two-level form
bool local2d_coarse_space(int nf, int mode, int variant);
// inverse coarse matrices of the two-level form (nf = 64, 128; boxes or general
// quadrilaterals): cinv [cells in class][49 * 49]
hipError_t launch_coarse_setup_2d(int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                                  const double *verts, const double *coef, const long long *coef_off, double *cinv,
                                  hipStream_t st);
// the intermediate levels' inverse diagonals of a 64^2 two-level class
// (mlinv [cells in class][kMlFloats])
hipError_t launch_ml_diag_2d(int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                             const double *verts, const double *coef, const long long *coef_off, float *mlinv,
                             hipStream_t st);
hipError_t launch_local_solve_2d(bool fp32, int mode, int nf, int variant, const LocalArgs &a, hipStream_t st);
// verts: general quadrilaterals [n_cells][4][2] or nullptr (boxes)
hipError_t launch_prep_couplings_2d(int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                                   const double *verts, const double *coef, const long long *coef_off,
                                   double *cond, const long long *cond_off, bool want32, hipStream_t st);
hipError_t launch_prep_cond_2d(int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                               const double *verts, const double *coef, const long long *coef_off, double *cond,
                               const long long *cond_off, hipStream_t st);
// Dirichlet data N_i (BasisQ1 by monomial inversion) of general quadrilaterals
// at their boundary fine nodes, written into every basis block.
hipError_t launch_quad_dirichlet_2d(int n_cells_class, const int *cells, int nf, const double *verts, double *bases,
                                    const long long *bas_off, hipStream_t st);

// local3d.hip
int local3d_variants(int nf);
hipError_t launch_local_solve_3d(bool fp32, int nf, int variant, const LocalArgs &a, hipStream_t st);

// direct.hip: the direct local solves in 2D (nested dissection, FP64).
struct DirectFront;
struct DirectLeaf;
struct DirectLeafType;
constexpr int kDirectLevels = 4; // front levels of the largest resolution
// What the host keeps of a resolution's plan (direct_plan.hpp); the tables are in device memory.
struct DirectHost {
  int nf, depth;
  int n_fronts[kDirectLevels], max_rows[kDirectLevels], max_elim[kDirectLevels];
  size_t fronts_at[kDirectLevels], leaves_at, types_at, tables_at; // byte offsets in the device tables
  long long cell_doubles;                                          // factor scratch of one cell
};
struct DirectArgs {
  int nf, depth, level, nb, nb_solve, coef_kind, q1_start;
  int second;                     // 1: the correction pass (unknown = a.corr, right-hand side = a.loads)
  int n_fronts[kDirectLevels];
  const DirectFront *fronts[kDirectLevels];
  const DirectLeaf *leaves;
  const DirectLeafType *types;
  const uint32_t *tables;
  const int *cells;               // batch cells of this chunk, one per slot
  const double *box, *verts, *coef;
  const long long *coef_off, *bas_off;
  double *bases;
  double *scratch;                // [slot][cell_doubles]
  long long cell_doubles;
  const int *need;                // correction pass: cells to work on; nullptr = all
  const double *loads;            // correction pass: residuals [slot][4][nodes]
  double *loads_out, *corr;       // [slot][4][nodes]
  double *cond;                   // stored fine cells: conductances [slot][6][nf^2]
  double *part;                   // residual sums [slot][task][12]
  int *need_out;                  // [slot]
  const double *ptol;
  double rel_tol, abs_tol;
  int *iters, *status;
  double *resid;
  // the pass's unknown: bases, or the corrections
  __device__ double *x_of(int slot, int cell) const
  {
    return second ? corr + (size_t)slot * 4 * (nf + 1) * (nf + 1) : bases + bas_off[cell];
  }
};
bool direct_supported(int dim, int nf);
void direct_host_plan(int nf, DirectHost &h, std::vector<char> &blob);
size_t direct_scratch_doubles(const DirectHost &h, int n_cells, int coef_kind, bool general);
hipError_t launch_direct_solve(const DirectHost &h, const char *blob, const LocalArgs &in, int n_cells, int coef_kind,
                               double *scratch, hipStream_t st);

// generic.hip: the local solve for resolutions and coefficient kinds outside the
// tuned kernels.  Element matrices [nf^d][2^d][2^d] per cell (offsets elem_off,
// generic_elem_doubles each); work: generic_work_doubles per problem.
size_t generic_elem_doubles(int dim, int nf);
size_t generic_work_doubles(int dim, int nf);
hipError_t launch_generic_prep(int dim, int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                               const double *verts, const double *coef, const long long *coef_off, double *elem,
                               const long long *elem_off, hipStream_t st);
hipError_t launch_generic_solve(int dim, int nf, const LocalArgs &a, double *work, hipStream_t st);
// Dirichlet data N_i (BasisQ1 by monomial inversion) of general hexahedra at
// their boundary fine nodes, written into every basis block.
hipError_t launch_hex_dirichlet_3d(int n_cells_class, const int *cells, int nf, const double *verts, double *bases,
                                   const long long *bas_off, hipStream_t st);

// element.hip: A^K, F^K of every cell of one size class; partition-of-unity fix-up.
struct ElementArgs {
  int n_cells_class;
  const int *cells;
  int dim, nf, nb;
  int coef_kind;              // coefficient kind of the batch (MSFEM_COEF_*)
  const double *box;
  const double *verts;        // general cells [n_cells][2^d][d] or nullptr
  const double *coef;
  const long long *coef_off;
  const double *cond;         // 2D conductance tiles when the class used kModeGlobal (else nullptr)
  const long long *cond_off;
  const double *bases;
  const long long *bas_off;
  int rhs_kind;
  double rhs_value;
  double *Ae, *Fe;
};
hipError_t launch_element(const ElementArgs &a, hipStream_t st);
hipError_t launch_pou_fixup(int n_cells_class, const int *cells, int dim, int nf, double *bases,
                            const long long *bas_off, hipStream_t st);

// energy.hip: energy-norm control of the local solves (box cells).  lam_lb
// [n_cells]: lower bound of lambda_min(K_II); ptol [n_cells][nb] (or nullptr):
// tau sqrt(lam_lb e_lb), the residual norm that guarantees a relative
// energy-norm error <= tau; bound [n_cells][nb]: the a posteriori bound from
// the final residual norms and A^K_ii (lam_lb nullptr: NaN).
hipError_t launch_energy_terms(int dim, int n_cells_class, const int *cells, int nf, int coef_kind, const double *box,
                               const double *coef, const long long *coef_off, double tau, double *lam_lb,
                               double *ptol, hipStream_t st);
hipError_t launch_energy_bound(int n_cells_class, const int *cells, int nb, int pou, const double *lam_lb,
                               const double *resid, const double *Ae, double *bound, hipStream_t st);
// d = x - y (n doubles); err[c][i] = sqrt(max(Ad_ii, 0) / Ar_ii)
hipError_t launch_sub(size_t n, const double *x, const double *y, double *d, hipStream_t st);
hipError_t launch_energy_ratio(int n_cells, int nb, const double *Ad, const double *Ar, double *err, hipStream_t st);

// mg.hip: multigrid-preconditioned CG on structured stencil matrices.
// Scratch layout (offsets in doubles).
constexpr int kMgMaxLevels = 15;
struct MgLayout {
  int levels, tail;                  // levels; the first of those that one workgroup keeps in LDS
  int n[kMgMaxLevels];               // cells per side of level l (n[0] = nc, n[l + 1] = ceil(n[l] / 2))
  long long nn[kMgMaxLevels];        // nodes of level l
  long long off_x[kMgMaxLevels], off_t[kMgMaxLevels], off_d[kMgMaxLevels], off_b[kMgMaxLevels], off_A[kMgMaxLevels];
  long long off_cx, off_cr, off_r1, off_cp, off_p1, off_cq; // CG vectors on level 0 (r and p twice)
  long long off_part, off_inv, off_state; // partial sums, inverse of the coarsest matrix, MgState
  long long total;
};
struct MgState {
  double rz[2], rnorm, tol, rel_tol;
  int iters, max_iter, done, converged, begun, parts_dir;
};
MgLayout mg_layout(int dim, int nc);
// Galerkin levels, x = Dirichlet values, residual, state; then blocks of an even number of
// iterations until the state says done (iterations past that end at once).  The solution is at
// w + off_cx.  launch_mg_small: the whole iteration of a 2D system with g.tail == 0.
hipError_t launch_mg_setup(int dim, const MgLayout &g, const double *Kc, const double *Fc, const unsigned char *cmask,
                           const double *cval, double rel_tol, int max_iter, double *w, hipStream_t st);
hipError_t launch_mg_iterations(int dim, const MgLayout &g, int count, const double *Kc, double *w, hipStream_t st);
hipError_t launch_mg_small(const MgLayout &g, const double *Kc, double *u, int *iters, double *w, hipStream_t st);

// coarse.hip
hipError_t launch_coarse_assemble(int dim, int nc, const double *Ae, const double *Fe, int bc_kind, double *Kc,
                                  double *Fc, unsigned char *cmask, double *cval, hipStream_t st);
hipError_t launch_coarse_solve(int dim, int nc, const double *Kc, const double *Fc, const unsigned char *cmask,
                               const double *cval, double rel_tol, int max_iter, double *u, int *iters,
                               double *work, size_t work_doubles, hipStream_t st);
size_t coarse_solve_work_doubles(int dim, int nc);  // scratch of the coarse solve
size_t coarse_solve_least_doubles(int dim, int nc); // the least it runs with
hipError_t launch_reconstruct(int n_cells, int nb, const long long *bas_off, const long long *out_off,
                              const int *n_nodes, const double *bases, const double *w, double *u, hipStream_t st);

// noalloc.hip: the fixed device scratch of the allocation-free entry point
// (one copy per GPU).  noalloc_register_device looks up this device's address
// (the device must be current); noalloc_scratch returns it (nullptr before).
hipError_t noalloc_register_device(int device);
double *noalloc_scratch(int device);
size_t noalloc_scratch_bytes();

// fine.hip: fine-scale standard FEM (element matrices and loads).
hipError_t launch_fine_elements_2d(int n, int coef_kind, const double *coef, int rhs_kind, double rhs_value,
                                   double *Ae, double *Fe, hipStream_t st);

} // namespace msfem
