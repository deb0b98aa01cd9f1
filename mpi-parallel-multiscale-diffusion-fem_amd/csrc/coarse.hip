// Coarse system of the MsFEM on the unit square/cube with nc cells per side:
//   assembly     DiffusionProblemMultiscale::assemble_system
//                (include/base/diffusion_problem_ms.tpp:161-255; Dirichlet
//                constraints :128-137, Neumann face terms :206-235)
//   solve        DiffusionProblemMultiscale::solve_iterative (:260-296): FP64 CG
//   weights      send_global_weights_to_cell (:301-325) and the fine
//                reconstruction of DiffusionProblemBasis::set_global_weights
//                (include/base/diffusion_problem_basis.tpp:354-377)
// The coarse matrix is kept in structured stencil form Kc[node][3^dim].
#include <algorithm>

#include "msfem_device.hpp"
#include "msfem_kernels.hpp"

namespace msfem {

namespace {

constexpr double kPiD = 3.14592653509793218403; // PI_D of include/coefficients/coefficients.h:21

__device__ __forceinline__ double dirichlet_g(double x, double y) { return (x - 0.5) * (x - 0.5) + (y - 0.5) * (y - 0.5); }
__device__ __forceinline__ double neumann_h(double x, double y) { return cos(2 * kPiD * x) * cos(2 * kPiD * y); }

// One thread per coarse node: gathers A^K, F^K of the <= 2^dim adjacent cells
// in a fixed order (deterministic), adds Neumann face integrals (QGauss(2) on
// faces) and marks the Dirichlet nodes.
template <int DIM>
__global__ void coarse_assemble_kernel(int nc, const double *Ae, const double *Fe, int bc_kind, double *Kc,
                                       double *Fc, unsigned char *cmask, double *cval)
{
  constexpr int NV = 1 << DIM, NS3 = DIM == 2 ? 9 : 27;
  const int np = nc + 1;
  const int nn = DIM == 2 ? np * np : np * np * np;
  const double H = 1.0 / nc, gs = 0.5 / sqrt(3.0);
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < nn; n += gridDim.x * blockDim.x)
    {
      const int I[3] = {n % np, (n / np) % np, DIM == 3 ? n / (np * np) : 0};
      double k[NS3];
#pragma unroll
      for (int t = 0; t < NS3; ++t)
        k[t] = 0;
      double f = 0;
      for (int a = 0; a < NV; ++a) // the node is vertex a of cell I - offset(a)
        {
          int ci[3];
          bool ok = true;
          for (int m = 0; m < DIM; ++m)
            {
              ci[m] = I[m] - ((a >> m) & 1);
              ok = ok && ci[m] >= 0 && ci[m] < nc;
            }
          if (!ok)
            continue;
          const size_t c = DIM == 2 ? (size_t)ci[0] + (size_t)nc * ci[1]
                                    : (size_t)ci[0] + (size_t)nc * (ci[1] + (size_t)nc * ci[2]);
          for (int b = 0; b < NV; ++b)
            {
              int t = 0, mul = 1;
              for (int m = 0; m < DIM; ++m)
                {
                  t += (((b >> m) & 1) - ((a >> m) & 1) + 1) * mul;
                  mul *= 3;
                }
              k[t] += Ae[c * NV * NV + a * NV + b];
            }
          f += Fe[c * NV + a];
          if (bc_kind == 1)
            for (int m = 0; m < DIM; ++m) // face x_m = 1 (boundary ids 1, 3, 5)
              {
                if (ci[m] != nc - 1 || !((a >> m) & 1))
                  continue;
                for (int q = 0; q < (1 << (DIM - 1)); ++q)
                  {
                    double xq[3], w = 1.0, psi = 1.0;
                    int tq = 0;
                    for (int mm = 0; mm < DIM; ++mm)
                      {
                        if (mm == m)
                          {
                            xq[mm] = 1.0;
                            continue;
                          }
                        const double xi = ((q >> tq) & 1) ? 0.5 + gs : 0.5 - gs;
                        ++tq;
                        xq[mm] = (ci[mm] + xi) * H;
                        w *= 0.5 * H;
                        psi *= ((a >> mm) & 1) ? xi : 1.0 - xi;
                      }
                    f += neumann_h(xq[0], xq[1]) * psi * w;
                  }
              }
        }
#pragma unroll
      for (int t = 0; t < NS3; ++t)
        Kc[(size_t)n * NS3 + t] = k[t];
      Fc[n] = f;
      bool con = false;
      for (int m = 0; m < DIM; ++m)
        con = con || I[m] == 0 || (bc_kind == 0 && I[m] == nc);
      cmask[n] = con ? 1 : 0;
      cval[n] = (con && bc_kind == 1) ? dirichlet_g(I[0] * H, I[1] * H) : 0.0;
    }
}

constexpr int kCoarseThreads = 1024;

__device__ __forceinline__ double block_sum(double v, double *red)
{
  v = group_sum<kWave>(v);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0)
    red[wave] = v;
  __syncthreads();
  double s = 0;
  for (int w = 0; w < kCoarseThreads / kWave; ++w)
    s += red[w];
  return s;
}

// Jacobi-preconditioned FP64 CG on the free coarse nodes, one workgroup; vectors in global
// memory.  With `st` it ends a multigrid-preconditioned solve (mg.hip): nothing is left to do if
// that is done, else the CG goes on from its x to its tolerance.  Without: systems whose
// multigrid scratch does not fit the fixed array of the allocation-free entry point.
struct CgVectors {
  double *x, *r, *p, *q, *dinv;
};

template <int DIM>
__global__ void __launch_bounds__(kCoarseThreads) coarse_cg_kernel(int nc, const double *Kc, const double *Fc,
                                                                    const unsigned char *cmask, const double *cval,
                                                                    double rel_tol, int max_iter, double *u,
                                                                    int *iters, CgVectors v5, const MgState *st)
{
  constexpr int NS3 = DIM == 2 ? 9 : 27;
  __shared__ double red[kCoarseThreads / kWave];
  const int np = nc + 1;
  const int nn = DIM == 2 ? np * np : np * np * np;
  double *x = v5.x, *r = v5.r, *p = v5.p, *q = v5.q, *dinv = v5.dinv;
  if (st && st->done)
    {
      for (int n = threadIdx.x; n < nn; n += blockDim.x)
        u[n] = x[n];
      if (threadIdx.x == 0)
        *iters = st->iters;
      return;
    }

  auto nbr = [&](int n, int t) -> int {
    const int ox = t % 3 - 1, oy = (t / 3) % 3 - 1, oz = DIM == 3 ? t / 9 - 1 : 0;
    const int X = n % np + ox, Y = (n / np) % np + oy, Z = (DIM == 3 ? n / (np * np) : 0) + oz;
    if (X < 0 || X >= np || Y < 0 || Y >= np || Z < 0 || Z >= (DIM == 3 ? np : 1))
      return -1;
    return X + np * (Y + np * Z);
  };
  auto matvec = [&](const double *v, int n) -> double { // (K v)_n over all neighbours
    double s = 0;
    for (int t = 0; t < NS3; ++t)
      {
        const int m = nbr(n, t);
        if (m >= 0)
          s += Kc[(size_t)n * NS3 + t] * v[m];
      }
    return s;
  };

  for (int n = threadIdx.x; n < nn; n += blockDim.x)
    {
      if (!st)
        x[n] = cmask[n] ? cval[n] : 0.0;
      p[n] = 0.0;
      dinv[n] = cmask[n] ? 0.0 : 1.0 / Kc[(size_t)n * NS3 + NS3 / 2];
    }
  __syncthreads();
  double bb = 0, rz = 0;
  for (int n = threadIdx.x; n < nn; n += blockDim.x)
    {
      const double rv = cmask[n] ? 0.0 : Fc[n] - matvec(x, n);
      r[n] = rv;
      bb += rv * rv;
      const double z = rv * dinv[n];
      p[n] = z;
      rz += rv * z;
    }
  bb = block_sum(bb, red);
  rz = block_sum(rz, red);
  const double tol = st ? st->tol : rel_tol * sqrt(bb);
  int it = st ? st->iters : 0;
  double rn = sqrt(bb);
  while (rn > tol && it < max_iter)
    {
      double pq = 0;
      for (int n = threadIdx.x; n < nn; n += blockDim.x)
        {
          const double qv = cmask[n] ? 0.0 : matvec(p, n);
          q[n] = qv;
          pq += p[n] * qv;
        }
      pq = block_sum(pq, red);
      const double alpha = rz / pq;
      double rz_new = 0, rr = 0;
      for (int n = threadIdx.x; n < nn; n += blockDim.x)
        {
          x[n] += alpha * p[n];
          const double rv = r[n] - alpha * q[n];
          r[n] = rv;
          rz_new += rv * rv * dinv[n];
          rr += rv * rv;
        }
      rz_new = block_sum(rz_new, red);
      rr = block_sum(rr, red);
      const double beta = rz_new / rz;
      rz = rz_new;
      for (int n = threadIdx.x; n < nn; n += blockDim.x)
        p[n] = r[n] * dinv[n] + beta * p[n];
      rn = sqrt(rr);
      ++it;
      __syncthreads();
    }
  for (int n = threadIdx.x; n < nn; n += blockDim.x)
    u[n] = x[n];
  if (threadIdx.x == 0)
    *iters = it;
}

__global__ void reconstruct_kernel(int n_cells, int nb, const long long *bas_off, const long long *out_off,
                                   const int *n_nodes, const double *bases, const double *w, double *u)
{
  const int cell = blockIdx.y;
  if (cell >= n_cells)
    return;
  const int nn = n_nodes[cell];
  const double *phi = bases + bas_off[cell];
  double wi[8];
  for (int i = 0; i < nb; ++i)
    wi[i] = w[(size_t)cell * nb + i];
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < nn; n += gridDim.x * blockDim.x)
    {
      double s = 0;
      for (int i = 0; i < nb; ++i)
        s += wi[i] * phi[(size_t)i * nn + n];
      u[out_off[cell] + n] = s;
    }
}

} // namespace

hipError_t launch_coarse_assemble(int dim, int nc, const double *Ae, const double *Fe, int bc_kind, double *Kc,
                                  double *Fc, unsigned char *cmask, double *cval, hipStream_t st)
{
  const int nn = dim == 2 ? (nc + 1) * (nc + 1) : (nc + 1) * (nc + 1) * (nc + 1);
  const int grid = (nn + 255) / 256;
  if (dim == 2)
    hipLaunchKernelGGL(coarse_assemble_kernel<2>, dim3(grid), dim3(256), 0, st, nc, Ae, Fe, bc_kind, Kc, Fc, cmask,
                       cval);
  else
    hipLaunchKernelGGL(coarse_assemble_kernel<3>, dim3(grid), dim3(256), 0, st, nc, Ae, Fe, bc_kind, Kc, Fc, cmask,
                       cval);
  return hipGetLastError();
}

// Iterations of the multigrid-preconditioned CG that one call enqueues (those not needed end at
// once, at ~2 us a launch); the Jacobi CG takes over what is not done then.  MsFEM
// systems of 2..128 cells per side reach 1e-13 in at most 10.
constexpr int kMgIterations = 16;

// Up to this many cells per side the Jacobi CG of one workgroup is done before the multigrid's
// chain of launches, in 2D and 3D (us, multigrid / Jacobi, zero and reference boundary data): 3D 3
// 228, 328 / 57, 120; 7 799, 829 / 211, 330; 11 1184, 1255 / 703, 1137; 12 1184, 1253 / 887, 1688;
// 2D 5 139, 160 / 77, 99; 11 232, 236 / 168, 220; 12 229, 235 / 191, 246.
constexpr int kJacobiMaxCells = 11;

static size_t jacobi_work_doubles(int dim, int nc)
{
  const size_t np = nc + 1;
  return 5 * (dim == 2 ? np * np : np * np * np);
}

// Sizes that halve evenly to a small grid; the others once had the Jacobi CG alone and its
// smaller scratch, which they still fall back to where the scratch is limited.
static bool halves_evenly(int dim, int nc)
{
  while (nc % 2 == 0 && nc >= 4)
    nc /= 2;
  return (dim == 2 ? (nc + 1) * (nc + 1) : (nc + 1) * (nc + 1) * (nc + 1)) <= 343;
}

size_t coarse_solve_work_doubles(int dim, int nc)
{
  return std::max((size_t)mg_layout(dim, nc).total, jacobi_work_doubles(dim, nc));
}

size_t coarse_solve_least_doubles(int dim, int nc)
{
  return halves_evenly(dim, nc) ? coarse_solve_work_doubles(dim, nc)
                                : std::min(coarse_solve_work_doubles(dim, nc), jacobi_work_doubles(dim, nc));
}

template <int DIM>
static hipError_t coarse_solve(int nc, const double *Kc, const double *Fc, const unsigned char *cmask, const double *cval,
                               double rel_tol, int max_iter, double *u, int *iters, double *work, size_t work_doubles,
                               hipStream_t st)
{
  const MgLayout g = mg_layout(DIM, nc);
  CgVectors v;
  const MgState *state = nullptr;
  if (nc > kJacobiMaxCells && (size_t)g.total <= work_doubles)
    {
      hipError_t e = launch_mg_setup(DIM, g, Kc, Fc, cmask, cval, rel_tol, max_iter, work, st);
      if constexpr (DIM == 2) // (3D grids beyond kJacobiMaxCells do not fit one workgroup)
        if (e == hipSuccess && g.tail == 0)
          return launch_mg_small(g, Kc, u, iters, work, st);
      if (e == hipSuccess)
        e = launch_mg_iterations(DIM, g, kMgIterations, Kc, work, st);
      if (e != hipSuccess)
        return e;
      v = {work + g.off_cx, work + g.off_cr, work + g.off_cp, work + g.off_cq, work + g.off_d[0]};
      state = (const MgState *)(work + g.off_state);
    }
  else
    {
      const size_t nn = jacobi_work_doubles(DIM, nc) / 5;
      v = {work, work + nn, work + 2 * nn, work + 3 * nn, work + 4 * nn};
    }
  hipLaunchKernelGGL(coarse_cg_kernel<DIM>, dim3(1), dim3(kCoarseThreads), 0, st, nc, Kc, Fc, cmask, cval, rel_tol,
                     max_iter, u, iters, v, state);
  return hipGetLastError();
}

hipError_t launch_coarse_solve(int dim, int nc, const double *Kc, const double *Fc, const unsigned char *cmask,
                               const double *cval, double rel_tol, int max_iter, double *u, int *iters, double *work,
                               size_t work_doubles, hipStream_t st)
{
  return dim == 2 ? coarse_solve<2>(nc, Kc, Fc, cmask, cval, rel_tol, max_iter, u, iters, work, work_doubles, st)
                  : coarse_solve<3>(nc, Kc, Fc, cmask, cval, rel_tol, max_iter, u, iters, work, work_doubles, st);
}

hipError_t launch_reconstruct(int n_cells, int nb, const long long *bas_off, const long long *out_off,
                              const int *n_nodes, const double *bases, const double *w, double *u, hipStream_t st)
{
  if (n_cells == 0)
    return hipSuccess;
  hipLaunchKernelGGL(reconstruct_kernel, dim3(16, n_cells), dim3(256), 0, st, n_cells, nb, bas_off, out_off, n_nodes,
                     bases, w, u);
  return hipGetLastError();
}

} // namespace msfem
