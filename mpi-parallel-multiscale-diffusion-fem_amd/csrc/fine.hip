// Fine-scale standard FEM on the unit square: the reference's
// DiffusionProblem<dim> (include/base/diffusion_problem.tpp:40-279), the
// single-scale Q1 solve on the fine mesh that the MsFEM approximates.
//   * element matrices and loads of every fine cell (QGauss(2), :150-183);
//   * assembly with the reference's boundary data: the coarse assembly kernel
//     applied to the fine cells (Dirichlet g on x_k = 0, Neumann h on x_k = 1);
//   * solve: the multigrid-preconditioned CG of mg.hip (the reference: CG +
//     AMG, :243-279), in blocks of iterations captured once as a HIP graph and
//     replayed until the device-side state says done.
#include "msfem.h"
#include "msfem_device.hpp"
#include "msfem_kernels.hpp"

namespace msfem {

namespace {

constexpr int kFineThreads = 256;

// QGauss(2) element matrix and load vector of fine cell f of an n x n mesh of
// the unit square (coefficient tile in the batch layout of one cell).
__global__ void fine_elements_2d_kernel(int n, int coef_kind, const double *coef, int rhs_kind, double rhs_value,
                                        double *Ae, double *Fe)
{
  const double h = 1.0 / n, gs = 0.5 / sqrt(3.0), jxw = 0.25 * h * h;
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < n * n; f += gridDim.x * blockDim.x)
    {
      double K[4][4];
      qg_element_2d(coef_kind, coef, f, h, h, K);
      for (int u = 0; u < 4; ++u)
        for (int v = 0; v < 4; ++v)
          Ae[(size_t)f * 16 + u * 4 + v] = K[u][v];
      const int fx = f % n, fy = f / n;
      double b[4] = {0, 0, 0, 0};
      for (int q = 0; q < 4; ++q)
        {
          const double xi = (q & 1) ? 0.5 + gs : 0.5 - gs, eta = (q & 2) ? 0.5 + gs : 0.5 - gs;
          double fv = rhs_value;
          if (rhs_kind == MSFEM_RHS_SINSIN)
            fv = sin(M_PI * (fx + xi) * h) * sin(M_PI * (fy + eta) * h);
          for (int v = 0; v < 4; ++v)
            b[v] += ((v & 1) ? xi : 1.0 - xi) * ((v & 2) ? eta : 1.0 - eta) * fv * jxw;
        }
      for (int v = 0; v < 4; ++v)
        Fe[(size_t)f * 4 + v] = b[v];
    }
}

} // namespace

hipError_t launch_fine_elements_2d(int n, int coef_kind, const double *coef, int rhs_kind, double rhs_value,
                                   double *Ae, double *Fe, hipStream_t st)
{
  int grid = (n * n + kFineThreads - 1) / kFineThreads;
  if (grid > 65535)
    grid = 65535;
  hipLaunchKernelGGL(fine_elements_2d_kernel, dim3(grid), dim3(kFineThreads), 0, st, n, coef_kind, coef, rhs_kind,
                     rhs_value, Ae, Fe);
  return hipGetLastError();
}

} // namespace msfem
