// Multigrid-preconditioned FP64 CG on structured stencil matrices (3^DIM entries per node): the
// coarse system of the MsFEM (the reference's AMG-preconditioned CG,
// include/base/diffusion_problem_ms.tpp:260-296) and the fine-scale Q1 system
// (include/base/diffusion_problem.tpp:243-279).
//
// The preconditioner is one V(2,2) cycle: levels n, ceil(n/2), ... down to 2 cells per side,
// bilinear/trilinear prolongation P, full weighting P^T, Galerkin operators A_{l+1} = P^T A_l P on
// the free nodes, damped Jacobi smoothing, the coarsest level's inverse.  With n odd the first
// coarse interval is one fine cell wide, so every size coarsens.  The first and not the last:
// sizes that stay odd (65, 33, 17, ...) keep that interval narrow on every level, and beside a
// Neumann side, which the last one can be, the point smoother loses it (65 cells per side: 108
// iterations there, 9 now); the first lies on a Dirichlet side in both kinds of boundary.
//
// Large levels run on many workgroups, a tile each: one kernel takes a level down (two sweeps
// from zero, the residual, its restriction), one up (prolongation, two sweeps), each reading
// its tile with a halo and doing the halo's part of the sweeps itself, so that a level costs two
// launches and no exchange.  The CG's vector updates ride on level 0's kernels (the residual
// update with the way down, the direction with the matrix product).  The small levels, whose
// matrices fit LDS, are one workgroup's V-cycle; a system that is small as a whole is solved by
// one launch.  A pass of one workgroup over a 129^2 level takes 40 us (the latency of its loads);
// a launch of all tiles takes 5.  What bounds it now is the chain of launches (4.5 us each empty).
//
// Measured, with one workgroup for the whole multigrid CG / Jacobi CG over many workgroups before:
// coarse systems of 128^2 cells 4.8 -> 1.0 ms (10 iterations), 64^2 with its build 13.3 -> 12.6,
// 16^3 with its build 29.5 -> 27.2; the 512^2 fine system 62.6 -> 3.0 ms with its assembly.
#include <algorithm>

#include "msfem_device.hpp"
#include "msfem_kernels.hpp"

namespace msfem {

namespace {

constexpr double kMgOmega = 0.7;
constexpr int kMgThreads = 256, kTailThreads = 1024;
constexpr int kTailLds = 20200;        // doubles of LDS for the small levels (161 600 of 163 840 bytes)
constexpr int kMgBlocks = 1024;        // most workgroups of a launch (and partial sums)

template <int DIM>
constexpr int mg_entries() { return DIM == 2 ? 9 : 27; }

template <int DIM>
constexpr int ipow(int b) { return DIM == 2 ? b * b : b * b * b; }

// State of the iteration in device memory (msfem_kernels.hpp: MgState).

__host__ __device__ constexpr int coarse_n(int n) { return (n + 1) / 2; }
// Fine position of coarse node I of a level above n fine cells.
__host__ __device__ constexpr int fine_of(int I, int n) { return n & 1 ? (I == 0 ? 0 : 2 * I - 1) : 2 * I; }
// Whether fine node i (0..n) lies between two coarse nodes (weight 1/2 each); the others are coarse nodes.
__host__ __device__ constexpr bool between(int i, int n) { return n & 1 ? !(i & 1) && i != 0 : i & 1; }
// The coarse node at fine node i, or the first of the two that i lies between.
__host__ __device__ constexpr int coarse_of(int i, int n) { return (n & 1) && !between(i, n) ? (i + 1) >> 1 : i >> 1; }

template <int DIM>
struct Grid {
  int n;
  __device__ int np() const { return n + 1; }
  __device__ bool inside(const int (&I)[3]) const
  {
    for (int k = 0; k < DIM; ++k)
      if (I[k] < 0 || I[k] > n)
        return false;
    return true;
  }
  __device__ int index(const int (&I)[3]) const { return I[0] + np() * (I[1] + (DIM == 3 ? np() * I[2] : 0)); }
  __device__ void coords(int node, int (&I)[3]) const
  {
    I[0] = node % np();
    const int q = node / np();
    I[1] = DIM == 2 ? q : q % np();
    I[2] = DIM == 2 ? 0 : q / np();
  }
};

// Sum over the workgroup in a fixed order, in every thread.
template <int NT>
__device__ __forceinline__ double wg_sum(double v, double *red)
{
  v = group_sum<kWave>(v);
  __syncthreads();
  if (threadIdx.x % kWave == 0)
    red[threadIdx.x / kWave] = v;
  __syncthreads();
  double s = 0;
  for (int w = 0; w < NT / kWave; ++w)
    s += red[w];
  return s;
}

// Sum of the partial sums of an earlier launch, the same in every workgroup.
template <int NT>
__device__ __forceinline__ double partials(const double *part, int n, double *red)
{
  double v = 0;
  for (int k = threadIdx.x; k < n; k += NT)
    v += part[k];
  return wg_sum<NT>(v, red);
}

// Entry t's neighbour offset along axis k.
__device__ __forceinline__ constexpr int off(int t, int k) { return k == 0 ? t % 3 - 1 : k == 1 ? t / 3 % 3 - 1 : t / 9 - 1; }

// ---- set-up ----------------------------------------------------------------------------------

// Level 0: x = Dirichlet values / 0, Jacobi diagonal (0 on constrained nodes), residual.
template <int DIM>
__global__ void __launch_bounds__(kMgThreads) mg_init_kernel(MgLayout g, const double *Kc, const double *Fc,
                                                             const unsigned char *cmask, const double *cval,
                                                             double rel_tol, int max_iter, double *w)
{
  constexpr int S = mg_entries<DIM>();
  Grid<DIM> G{g.n[0]};
  double *x = w + g.off_cx, *r = w + g.off_cr, *p = w + g.off_cp, *d = w + g.off_d[0];
  for (int n = blockIdx.x * kMgThreads + threadIdx.x; n < (int)g.nn[0]; n += gridDim.x * kMgThreads)
    {
      const bool con = cmask[n] != 0;
      double v = 0;
      int I[3];
      G.coords(n, I);
      for (int t = 0; t < S; ++t)
        {
          int J[3] = {I[0] + off(t, 0), I[1] + off(t, 1), DIM == 3 ? I[2] + off(t, 2) : 0};
          if (G.inside(J))
            {
              const int m = G.index(J);
              if (cmask[m])
                v += Kc[(size_t)n * S + t] * cval[m];
            }
        }
      x[n] = con ? cval[n] : 0.0;
      d[n] = con ? 0.0 : kMgOmega / Kc[(size_t)n * S + S / 2];
      r[n] = con ? 0.0 : Fc[n] - v;
      p[n] = 0.0;
    }
  if (blockIdx.x == 0 && threadIdx.x == 0)
    {
      MgState *st = (MgState *)(w + g.off_state);
      st->rel_tol = rel_tol;
      st->max_iter = max_iter;
      st->iters = st->done = st->converged = st->begun = 0;
    }
}

// Galerkin operator of level l >= 1 from level l - 1, and its Jacobi diagonal.  One thread per
// (coarse node, fine node of its support): each sums its fine row's part into a private stencil,
// the partial stencils of a coarse node are added in a fixed order.
template <int DIM>
constexpr int galerkin_nodes() { return DIM == 2 ? 28 : 9; } // coarse nodes per workgroup

template <int DIM>
__global__ void __launch_bounds__(galerkin_nodes<DIM>() * mg_entries<DIM>())
  mg_galerkin_kernel(MgLayout g, int l, const double *A0, double *w)
{
  constexpr int S = mg_entries<DIM>(), NPB = galerkin_nodes<DIM>();
  __shared__ double part[NPB][S][S];
  Grid<DIM> Gf{g.n[l - 1]}, Gc{g.n[l]};
  const double *Af = l == 1 ? A0 : w + g.off_A[l - 1], *df = w + g.off_d[l - 1];
  double *Ac = w + g.off_A[l], *dc = w + g.off_d[l];
  const int cn = threadIdx.x / S, o = threadIdx.x % S, c = blockIdx.x * NPB + cn, n = Gf.n;
  double acc[S];
#pragma unroll
  for (int t = 0; t < S; ++t)
    acc[t] = 0;
  bool con = true; // a coarse node is constrained when the fine node at its position is
  if (c < (int)g.nn[l])
    {
      int I[3], i[3] = {0, 0, 0};
      Gc.coords(c, I);
      double wi = 1;
      int at[3] = {0, 0, 0};
      for (int k = 0; k < DIM; ++k)
        {
          at[k] = fine_of(I[k], n);
          i[k] = at[k] + off(o, k);
          wi *= off(o, k) == 0 ? 1.0 : between(i[k], n) ? 0.5 : 0.0;
        }
      con = df[Gf.index(at)] == 0.0;
      if (!con && wi != 0.0 && Gf.inside(i) && df[Gf.index(i)] != 0.0)
        {
          const int fi = Gf.index(i);
          for (int t = 0; t < S; ++t)
            {
              int j[3] = {i[0] + off(t, 0), i[1] + off(t, 1), DIM == 3 ? i[2] + off(t, 2) : 0};
              if (!Gf.inside(j) || df[Gf.index(j)] == 0.0)
                continue;
              const double a = wi * Af[(size_t)fi * S + t];
              int nb = 0;
              for (int k = 0; k < DIM; ++k)
                nb += between(j[k], n);
              for (int comb = 0; comb < (1 << nb); ++comb)
                {
                  int J[3] = {0, 0, 0}, bit = 0, tt = 0, mul = 1, Jf[3] = {0, 0, 0};
                  double wj = 1;
                  for (int k = 0; k < DIM; ++k)
                    {
                      J[k] = coarse_of(j[k], n);
                      if (between(j[k], n))
                        {
                          J[k] += (comb >> bit++) & 1;
                          wj *= 0.5;
                        }
                      Jf[k] = fine_of(J[k], n);
                      tt += (J[k] - I[k] + 1) * mul;
                      mul *= 3;
                    }
                  if (df[Gf.index(Jf)] != 0.0)
                    acc[tt] += a * wj;
                }
            }
        }
    }
#pragma unroll
  for (int t = 0; t < S; ++t)
    part[cn][o][t] = acc[t];
  __syncthreads();
  if (c < (int)g.nn[l])
    {
      double v = 0;
      for (int k = 0; k < S; ++k)
        v += part[cn][k][o];
      Ac[(size_t)c * S + o] = v;
      if (o == S / 2)
        dc[c] = con ? 0.0 : kMgOmega / v;
    }
}

// ---- tiles --------------------------------------------------------------------------------------

// Coarse nodes per side of a tile (the fine side is twice that).
template <int DIM>
constexpr int tile_side() { return DIM == 2 ? 8 : 4; }

// Node `e` of a cube of side SIDE starting at grid position lo.
template <int DIM, int SIDE>
__device__ __forceinline__ void cube_node(int e, const int (&lo)[3], int (&I)[3])
{
  I[0] = lo[0] + e % SIDE;
  I[1] = lo[1] + e / SIDE % SIDE;
  I[2] = DIM == 3 ? lo[2] + e / (SIDE * SIDE) : 0;
}

// sum_t A[t] v(neighbour t), v in a cube of side SIDE with the row's own node at entry e
template <int DIM, int SIDE>
__device__ __forceinline__ double stencil(const double *A, const double *v, int e)
{
  double s = 0;
#pragma unroll
  for (int t = 0; t < mg_entries<DIM>(); ++t)
    s += A[t] * v[e + off(t, 0) + SIDE * off(t, 1) + (DIM == 3 ? SIDE * SIDE * off(t, 2) : 0)];
  return s;
}

// Entry of the cube of side TO (starting `d` before the cube of side FROM) of FROM's entry e.
template <int DIM, int FROM, int TO>
__device__ __forceinline__ int cube_in(int e, int d)
{
  const int x = e % FROM + d, y = e / FROM % FROM + d, z = DIM == 3 ? e / (FROM * FROM) + d : 0;
  return x + TO * (y + (DIM == 3 ? TO * z : 0));
}

// A level's way down: x2 after two sweeps from zero on b, and P^T of the residual as the next
// level's b.  Level 0: b is the CG residual, first updated (r -= alpha q, x += alpha p; partial
// sums of r.r), read from buffer `par` and written to the other.
template <int DIM>
__global__ void __launch_bounds__(kMgThreads) mg_down_kernel(MgLayout g, int l, int par, const double *A0, double *w)
{
  constexpr int S = mg_entries<DIM>(), TC = tile_side<DIM>(), TF = 2 * TC, NB = TF + 6, NT = TF + 4, NU = TF + 2;
  __shared__ double db[ipow<DIM>(NB)], dt[ipow<DIM>(NT)], uu[ipow<DIM>(NU)], red[kMgThreads / kWave];
  const MgState *st = (const MgState *)(w + g.off_state);
  if (st->done)
    return;
  Grid<DIM> Gf{g.n[l]}, Gc{g.n[l + 1]};
  const double *A = l == 0 ? A0 : w + g.off_A[l], *d = w + g.off_d[l];
  double *x2 = w + g.off_x[l], *bc = w + g.off_b[l + 1];
  const double *r = l == 0 ? w + (par ? g.off_r1 : g.off_cr) : w + g.off_b[l];
  double *rn = w + (par ? g.off_cr : g.off_r1), *cx = w + g.off_cx;
  const double *q = w + g.off_cq, *p = w + (par ? g.off_p1 : g.off_cp);
  const bool update = l == 0 && st->begun;
  double alpha = 0;
  if (update)
    alpha = st->rz[1 - par] / partials<kMgThreads>(w + g.off_part + 2 * kMgBlocks, st->parts_dir, red);
  const int tiles = Gc.n / TC + 1, nt = ipow<DIM>(tiles);
  double rr = 0;
  for (int tile = blockIdx.x; tile < nt; tile += gridDim.x)
    {
      const int T[3] = {tile % tiles, tile / tiles % tiles, DIM == 3 ? tile / (tiles * tiles) : 0};
      const int c0[3] = {TC * T[0], TC * T[1], TC * T[2]};
      const int lob[3] = {2 * c0[0] - 4, 2 * c0[1] - 4, 2 * c0[2] - 4}, lot[3] = {lob[0] + 1, lob[1] + 1, lob[2] + 1},
                lou[3] = {lob[0] + 2, lob[1] + 2, lob[2] + 2};
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NB); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NB>(e, lob, I);
          double v = 0;
          if (Gf.inside(I))
            {
              const int n = Gf.index(I);
              const double b = update ? r[n] - alpha * q[n] : r[n];
              v = d[n] * b;
            }
          db[e] = v;
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NT); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NT>(e, lot, I);
          double v = 0, b = 0;
          if (Gf.inside(I))
            {
              const int n = Gf.index(I);
              const double dn = d[n];
              if (dn != 0.0)
                {
                  b = update ? r[n] - alpha * q[n] : r[n];
                  b -= stencil<DIM, NB>(A + (size_t)n * S, db, cube_in<DIM, NT, NB>(e, 1));
                  v = dn * b;
                }
            }
          dt[e] = v; // D t1
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NU); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NU>(e, lou, I);
          double u = 0;
          if (Gf.inside(I))
            {
              const int n = Gf.index(I), et = cube_in<DIM, NU, NT>(e, 1);
              const double dn = d[n], x1 = db[cube_in<DIM, NU, NB>(e, 2)];
              if (dn != 0.0)
                u = dt[et] / dn - stencil<DIM, NT>(A + (size_t)n * S, dt, et);
              bool own = true;
              for (int k = 0; k < DIM; ++k)
                own = own && I[k] >= 2 * c0[k];
              if (own)
                {
                  x2[n] = x1 + dt[et];
                  if (l == 0)
                    {
                      const double b = update ? r[n] - alpha * q[n] : r[n];
                      rn[n] = b;
                      rr += b * b;
                      if (update)
                        cx[n] += alpha * p[n];
                    }
                }
            }
          uu[e] = u;
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(TC); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, TC>(e, c0, I);
          if (!Gc.inside(I))
            continue;
          double s = 0;
          int f[3] = {0, 0, 0};
          for (int k = 0; k < DIM; ++k)
            f[k] = fine_of(I[k], Gf.n);
          if (d[Gf.index(f)] != 0.0)
            for (int t = 0; t < S; ++t)
              {
                double wi = 1;
                int at = 0;
                for (int k = DIM - 1; k >= 0; --k)
                  {
                    const int i = f[k] + off(t, k);
                    wi *= off(t, k) == 0 ? 1.0 : between(i, Gf.n) && i > 0 && i < Gf.n + 1 ? 0.5 : 0.0;
                    at = at * NU + i - lou[k];
                  }
                if (wi != 0.0)
                  s += wi * uu[at];
              }
          bc[Gc.index(I)] = s;
        }
    }
  if (l == 0)
    {
      rr = wg_sum<kMgThreads>(rr, red);
      if (threadIdx.x == 0)
        w[g.off_part + blockIdx.x] = rr;
    }
}

// A level's way up: z = x2 + P z_{l+1}, then two sweeps.  Level 0 (b = the residual in buffer
// `par`'s successor): partial sums of r.z.
template <int DIM>
__global__ void __launch_bounds__(kMgThreads) mg_up_kernel(MgLayout g, int l, int par, const double *A0, double *w)
{
  constexpr int S = mg_entries<DIM>(), TF = 2 * tile_side<DIM>(), NX = TF + 4, NT = TF + 2;
  __shared__ double xx[ipow<DIM>(NX)], dt[ipow<DIM>(NT)], red[kMgThreads / kWave];
  const MgState *st = (const MgState *)(w + g.off_state);
  if (st->done)
    return;
  Grid<DIM> Gf{g.n[l]}, Gc{g.n[l + 1]};
  const double *A = l == 0 ? A0 : w + g.off_A[l], *d = w + g.off_d[l], *x2 = w + g.off_x[l], *zc = w + g.off_t[l + 1];
  const double *b = l == 0 ? w + (par ? g.off_cr : g.off_r1) : w + g.off_b[l];
  double *z = w + g.off_t[l];
  const int tiles = Gf.n / TF + 1, nt = ipow<DIM>(tiles);
  double rz = 0;
  for (int tile = blockIdx.x; tile < nt; tile += gridDim.x)
    {
      const int f0[3] = {TF * (tile % tiles), TF * (tile / tiles % tiles), DIM == 3 ? TF * (tile / (tiles * tiles)) : 0};
      const int lox[3] = {f0[0] - 2, f0[1] - 2, f0[2] - 2}, lot[3] = {f0[0] - 1, f0[1] - 1, f0[2] - 1};
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NX); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NX>(e, lox, I);
          double v = 0;
          if (Gf.inside(I) && d[Gf.index(I)] != 0.0)
            {
              v = x2[Gf.index(I)];
              int nb = 0;
              for (int k = 0; k < DIM; ++k)
                nb += between(I[k], Gf.n);
              double s = 0;
              for (int comb = 0; comb < (1 << nb); ++comb)
                {
                  int J[3] = {0, 0, 0}, bit = 0;
                  for (int k = 0; k < DIM; ++k)
                    {
                      J[k] = coarse_of(I[k], Gf.n);
                      if (between(I[k], Gf.n))
                        J[k] += (comb >> bit++) & 1;
                    }
                  s += zc[Gc.index(J)];
                }
              v += s / (1 << nb);
            }
          xx[e] = v;
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NT); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NT>(e, lot, I);
          double v = 0;
          if (Gf.inside(I))
            {
              const int n = Gf.index(I);
              const double dn = d[n];
              if (dn != 0.0)
                v = dn * (b[n] - stencil<DIM, NX>(A + (size_t)n * S, xx, cube_in<DIM, NT, NX>(e, 1)));
            }
          dt[e] = v;
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(TF); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, TF>(e, f0, I);
          if (!Gf.inside(I))
            continue;
          const int n = Gf.index(I), et = cube_in<DIM, TF, NT>(e, 1);
          const double dn = d[n];
          double v = 0;
          if (dn != 0.0)
            v = xx[cube_in<DIM, TF, NX>(e, 2)] + 2.0 * dt[et] - dn * stencil<DIM, NT>(A + (size_t)n * S, dt, et);
          z[n] = v;
          if (l == 0)
            rz += b[n] * v;
        }
    }
  if (l == 0)
    {
      rz = wg_sum<kMgThreads>(rz, red);
      if (threadIdx.x == 0)
        w[g.off_part + kMgBlocks + blockIdx.x] = rz;
    }
}

// p = z + beta p (buffer `par` to the other) and q = A p; partial sums of p.q.
template <int DIM>
__global__ void __launch_bounds__(kMgThreads) mg_direction_kernel(MgLayout g, int par, int parts_up, const double *A0, double *w)
{
  constexpr int S = mg_entries<DIM>(), TF = 2 * tile_side<DIM>(), NX = TF + 2;
  __shared__ double pp[ipow<DIM>(NX)], red[kMgThreads / kWave];
  MgState *st = (MgState *)(w + g.off_state);
  if (st->done)
    return;
  Grid<DIM> G{g.n[0]};
  const double *z = w + g.off_t[0], *p = w + (par ? g.off_p1 : g.off_cp), *d = w + g.off_d[0];
  double *pn = w + (par ? g.off_cp : g.off_p1), *q = w + g.off_cq;
  const double rz = partials<kMgThreads>(w + g.off_part + kMgBlocks, parts_up, red);
  const double beta = st->iters > 0 ? rz / st->rz[1 - par] : 0.0;
  const int tiles = G.n / TF + 1, nt = ipow<DIM>(tiles);
  double pq = 0;
  for (int tile = blockIdx.x; tile < nt; tile += gridDim.x)
    {
      const int f0[3] = {TF * (tile % tiles), TF * (tile / tiles % tiles), DIM == 3 ? TF * (tile / (tiles * tiles)) : 0};
      const int lo[3] = {f0[0] - 1, f0[1] - 1, f0[2] - 1};
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(NX); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, NX>(e, lo, I);
          double v = 0;
          if (G.inside(I))
            {
              const int n = G.index(I);
              v = beta != 0.0 ? z[n] + beta * p[n] : z[n];
            }
          pp[e] = v;
        }
      __syncthreads();
      for (int e = threadIdx.x; e < ipow<DIM>(TF); e += kMgThreads)
        {
          int I[3];
          cube_node<DIM, TF>(e, f0, I);
          if (!G.inside(I))
            continue;
          const int n = G.index(I), ep = cube_in<DIM, TF, NX>(e, 1);
          const double v = pp[ep];
          double s = 0;
          if (d[n] != 0.0)
            s = stencil<DIM, NX>(A0 + (size_t)n * S, pp, ep);
          pn[n] = v;
          q[n] = s;
          pq += v * s;
        }
    }
  pq = wg_sum<kMgThreads>(pq, red);
  if (threadIdx.x == 0)
    w[g.off_part + 2 * kMgBlocks + blockIdx.x] = pq;
  if (blockIdx.x == 0 && threadIdx.x == 0)
    {
      st->rz[par] = rz; // (the other slot is being read)
      st->parts_dir = gridDim.x;
    }
}

// ---- the small levels, one workgroup --------------------------------------------------------------

constexpr int kMaxCoarsest = 27; // nodes of the coarsest level (2 cells per side)

// Levels ls.. of the hierarchy in LDS and one V-cycle on them.  lv[l] = {n, nodes, place of the
// level's data in lds}: the matrix, then d, x, t, b; the inverse of the coarsest matrix follows
// (zero rows and columns on constrained nodes do no harm: their right-hand side is 0).
struct TailLevel {
  int n, nn, at;
};

template <int DIM>
struct Tail {
  static constexpr int S = mg_entries<DIM>();
  double *lds;
  const TailLevel *lv;
  int ls, L, at_inv;

  __device__ __forceinline__ double *A(int l) const { return lds + lv[l].at; }
  __device__ __forceinline__ double *vec(int l, int k) const { return lds + lv[l].at + (S + k) * lv[l].nn; }
  __device__ __forceinline__ double *d(int l) const { return vec(l, 0); }
  __device__ __forceinline__ double *x(int l) const { return vec(l, 1); }
  __device__ __forceinline__ double *t(int l) const { return vec(l, 2); }
  __device__ __forceinline__ double *b(int l) const { return vec(l, 3); }
  __device__ __forceinline__ double *inv() const { return lds + at_inv; }

  // the level table and the levels' matrices; lv_: LDS, kMgMaxLevels entries
  __device__ __forceinline__ Tail(const MgLayout &g, int first, double *lds_, TailLevel *lv_, const double *A0, const double *w)
    : lds(lds_), lv(lv_), ls(first), L(g.levels)
  {
    int at = 0;
    for (int l = first; l < L; ++l)
      {
        const int n = g.n[l], nn = (int)g.nn[l];
        if (threadIdx.x == 0)
          lv_[l] = {n, nn, at};
        const double *Ag = l == 0 ? A0 : w + g.off_A[l], *dg = w + g.off_d[l];
        for (int k = threadIdx.x; k < nn * S; k += kTailThreads)
          lds[at + k] = Ag[k];
        for (int k = threadIdx.x; k < nn; k += kTailThreads)
          lds[at + nn * S + k] = dg[k];
        at += nn * (S + 4);
      }
    at_inv = at;
    __syncthreads();
  }

  // The coarsest matrix on its free nodes, inverted in place (Gauss-Jordan, SPD) by one wave,
  // column c in lane c.
  __device__ __forceinline__ void invert() const
  {
    const int l = L - 1, nn = lv[l].nn;
    Grid<DIM> G{lv[l].n};
    double *M = inv();
    const double *dl = d(l), *Al = A(l);
    for (int e = threadIdx.x; e < nn * nn; e += kTailThreads)
      M[e] = e / nn == e % nn && dl[e / nn] == 0.0 ? 1.0 : 0.0;
    __syncthreads();
    for (int e = threadIdx.x; e < nn * S; e += kTailThreads)
      {
        int I[3];
        G.coords(e / S, I);
        int J[3] = {I[0] + off(e % S, 0), I[1] + off(e % S, 1), DIM == 3 ? I[2] + off(e % S, 2) : 0};
        if (G.inside(J) && dl[e / S] != 0.0 && dl[G.index(J)] != 0.0)
          M[e / S * nn + G.index(J)] = Al[e];
      }
    __syncthreads();
    if (threadIdx.x < kWave)
      {
        const int c = threadIdx.x < nn ? threadIdx.x : 0;
        const bool mine = threadIdx.x < nn;
        for (int k = 0; k < nn; ++k)
          {
            const double piv = 1.0 / M[k * nn + k];
            const double rowk = c == k ? piv : M[k * nn + c] * piv;
            for (int i = 0; i < nn; ++i)
              {
                const double f = M[i * nn + k], v = M[i * nn + c];
                wave_fence();
                if (mine)
                  M[i * nn + c] = i == k ? rowk : c == k ? -f * piv : v - f * rowk;
                wave_fence();
              }
          }
      }
    __syncthreads();
  }

  static __device__ __forceinline__ void wave_fence()
  {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // (A v)_n at a free node n at I
  __device__ __forceinline__ double apply(int l, const double *v, int n, const int (&I)[3]) const
  {
    const int m = lv[l].n, np = m + 1;
    const double *Al = A(l) + n * S;
    double s = 0;
#pragma unroll
    for (int q = 0; q < S; ++q)
      {
        const int J[3] = {I[0] + off(q, 0), I[1] + off(q, 1), DIM == 3 ? I[2] + off(q, 2) : 0};
        if (Grid<DIM>{m}.inside(J))
          s += Al[q] * v[n + off(q, 0) + np * (off(q, 1) + (DIM == 3 ? np * off(q, 2) : 0))];
      }
    return s;
  }

  // x[ls] = V(b[ls])
  __device__ __forceinline__ void cycle() const
  {
    for (int l = ls; l + 1 < L; ++l)
      {
        const int nn = lv[l].nn;
        Grid<DIM> Gf{lv[l].n}, Gc{lv[l + 1].n};
        double *xl = x(l), *tl = t(l), *bl = b(l);
        const double *dl = d(l), *dn = d(l + 1);
        for (int n = threadIdx.x; n < nn; n += kTailThreads)
          xl[n] = dl[n] * bl[n];
        __syncthreads();
        // second sweep, then the residual (each from the neighbours of the one before)
        for (int sweep = 0; sweep < 2; ++sweep)
          {
            for (int n = threadIdx.x; n < nn; n += kTailThreads)
              {
                int I[3];
                Gf.coords(n, I);
                const double r = dl[n] == 0.0 ? 0.0 : bl[n] - apply(l, xl, n, I);
                tl[n] = sweep ? r : dl[n] * r;
              }
            __syncthreads();
            if (sweep == 0)
              {
                for (int n = threadIdx.x; n < nn; n += kTailThreads)
                  xl[n] += tl[n];
                __syncthreads();
              }
          }
        for (int c = threadIdx.x; c < lv[l + 1].nn; c += kTailThreads)
          {
            double s = 0;
            if (dn[c] != 0.0)
              {
                int I[3];
                Gc.coords(c, I);
                for (int q = 0; q < S; ++q)
                  {
                    double wi = 1;
                    int f[3] = {0, 0, 0};
                    for (int k = 0; k < DIM; ++k)
                      {
                        f[k] = fine_of(I[k], Gf.n) + off(q, k);
                        wi *= off(q, k) == 0 ? 1.0 : between(f[k], Gf.n) ? 0.5 : 0.0;
                      }
                    if (wi != 0.0 && Gf.inside(f))
                      s += wi * tl[Gf.index(f)];
                  }
              }
            b(l + 1)[c] = s;
          }
        __syncthreads();
      }
    {
      const int l = L - 1, nn = lv[l].nn;
      if (threadIdx.x < nn)
        {
          double s = 0;
          for (int k = 0; k < nn; ++k)
            s += inv()[threadIdx.x * nn + k] * b(l)[k];
          x(l)[threadIdx.x] = d(l)[threadIdx.x] == 0.0 ? 0.0 : s;
        }
      __syncthreads();
    }
    for (int l = L - 2; l >= ls; --l)
      {
        const int nn = lv[l].nn;
        Grid<DIM> Gf{lv[l].n}, Gc{lv[l + 1].n};
        double *xl = x(l), *tl = t(l);
        const double *dl = d(l), *bl = b(l), *xc = x(l + 1);
        for (int n = threadIdx.x; n < nn; n += kTailThreads)
          if (dl[n] != 0.0)
            {
              int I[3], nb = 0;
              Gf.coords(n, I);
              for (int k = 0; k < DIM; ++k)
                nb += between(I[k], Gf.n);
              double s = 0;
              for (int comb = 0; comb < (1 << nb); ++comb)
                {
                  int J[3] = {0, 0, 0}, bit = 0;
                  for (int k = 0; k < DIM; ++k)
                    {
                      J[k] = coarse_of(I[k], Gf.n);
                      if (between(I[k], Gf.n))
                        J[k] += (comb >> bit++) & 1;
                    }
                  s += xc[Gc.index(J)];
                }
              xl[n] += s / (1 << nb);
            }
        __syncthreads();
        for (int sweep = 0; sweep < 2; ++sweep)
          {
            for (int n = threadIdx.x; n < nn; n += kTailThreads)
              {
                int I[3];
                Gf.coords(n, I);
                tl[n] = dl[n] == 0.0 ? 0.0 : dl[n] * (bl[n] - apply(l, xl, n, I));
              }
            __syncthreads();
            for (int n = threadIdx.x; n < nn; n += kTailThreads)
              xl[n] += tl[n];
            __syncthreads();
          }
      }
  }
};

// Test of the residual (partial sums in the scratch), then the V-cycle's small levels.
template <int DIM>
__global__ void __launch_bounds__(kTailThreads) mg_tail_kernel(MgLayout g, int ls, int parts, const double *A0, double *w)
{
  __shared__ double lds[kTailLds];
  __shared__ double red[kTailThreads / kWave];
  __shared__ TailLevel lv[kMgMaxLevels];
  MgState *st = (MgState *)(w + g.off_state);
  if (st->done)
    return;
  const double rn = sqrt(partials<kTailThreads>(w + g.off_part, parts, red));
  // (every thread has read the state before thread 0 changes it: the barriers in partials)
  const int begun = st->begun, iters = st->iters, max_iter = st->max_iter;
  const double tol = begun ? st->tol : st->rel_tol * rn;
  const int it = begun ? iters + 1 : 0;
  const bool conv = rn <= tol, stop = conv || it >= max_iter;
  __syncthreads();
  if (threadIdx.x == 0)
    {
      st->iters = it;
      st->tol = tol;
      st->rnorm = rn;
      st->begun = 1;
      st->converged = conv ? 1 : 0;
      st->done = stop ? 1 : 0;
    }
  if (stop)
    return;
  const Tail<DIM> tail(g, ls, lds, lv, A0, w);
  const int ni = lv[tail.L - 1].nn * lv[tail.L - 1].nn, nn = lv[ls].nn;
  double *saved = w + g.off_inv, *z = w + g.off_t[ls];
  const double *b = w + g.off_b[ls];
  if (!begun) // the first iteration leaves the inverse for the others
    tail.invert();
  for (int k = threadIdx.x; k < ni; k += kTailThreads)
    if (begun)
      tail.inv()[k] = saved[k];
    else
      saved[k] = tail.inv()[k];
  for (int n = threadIdx.x; n < nn; n += kTailThreads)
    tail.b(ls)[n] = b[n];
  __syncthreads();
  tail.cycle();
  for (int n = threadIdx.x; n < nn; n += kTailThreads)
    z[n] = tail.x(ls)[n];
}

// The whole iteration for a system whose level 0 fits LDS.
template <int DIM>
__global__ void __launch_bounds__(kTailThreads) mg_small_kernel(MgLayout g, const double *A0, double *u, int *iters, double *w)
{
  __shared__ double lds[kTailLds];
  __shared__ double red[kTailThreads / kWave];
  __shared__ TailLevel lv[kMgMaxLevels];
  MgState *st = (MgState *)(w + g.off_state);
  const int nn = (int)g.nn[0], max_iter = st->max_iter;
  const Tail<DIM> tail(g, 0, lds, lv, A0, w);
  Grid<DIM> G{g.n[0]};
  double *x = w + g.off_cx, *r = tail.b(0), *z = tail.x(0), *q = tail.t(0);
  double *p = tail.inv() + kMaxCoarsest * kMaxCoarsest;
  const double *d = tail.d(0);
  tail.invert();
  double s = 0;
  for (int n = threadIdx.x; n < nn; n += kTailThreads)
    {
      r[n] = (w + g.off_cr)[n];
      p[n] = 0;
      s += r[n] * r[n];
    }
  double rn = sqrt(wg_sum<kTailThreads>(s, red)), rz = 1;
  const double tol = st->rel_tol * rn;
  int it = 0;
  while (rn > tol && it < max_iter)
    {
      tail.cycle();
      s = 0;
      for (int n = threadIdx.x; n < nn; n += kTailThreads)
        s += r[n] * z[n];
      const double rzn = wg_sum<kTailThreads>(s, red), beta = it ? rzn / rz : 0.0;
      rz = rzn;
      for (int n = threadIdx.x; n < nn; n += kTailThreads)
        p[n] = z[n] + beta * p[n];
      __syncthreads();
      s = 0;
      for (int n = threadIdx.x; n < nn; n += kTailThreads)
        {
          int I[3];
          G.coords(n, I);
          q[n] = d[n] == 0.0 ? 0.0 : tail.apply(0, p, n, I);
          s += p[n] * q[n];
        }
      const double alpha = rz / wg_sum<kTailThreads>(s, red);
      s = 0;
      for (int n = threadIdx.x; n < nn; n += kTailThreads)
        {
          x[n] += alpha * p[n];
          r[n] -= alpha * q[n];
          s += r[n] * r[n];
        }
      rn = sqrt(wg_sum<kTailThreads>(s, red));
      ++it;
    }
  __syncthreads();
  for (int n = threadIdx.x; n < nn; n += kTailThreads)
    u[n] = x[n];
  if (threadIdx.x == 0)
    {
      *iters = it;
      st->iters = it;
      st->rnorm = rn;
      st->tol = tol;
      st->converged = rn <= tol ? 1 : 0;
      st->done = 1;
    }
}

int mg_blocks(long long items) { return (int)std::min<long long>(kMgBlocks, std::max<long long>(1, items)); }

template <int DIM>
hipError_t setup(const MgLayout &g, const double *Kc, const double *Fc, const unsigned char *cmask, const double *cval,
                 double rel_tol, int max_iter, double *w, hipStream_t st)
{
  hipLaunchKernelGGL(mg_init_kernel<DIM>, dim3(mg_blocks((g.nn[0] + kMgThreads - 1) / kMgThreads)), dim3(kMgThreads), 0,
                     st, g, Kc, Fc, cmask, cval, rel_tol, max_iter, w);
  for (int l = 1; l < g.levels; ++l)
    hipLaunchKernelGGL(mg_galerkin_kernel<DIM>, dim3((unsigned)((g.nn[l] + galerkin_nodes<DIM>() - 1) / galerkin_nodes<DIM>())),
                       dim3(galerkin_nodes<DIM>() * mg_entries<DIM>()), 0, st, g, l, Kc, w);
  return hipGetLastError();
}

template <int DIM>
int tiles_of(int n, int side)
{
  const int t = n / side + 1;
  return mg_blocks(ipow<DIM>(t));
}

template <int DIM>
hipError_t iterations(const MgLayout &g, int count, const double *Kc, double *w, hipStream_t st)
{
  constexpr int TC = tile_side<DIM>(), TF = 2 * TC;
  const int ls = g.tail;
  for (int k = 0; k < count; ++k)
    {
      const int par = k & 1;
      for (int l = 0; l < ls; ++l)
        hipLaunchKernelGGL(mg_down_kernel<DIM>, dim3(tiles_of<DIM>(g.n[l + 1], TC)), dim3(kMgThreads), 0, st, g, l, par, Kc, w);
      hipLaunchKernelGGL(mg_tail_kernel<DIM>, dim3(1), dim3(kTailThreads), 0, st, g, ls,
                         tiles_of<DIM>(g.n[1], TC), Kc, w);
      for (int l = ls - 1; l >= 0; --l)
        hipLaunchKernelGGL(mg_up_kernel<DIM>, dim3(tiles_of<DIM>(g.n[l], TF)), dim3(kMgThreads), 0, st, g, l, par, Kc, w);
      hipLaunchKernelGGL(mg_direction_kernel<DIM>, dim3(tiles_of<DIM>(g.n[0], TF)), dim3(kMgThreads), 0, st, g, par,
                         tiles_of<DIM>(g.n[0], TF), Kc, w);
    }
  return hipGetLastError();
}

} // namespace

MgLayout mg_layout(int dim, int nc)
{
  MgLayout g = {};
  auto nodes = [dim](long long n) { return dim == 2 ? (n + 1) * (n + 1) : (n + 1) * (n + 1) * (n + 1); };
  const long long S = dim == 2 ? 9 : 27;
  int L = 0;
  g.n[L++] = nc;
  while (g.n[L - 1] > 2)
    {
      g.n[L] = coarse_n(g.n[L - 1]);
      ++L;
    }
  g.levels = L;
  for (int l = 0; l < L; ++l)
    g.nn[l] = nodes(g.n[l]);
  // the small levels are those that fit LDS together: 32 cells per side and below in 2D, 6 in
  // 3D; a whole system needs one vector more
  auto lds = [&](int first, bool whole) {
    long long n = kMaxCoarsest * kMaxCoarsest + (whole ? g.nn[first] : 0);
    for (int l = first; l < L; ++l)
      n += g.nn[l] * (S + 4);
    return n;
  };
  g.tail = lds(0, true) <= kTailLds ? 0 : 1;
  while (g.tail > 0 && lds(g.tail, false) > kTailLds)
    ++g.tail;
  long long at = 0;
  auto take = [&at](long long n) {
    const long long o = at;
    at += (n + 1) & ~1LL;
    return o;
  };
  for (long long *o : {&g.off_cx, &g.off_cr, &g.off_r1, &g.off_cp, &g.off_p1, &g.off_cq})
    *o = take(g.nn[0]);
  for (int l = 0; l < L; ++l)
    {
      g.off_x[l] = take(g.nn[l]);
      g.off_t[l] = take(g.nn[l]);
      g.off_d[l] = take(g.nn[l]);
      g.off_b[l] = take(l > 0 ? g.nn[l] : 0);     // level 0's right-hand side is the CG residual
      g.off_A[l] = take(l > 0 ? g.nn[l] * S : 0); // level 0's operator is the caller's matrix
    }
  g.off_part = take(3 * kMgBlocks);
  g.off_inv = take(kMaxCoarsest * kMaxCoarsest);
  g.off_state = take((sizeof(MgState) + 7) / 8);
  g.total = at;
  return g;
}

hipError_t launch_mg_setup(int dim, const MgLayout &g, const double *Kc, const double *Fc, const unsigned char *cmask,
                           const double *cval, double rel_tol, int max_iter, double *w, hipStream_t st)
{
  return dim == 2 ? setup<2>(g, Kc, Fc, cmask, cval, rel_tol, max_iter, w, st)
                  : setup<3>(g, Kc, Fc, cmask, cval, rel_tol, max_iter, w, st);
}

hipError_t launch_mg_iterations(int dim, const MgLayout &g, int count, const double *Kc, double *w, hipStream_t st)
{
  return dim == 2 ? iterations<2>(g, count, Kc, w, st) : iterations<3>(g, count, Kc, w, st);
}

hipError_t launch_mg_small(const MgLayout &g, const double *Kc, double *u, int *iters, double *w, hipStream_t st)
{
  hipLaunchKernelGGL(mg_small_kernel<2>, dim3(1), dim3(kTailThreads), 0, st, g, Kc, u, iters, w);
  return hipGetLastError();
}

} // namespace msfem
