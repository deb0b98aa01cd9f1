// Direct local solves in 2D (9 <= nf <= 128): a batched FP64 nested dissection
// that factors every cell's fine matrix once for its four bases, in place of a
// Krylov iteration per basis.  It replaces the assembly and the four CG+SSOR
// solves of DiffusionProblemBasis<dim>::run()
// (include/base/diffusion_problem_basis.tpp:161-242, :295-317, :450-465).
//
// One cell, bottom up (direct_plan.hpp has the blocks):
//   direct_leaf_forward   one workgroup per 16 x 16 block: fine-cell matrices, patch
//                         centres, four leaves (a wave each), the block's own front
//   direct_front          one workgroup per larger block: the children's Schur
//                         complements, the front's elimination
// and top down:
//   direct_front_back     the values on the lines between the children
//   direct_leaf_back      the same for the 16 x 16 block, then the leaves, whose
//                         small factors are formed again instead of stored
// A front lives in the accumulators of v_mfma_f64_16x16x4 tiles and is eliminated
// four pivots at a time: the four columns go to LDS, every wave inverts the 4 x 4
// pivot block D, and each tile takes C_ij -= (A_i D^-1) A_j^T, one matrix
// instruction.  The operators W = A D^-1 are all the top-down pass needs:
// x_p = W_rhs,p - sum_r W_rp x_r, no triangular solve.  The right-hand sides are
// four more rows of the front, eliminated with it.
// direct_residual then measures the true FP64 residual of every basis against the
// caller's tolerance; cells that miss it are solved again for the residual and
// corrected (iterative refinement) by the same kernels, the others skip that pass.
#include <algorithm>

#include "direct_plan.hpp"
#include "msfem_device.hpp"
#include "msfem_kernels.hpp"

namespace msfem {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTpb = 256;
constexpr unsigned kNone = 255;

// Orders a wave's own LDS accesses (no other wave involved).
__device__ __forceinline__ void wave_lds_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup barrier for LDS exchanges: waits for LDS accesses only (__syncthreads would also
// wait for the W stores on their way to memory, which no wave of this launch reads).
__device__ __forceinline__ void lds_barrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Classes whose fine cells are formed where they are needed (box cells, coefficients per fine
// cell), and classes that read what direct_conductances stored (quadrature-point coefficients
// and quadrilaterals: ~500 instructions a fine cell, needed four times).
enum { kFormed = 0, kStored = 1 };

// The six conductances of fine cell (fx, fy) (vertices (0,0), (1,0), (0,1), (1,1)): pairs (0,1),
// (2,3), (0,2), (1,3), (0,3), (1,2); the element matrix is their graph Laplacian.
template <int CELLS>
__device__ __forceinline__ void fine_conductances(const DirectArgs &a, int slot, int cell, int fx, int fy, double (&c)[6])
{
  const int f = fy * a.nf + fx;
  if constexpr (CELLS == kFormed)
    {
      const double *cf = a.coef + a.coef_off[cell];
      const double *bx = a.box + 4 * (size_t)cell;
      const double rho = (bx[3] - bx[2]) / (bx[1] - bx[0]);
      const Cond4 k = a.coef_kind == 0 ? cond_scalar(cf[f], rho)
                                       : cond_tensor(cf[3 * (size_t)f], cf[3 * (size_t)f + 1], cf[3 * (size_t)f + 2], rho);
      c[0] = c[1] = k.ch;
      c[2] = c[3] = k.cv;
      c[4] = k.cd;
      c[5] = k.ca;
    }
  else
    {
      const size_t n = (size_t)a.nf * a.nf;
      const double *q = a.cond + slot * 6 * n + f;
#pragma unroll
      for (int k = 0; k < 6; ++k)
        c[k] = q[k * n];
    }
}

__global__ void __launch_bounds__(kTpb) direct_conductances(DirectArgs a)
{
  const int n = a.nf * a.nf, per = (n + kTpb - 1) / kTpb, slot = blockIdx.x / per;
  const int f = (blockIdx.x % per) * kTpb + threadIdx.x, cell = a.cells[slot];
  if (f >= n)
    return;
  const double *cf = a.coef + a.coef_off[cell];
  double K[4][4];
  if (a.verts)
    {
      const QuadMap m(a.verts + 8 * (size_t)cell);
      qg_element_quad(a.coef_kind, cf, f, a.nf, m, K, 0, 0.0, nullptr);
    }
  else
    {
      const double *bx = a.box + 4 * (size_t)cell;
      qg_element_2d(a.coef_kind, cf, f, (bx[1] - bx[0]) / a.nf, (bx[3] - bx[2]) / a.nf, K);
    }
  double *o = a.cond + (size_t)slot * 6 * n + f;
  o[0] = -K[0][1];
  o[n] = -K[2][3];
  o[2 * (size_t)n] = -K[0][2];
  o[3 * (size_t)n] = -K[1][3];
  o[4 * (size_t)n] = -K[0][3];
  o[5 * (size_t)n] = -K[1][2];
}

__device__ __forceinline__ constexpr int tri(int a, int b) { return a >= b ? a * (a + 1) / 2 + b : b * (b + 1) / 2 + a; }

// ---- front elimination -----------------------------------------------------------------

// -(column kk of the inverse of the leading nv x nv part of the SPD 4 x 4 block D), zero
// beyond: two 2 x 2 steps.  Every lane forms it for its kk; the pivot loop is bound by the
// instructions it issues, of which these are the largest part.
__device__ __forceinline__ void neg_inverse_column(const double *D, int nv, int kk, double (&z)[4])
{
  double a00 = D[0], a10 = D[4], a11 = D[5], a20 = D[8], a21 = D[9], a22 = D[10], a30 = D[12], a31 = D[13], a32 = D[14],
         a33 = D[15];
  double e0 = kk == 0 ? -1.0 : 0.0, e1 = kk == 1 ? -1.0 : 0.0, e2 = kk == 2 ? -1.0 : 0.0, e3 = kk == 3 ? -1.0 : 0.0;
  if (nv < 4) // the last pivots: rows beyond them stay
    {
      if (nv < 2)
        a10 = 0, a11 = 1, e1 = 0;
      if (nv < 3)
        a20 = 0, a21 = 0, a22 = 1, e2 = 0;
      a30 = 0, a31 = 0, a32 = 0, a33 = 1, e3 = 0;
    }
  const double r1 = reciprocal(__builtin_fma(-a10, a10, a00 * a11));
  const double p00 = a11 * r1, p10 = -a10 * r1, p11 = a00 * r1;
  const double u20 = a20 * p00 + a21 * p10, u21 = a20 * p10 + a21 * p11;
  const double u30 = a30 * p00 + a31 * p10, u31 = a30 * p10 + a31 * p11;
  const double s22 = a22 - (u20 * a20 + u21 * a21), s32 = a32 - (u30 * a20 + u31 * a21),
               s33 = a33 - (u30 * a30 + u31 * a31);
  const double r2 = reciprocal(__builtin_fma(-s32, s32, s22 * s33));
  const double y2 = (e2 - (u20 * e0 + u21 * e1)) * r2, y3 = (e3 - (u30 * e0 + u31 * e1)) * r2;
  z[2] = s33 * y2 - s32 * y3;
  z[3] = s22 * y3 - s32 * y2;
  z[0] = (p00 * e0 + p10 * e1) - (u20 * z[2] + u30 * z[3]);
  z[1] = (p10 * e0 + p11 * e1) - (u21 * z[2] + u31 * z[3]);
}

// Single-wave form: lower tiles (i, j) of a TILES x TILES front in acc, row by row, at most MAXE
// eliminated rows (the pivot loop is unrolled, so a step touches exactly the tiles it needs).
// P: LDS, 16 TILES x 4.  STORE: row r > p of W = A D^-1 at W[r (r + 1) / 2 + p].
template <int TILES, int MAXE, bool STORE>
__device__ __forceinline__ void eliminate_wave(d4 (&acc)[TILES * (TILES + 1) / 2], int ne, int m, double *P, double *W,
                                               int lane)
{
  const int l16 = lane & 15, kk = lane >> 4;
#pragma unroll
  for (int p0 = 0; p0 < MAXE; p0 += 4)
    if (p0 < ne)
      {
        const int jt = p0 >> 4, po = p0 & 15, nv = ne - p0 < 4 ? ne - p0 : 4;
        if (l16 >= po && l16 < po + 4)
#pragma unroll
          for (int i = jt; i < TILES; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              P[(16 * i + mfma_row(lane, v)) * 4 + l16 - po] = acc[i * (i + 1) / 2 + jt][v];
        wave_lds_fence();
        double dc[4], w[TILES], c[TILES];
        neg_inverse_column(P + 4 * p0, nv, kk, dc);
#pragma unroll
        for (int i = jt; i < TILES; ++i)
          {
            const double *q = P + (16 * i + l16) * 4;
            w[i] = (q[0] * dc[0] + q[1] * dc[1]) + (q[2] * dc[2] + q[3] * dc[3]);
            c[i] = P[(16 * i + l16) * 4 + kk];
          }
        if constexpr (STORE)
#pragma unroll
          for (int i = jt; i < TILES; ++i)
            {
              const int r = 16 * i + l16;
              if (r >= p0 + nv && r < m && kk < nv)
                W[r * (r + 1) / 2 + p0 + kk] = -w[i];
            }
#pragma unroll
        for (int i = jt; i < TILES; ++i)
          if (16 * i < m)
#pragma unroll
            for (int j = jt; j <= i; ++j)
              if (j > jt || po < 12 || nv < 4) // (a column of tiles with nothing left is done)
                acc[i * (i + 1) / 2 + j] =
                  __builtin_amdgcn_mfma_f64_16x16x4f64(w[i], c[j], acc[i * (i + 1) / 2 + j], 0, 0, 0);
        wave_lds_fence(); // P is written again
      }
}

// Sum of the two doubles at the byte offsets in the halves of k.
__device__ __forceinline__ double two(const double *pool, uint32_t k)
{
  return *(const double *)((const char *)pool + (k & 0xFFFF)) + *(const double *)((const char *)pool + (k >> 16));
}

// Lower tiles of a front of TILES tile rows dealt out to WR x WC waves, wave (wr, wc) holding
// tiles (WR a + wr, WC b + wc): each wave has its share of what is left after any pivot, and
// reads one operand per tile row and one per tile column instead of two per tile.
template <int TILES, int WR, int WC>
struct FrontTiles {
  static constexpr int A = (TILES + WR - 1) / WR, B = (TILES + WC - 1) / WC;
  d4 acc[A][B];
  int wr, wc;

  static constexpr bool any(int a, int b) { return WC * b <= WR * a + WR - 1; } // some wave has the tile
  __device__ bool mine(int a, int b, int tm) const
  {
    return WC * b + wc <= WR * a + wr && WR * a + wr < tm;
  }

  // Rows 0..ne-1 eliminated; P: LDS, two buffers of 16 TILES x 4.  Row r > p of W at W[r * ldw + p].
  __device__ __forceinline__ void eliminate(int ne, int m, double *P, double *W, int ldw, int lane)
  {
    constexpr int ROWS = 16 * (WR * A > WC * B ? WR * A : WC * B);
    const int l16 = lane & 15, kk = lane >> 4, tm = (m + 15) >> 4;
    for (int p0 = 0; p0 < ne; p0 += 4)
      {
        const int jt = p0 >> 4, po = p0 & 15, nv = ne - p0 < 4 ? ne - p0 : 4;
        double *Pb = P + ((p0 >> 2) & 1) * ROWS * 4;
        if (jt % WC == wc && l16 >= po && l16 < po + 4)
#pragma unroll
          for (int b = 0; b < B; ++b)
            if (b == jt / WC)
#pragma unroll
              for (int a = 0; a < A; ++a)
                if (any(a, b) && mine(a, b, tm))
#pragma unroll
                  for (int v = 0; v < 4; ++v)
                    Pb[(16 * (WR * a + wr) + mfma_row(lane, v)) * 4 + l16 - po] = acc[a][b][v];
        lds_barrier();
        double dc[4], w[A], c[B];
        neg_inverse_column(Pb + 4 * p0, nv, kk, dc);
#pragma unroll
        for (int a = 0; a < A; ++a)
          {
            const double *q = Pb + (16 * (WR * a + wr) + l16) * 4;
            w[a] = (q[0] * dc[0] + q[1] * dc[1]) + (q[2] * dc[2] + q[3] * dc[3]);
          }
#pragma unroll
        for (int b = 0; b < B; ++b)
          c[b] = Pb[(16 * (WC * b + wc) + l16) * 4 + kk];
        const int jn = (p0 + nv) >> 4; // first tile column with anything left
#pragma unroll
        for (int b = 0; b < B; ++b)
          if (WC * b + wc >= jn)
#pragma unroll
            for (int a = 0; a < A; ++a)
              if (any(a, b) && mine(a, b, tm))
                acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[a], c[b], acc[a][b], 0, 0, 0);
#pragma unroll
        for (int a = 0; a < A; ++a) // tile row's W: one wave of the row writes it
          {
            const int r = 16 * (WR * a + wr) + l16;
            if (a % WC == wc && r >= p0 + nv && r < m && kk < nv)
              W[(size_t)r * ldw + p0 + kk] = -w[a];
          }
      }
  }

  // Lower part of the Schur complement (rows and columns >= ne) to S.
  __device__ __forceinline__ void store_schur(int ne, int m, double *S, int ld, int lane) const
  {
    const int l16 = lane & 15, tm = (m + 15) >> 4;
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int b = 0; b < B; ++b)
        if (any(a, b) && mine(a, b, tm) && 16 * (WC * b + wc) + 15 >= ne)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            {
              const int r = 16 * (WR * a + wr) + mfma_row(lane, v) - ne, c = 16 * (WC * b + wc) + l16 - ne;
              if (c >= 0 && r >= c && r < m - ne)
                S[r * ld + c] = acc[a][b][v];
            }
  }

  // Entry (r, c) of every tile = the sources that the tables name in the leaves' Schur complements.
  __device__ __forceinline__ void assemble(const uint32_t *tables, const DirectFront &f, const double *pool, int tm, int lane)
  {
    const uint4 *tab = (const uint4 *)(tables + f.tab) + lane, *tabx = (const uint4 *)(tables + f.tabx) + lane;
    uint4 s[A][B];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int b = 0; b < B; ++b)
        if (any(a, b))
          {
            const int i = min(WR * a + wr, tm - 1), j = min(WC * b + wc, i); // (a tile that is not there: another)
            s[a][b] = tab[64 * (i * (i + 1) / 2 + j)];
          }
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int b = 0; b < B; ++b)
        if (any(a, b))
          {
            const uint4 &k = s[a][b];
            acc[a][b] = (d4){two(pool, k.x), two(pool, k.y), two(pool, k.z), two(pool, k.w)};
            const int q = (WR * a + wr) * (WR * a + wr + 1) / 2 + WC * b + wc;
            if (mine(a, b, tm) && ((f.extra >> q) & 1))
              {
                const uint4 x = tabx[64 * __builtin_popcount(f.extra & ((1u << q) - 1))];
                acc[a][b] += (d4){two(pool, x.x), two(pool, x.y), two(pool, x.z), two(pool, x.w)};
              }
          }
  }

  // Entry (r, c) of every tile = sum over the children that have both rows; child(k, ra, ca, ok):
  // its entry, 0 if not ok.  code: byte k of row r = its row in child k, 255 = none.  A tile
  // column's loads from a child are all on their way before the first is used (128-row fronts:
  // 352 -> 314 us for 4076 with this and without a branch around each load).
  template <typename Child>
  __device__ __forceinline__ void assemble(const uint32_t *code, const uint8_t *kids, int tm, int lane, Child child)
  {
    uint32_t rc[A][4];
    int ka[A];
#pragma unroll
    for (int a = 0; a < A; ++a)
      {
        ka[a] = WR * a + wr < tm ? kids[WR * a + wr] : 0;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          rc[a][v] = code[16 * (WR * a + wr) + mfma_row(lane, v)];
      }
#pragma unroll
    for (int b = 0; b < B; ++b)
      {
        const int kb = WC * b + wc < tm ? kids[WC * b + wc] : 0;
        const uint32_t cc = code[16 * (WC * b + wc) + (lane & 15)];
#pragma unroll
        for (int a = 0; a < A; ++a)
          if (any(a, b))
            acc[a][b] = (d4){0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if ((kb >> k) & 1)
            {
              const uint32_t ca = (cc >> (8 * k)) & 255;
              double t[A][4];
#pragma unroll
              for (int a = 0; a < A; ++a)
                if (any(a, b))
                  {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                      t[a][v] = 0;
                    if (mine(a, b, tm) && ((ka[a] >> k) & 1))
#pragma unroll
                      for (int v = 0; v < 4; ++v)
                        {
                          const uint32_t ra = (rc[a][v] >> (8 * k)) & 255;
                          t[a][v] = child(k, ra, ca, ra != kNone && ca != kNone);
                        }
                  }
#pragma unroll
              for (int a = 0; a < A; ++a)
                if (any(a, b))
#pragma unroll
                  for (int v = 0; v < 4; ++v)
                    acc[a][b][v] += t[a][v];
            }
      }
  }
};

// ---- leaves -------------------------------------------------------------------------------

// Place of fine cell (lx, ly) of leaf q in an array of fine cells: the padding puts the 32
// patches' reads (every second cell of every second row) on 32 different pairs of LDS banks.
constexpr int kElemRow = 12, kElemLeaf = 97, kElemCells = 4 * kElemLeaf;
__device__ __forceinline__ constexpr int elem_at(int q, int lx, int ly) { return q * kElemLeaf + ly * kElemRow + lx; }

// Fine-cell conductances of a <= 16 x 16 block into elem[6][kElemCells] (leaf q: children
// (q & 1, q >> 1)), thread per fine cell; zero beyond a leaf.
template <int CELLS>
__device__ __forceinline__ void block_conductances(const DirectArgs &a, int slot, int cell, const DirectFront &f, double *elem)
{
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63, lx = lane & 7, ly = lane >> 3;
  const DirectLeaf &lf = a.leaves[f.child[q]];
  double c[6] = {0, 0, 0, 0, 0, 0};
  if (lx < lf.w && ly < lf.h)
    fine_conductances<CELLS>(a, slot, cell, lf.x0 + lx, lf.y0 + ly, c);
#pragma unroll
  for (int k = 0; k < 6; ++k)
    elem[k * kElemCells + elem_at(q, lx, ly)] = c[k];
}

constexpr int kNp = 17, kNx = 20; // nodes per side of a block; row of its nodes' values (padded like the fine cells)

// One 2 x 2 patch of a leaf (lane: leaf lane >> 4, patch lane & 15: a wave has the 64 patches of
// a block): its 9-node matrix with the centre of a full patch eliminated, and one right-hand
// side, -sum_B S_Bc x(B) over the given values x (0 at the other nodes), plus the loads of the
// nodes it owns.  All four waves form the matrix, each for its own right-hand side.
// Then the pair's middle node: the partner patch is the neighbouring lane.
struct Patch {
  double S[45], v[9], inv; // inv: 1 / the centre's diagonal, 0 without a centre
  double s[9], invm;       // column of the pair's middle node; 1 / its diagonal, 0 without one
  bool valid, full;

  // elem: the leaf's fine cells; x: block nodes from the patch's first one; load(lx, ly): the
  // load of a node of the leaf
  template <typename Load>
  __device__ __forceinline__ void form(const DirectLeaf &lf, int px, int py, const double *elem, bool any_given,
                                       const double *x, bool loads, Load load)
  {
    valid = 2 * px < lf.w && 2 * py < lf.h;
    const double *e = elem + elem_at(0, 2 * px, 2 * py);
#pragma unroll
    for (int k = 0; k < 45; ++k)
      S[k] = 0;
#pragma unroll
    for (int cy = 0; cy < 2; ++cy)
#pragma unroll
      for (int cx = 0; cx < 2; ++cx)
        {
          const int n[4] = {cx + 3 * cy, cx + 1 + 3 * cy, cx + 3 * cy + 3, cx + 3 * cy + 4};
          constexpr int va[6] = {0, 2, 0, 1, 0, 1}, vb[6] = {1, 3, 2, 3, 3, 2};
#pragma unroll
          for (int k = 0; k < 6; ++k)
            {
              const double c = e[k * kElemCells + elem_at(0, cx, cy)];
              const int a = n[va[k]], b = n[vb[k]];
              S[tri(a, a)] += c;
              S[tri(b, b)] += c;
              S[tri(a, b)] -= c;
            }
        }
    full = 2 * px + 2 <= lf.w && 2 * py + 2 <= lf.h;
    inv = full ? reciprocal(S[tri(4, 4)]) : 0.0;
#pragma unroll
    for (int a = 0; a < 9; ++a)
      {
        const double s = a == 4 ? 0.0 : S[tri(a, 4)] * inv;
#pragma unroll
        for (int b = 0; b <= a; ++b)
          if (a != 4 && b != 4)
            S[tri(a, b)] -= s * S[tri(b, 4)];
      }
#pragma unroll
    for (int c = 0; c < 9; ++c)
      v[c] = 0;
    if (any_given)
#pragma unroll
      for (int b = 0; b < 9; ++b)
        {
          const double xb = x[b / 3 * kNx + b % 3];
#pragma unroll
          for (int c = 0; c < 9; ++c)
            v[c] -= S[tri(b, c)] * xb;
        }
    if (loads && valid)
      {
        // a node's load enters with the patch that has it at (0, 0), (1, 0), (0, 1) or (1, 1)
        const double rc = full ? load(2 * px + 1, 2 * py + 1) * inv : 0.0;
#pragma unroll
        for (int c = 0; c < 9; ++c)
          {
            if (c % 3 < 2 && c / 3 < 2 && !(c == 4 && full) && 2 * px + c % 3 < lf.w && 2 * py + c / 3 < lf.h)
              v[c] += load(2 * px + c % 3, 2 * py + c / 3);
            if (c != 4)
              v[c] -= S[tri(c, 4)] * rc;
          }
      }
  }

  static __device__ __forceinline__ double partner(double x) { return dpp_f64<0xB1>(x); } // quad_perm [1, 0, 3, 2]

  // The middle node of the pair (node 5 of the left patch, 3 of the right one): its column, the
  // right-hand side without it.
  __device__ __forceinline__ void middle(const DirectLeaf &lf, int px, int py)
  {
    const bool odd = px & 1, merged = 2 * (px | 1) < lf.w && 2 * py + 2 <= lf.h;
#pragma unroll
    for (int b = 0; b < 9; ++b)
      s[b] = b == 4 && full ? 0.0 : odd ? S[tri(b, 3)] : S[tri(b, 5)];
    const double d = odd ? s[3] : s[5];
    const double dm = d + partner(d);
    // the two nodes that the patches share (2 and 8 of the left one, 0 and 6 of the right one)
    // have both patches' part; what they alone take part in counts with the left patch
    const double s0 = odd ? s[0] : s[2], s1 = odd ? s[6] : s[8], t0 = s0 + partner(s0), t1 = s1 + partner(s1);
    s[0] = odd ? t0 : s[0];
    s[2] = odd ? s[2] : t0;
    s[6] = odd ? t1 : s[6];
    s[8] = odd ? s[8] : t1;
    invm = merged ? reciprocal(dm) : 0.0;
    const double ve = odd ? v[3] : v[5];
    const double q = (ve + partner(ve)) * invm;
#pragma unroll
    for (int b = 0; b < 9; ++b)
      v[b] -= (b == 0 || b == 6) && odd ? 0.0 : s[b] * q;
  }

  // to the leaf's pool: the matrix without the middle node (by one wave), right-hand side i
  __device__ __forceinline__ void store(double *pool, int p, int i, bool matrix) const
  {
    double *o = pool + p * kPatchDoubles;
    if (matrix && p == 0)
      pool[kLeafDoubles - 1] = 0.0;
    if (valid)
#pragma unroll
      for (int c = 0; c < 9; ++c)
        o[45 + i * 9 + c] = v[c];
    if (!matrix)
      return;
    const bool odd = p & 1;
    if (valid)
#pragma unroll
      for (int a = 0; a < 9; ++a)
        {
          const double t = s[a] * invm;
#pragma unroll
          for (int b = 0; b <= a; ++b)
            o[tri(a, b)] = S[tri(a, b)] - (a % 6 == 0 && b % 6 == 0 && odd ? 0.0 : t * s[b]);
        }
    // then the entries between the patches of the pair, in place of the eliminated nodes'
    double l[5], r[5];
#pragma unroll
    for (int k = 0; k < 5; ++k)
      {
        const double mine = kPairRight[k] == 5 && !full ? s[4] : s[kPairRight[k]], pr = partner(mine),
                     pl = partner(s[kPairLeft[k]]);
        l[k] = -(odd ? pl : s[kPairLeft[k]]) * invm;
        r[k] = odd ? mine : pr;
      }
    if (invm != 0.0 && !odd)
#pragma unroll
      for (int e = 0; e < kPairSlotsLeft; ++e)
        o[kPairSlot[e]] = l[e / 5] * r[e % 5];
    if (invm != 0.0 && odd)
#pragma unroll
      for (int e = kPairSlotsLeft; e < 25; ++e)
        o[kPairSlot[e]] = l[e / 5] * r[e % 5];
  }
};

// Tiles of a leaf's front from its patches.  load() asks for the tables, without a branch around
// any load, ahead of the work on the patches: waited for tile by tile they took 10k cycles.
template <int TILES>
struct LeafTables {
  static constexpr int N = TILES * (TILES + 1) / 2;
  uint4 s[N];

  __device__ __forceinline__ void load(const uint32_t *tables, const DirectLeafType &t, int lane)
  {
    const uint4 *tab = (const uint4 *)(tables + t.tab) + lane;
#pragma unroll
    for (int q = 0; q < N; ++q)
      s[q] = tab[64 * q];
  }

  __device__ __forceinline__ void front(const uint32_t *tables, const DirectLeafType &t, const double *pool, int lane,
                                        d4 (&acc)[N]) const
  {
    const uint4 *tabx = (const uint4 *)(tables + t.tabx) + lane;
    // entries of three or four patches are a patch corner's with itself and with the right-hand
    // sides: in the first two tile columns
#pragma unroll
    for (int q = 0; q < N; ++q)
      acc[q] = (d4){two(pool, s[q].x), two(pool, s[q].y), two(pool, s[q].z), two(pool, s[q].w)};
    uint4 x[TILES][2];
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int j = 0; j <= i && j < 2; ++j)
        x[i][j] = tabx[64 * (i * (i + 1) / 2 + j)];
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int j = 0; j <= i && j < 2; ++j)
        if ((t.extra >> (i * (i + 1) / 2 + j)) & 1)
          acc[i * (i + 1) / 2 + j] += (d4){two(pool, x[i][j].x), two(pool, x[i][j].y), two(pool, x[i][j].z), two(pool, x[i][j].w)};
  }
};

// Node (t along side s) of a block's outline, s = bottom, top, left, right.
__device__ __forceinline__ bool outline_node(const DirectFront &f, int s, int t, int &X, int &Y)
{
  X = s < 2 ? t : s == 2 ? 0 : f.w;
  Y = s == 0 ? 0 : s == 1 ? f.h : t;
  return X <= f.w && Y <= f.h;
}

constexpr int kLdsThird = 42 * 1280; // most LDS of a workgroup of which a CU holds three (160 KB in units of 1280 B)
constexpr int kBlockTiles = 7, kBlockElim = 29; // a 16 x 16 block's front: 29 + 64 + 4 rows
constexpr int kBlockRows = 16 * 8;              // (in tiles dealt out to 2 x 2 waves)
constexpr int kLeafWork = 16 * kLeafTiles * 4;  // pivot columns of a leaf

// Bottom-up pass of one block of the last front level: its four leaves, then its own front.
// Bound by latency and issue together: of the 31k cycles of a CU that a block takes, the LDS is
// busy for 15k, each SIMD's vector pipe for 11k and its matrix pipe for 5k.  Three workgroups a CU,
// which 10 tiles a leaf and 53 KB of LDS admit, cover each other's waits; what does not depend on
// the pivots is kept out of the pivot loops.  16304 blocks of 64^2 cells: 876 us, against 1250 with
// two workgroups a CU, leaf fronts of 69 rows and row codes in place of the tables.
template <int CELLS>
__global__ void __launch_bounds__(kTpb, 3) direct_leaf_forward(DirectArgs a)
{
  __shared__ double pool[4 * kLeafDoubles]; // fine cells; patches of the four leaves; their Schur complements
  __shared__ double work[kDirectRhs * kNp * kNx]; // given values of the block's nodes; pivot columns
  static_assert(6 * kElemCells <= 4 * kLeafDoubles && 4 * kLeafWork <= kDirectRhs * kNp * kNx &&
                  2 * kBlockRows * 4 <= kDirectRhs * kNp * kNx && kLeafLd * kLeafLd < kLeafDoubles &&
                  sizeof(pool) + sizeof(work) <= kLdsThird, "shared regions");
  const int nblk = a.n_fronts[a.depth - 1];
  const int slot = blockIdx.x / nblk;
  if (a.need && !a.need[slot])
    return;
  const int cell = a.cells[slot], lane = threadIdx.x & 63, np = a.nf + 1, nf = a.nf;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DirectFront &f = a.fronts[a.depth - 1][blockIdx.x % nblk];
  const int m = f.ne + f.nb + kDirectRhs;
  const double *R = a.loads ? a.loads + (size_t)slot * kDirectRhs * np * np : nullptr;
  const bool touches = !R && (f.x0 == 0 || f.y0 == 0 || f.x0 + f.w == nf || f.y0 + f.h == nf);
  if (touches)
    {
      for (int k = threadIdx.x; k < kDirectRhs * kNp * kNx; k += kTpb)
        work[k] = 0;
      __syncthreads();
      // the Dirichlet values on the block's outline
      const double *x = a.x_of(slot, cell);
      for (int k = threadIdx.x; k < kDirectRhs * 4 * kNp; k += kTpb)
        {
          const int i = k / (4 * kNp);
          int X, Y;
          if (outline_node(f, k / kNp & 3, k % kNp, X, Y) &&
              (f.x0 + X == 0 || f.y0 + Y == 0 || f.x0 + X == nf || f.y0 + Y == nf))
            work[(i * kNp + Y) * kNx + X] = x[((size_t)i * np + f.y0 + Y) * np + f.x0 + X];
        }
    }
  block_conductances<CELLS>(a, slot, cell, f, pool);
  const DirectLeafType &t = a.types[a.leaves[f.child[wave]].fwd];
  LeafTables<kLeafTiles> tab;
  __syncthreads();
  {
    const DirectLeaf &lf = a.leaves[f.child[lane >> 4]];
    const int px = lane & 3, py = (lane >> 2) & 3;
    Patch p;
    // (a patch beyond its leaf reads within work and pool and is not stored)
    const int X = min(lf.x0 - f.x0 + 2 * px, kNp - 3), Y = min(lf.y0 - f.y0 + 2 * py, kNp - 3);
    p.form(lf, px, py, pool + elem_at(lane >> 4, 0, 0), touches, work + (wave * kNp + Y) * kNx + X, R != nullptr,
           [&](int lx, int ly) { return R[((size_t)wave * np + lf.y0 + ly) * np + lf.x0 + lx]; });
    p.middle(lf, px, py);
    __syncthreads(); // fine cells and given values read by all
    p.store(pool + (lane >> 4) * kLeafDoubles, lane & 15, wave, wave == 0);
    tab.load(a.tables, t, lane);
  }
  __syncthreads();
  {
    double *mine = pool + wave * kLeafDoubles;
    const int ne = t.ne, lm = ne + t.nb + kDirectRhs, l16 = lane & 15;
    d4 acc[kLeafTiles * (kLeafTiles + 1) / 2];
    tab.front(a.tables, t, mine, lane, acc);
    wave_lds_fence();
    eliminate_wave<kLeafTiles, kLeafElim, false>(acc, ne, lm, work + wave * kLeafWork, nullptr, lane);
    // its Schur complement's lower part in place of its patches
#pragma unroll
    for (int i = 0; i < kLeafTiles; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j)
        if (16 * j + 15 >= ne && 16 * i < lm)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            {
              const int r = 16 * i + mfma_row(lane, v) - ne, c = 16 * j + l16 - ne;
              if (c >= 0 && (j < i || r >= c) && r < lm - ne)
                mine[r * kLeafLd + c] = acc[i * (i + 1) / 2 + j][v];
            }
    if (lane == 0)
      mine[kLeafDoubles - 1] = 0.0; // what absent entries read
  }
  __syncthreads();
  FrontTiles<kBlockTiles, 2, 2> front;
  front.wr = wave >> 1;
  front.wc = wave & 1;
  front.assemble(a.tables, f, pool, (m + 15) >> 4, lane);
  double *base = a.scratch + (size_t)slot * a.cell_doubles;
  front.eliminate(f.ne, m, work, base + f.w_off, f.ldw, lane);
  if (a.depth > 1)
    front.store_schur(f.ne, m, base + f.s_off, f.lds, lane);
}

// Elimination of one front of level a.level from its children's Schur complements.
template <int TILES, int WR, int WC>
__global__ void __launch_bounds__(64 * WR * WC, 2) direct_front(DirectArgs a)
{
  using Tiles = FrontTiles<TILES, WR, WC>;
  constexpr int NT = 64 * WR * WC, ROWS = 16 * (WR * Tiles::A > WC * Tiles::B ? WR * Tiles::A : WC * Tiles::B);
  __shared__ double P[2 * ROWS * 4];
  __shared__ uint32_t code[ROWS];
  const int nblk = a.n_fronts[a.level];
  const int slot = blockIdx.x / nblk;
  if (a.need && !a.need[slot])
    return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DirectFront &f = a.fronts[a.level][blockIdx.x % nblk];
  const int m = f.ne + f.nb + kDirectRhs;
  for (int r = threadIdx.x; r < ROWS; r += NT)
    code[r] = r < m ? a.tables[f.codes + r] : 0xFFFFFFFFu;
  __syncthreads();
  double *base = a.scratch + (size_t)slot * a.cell_doubles;
  const double *S[4];
  int ld[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    {
      const DirectFront &c = a.fronts[a.level + 1][f.child[k]];
      S[k] = base + c.s_off;
      ld[k] = c.lds;
    }
  Tiles front;
  front.wr = wave / WC;
  front.wc = wave % WC;
  front.assemble(code, f.kids, (m + 15) >> 4, lane, [&](int k, uint32_t ra, uint32_t ca, bool ok) {
    // a child keeps the rows in this order: its lower part.  (No branch around the load, which
    // would be waited for before the next.)
    const double v = S[k][ok ? max(ra, ca) * ld[k] + min(ra, ca) : 0];
    return ok ? v : 0.0;
  });
  front.eliminate(f.ne, m, P, base + f.w_off, f.ldw, lane);
  if (a.level > 0)
    front.store_schur(f.ne, m, base + f.s_off, f.lds, lane);
}

// Rows ne-1..0 of the top-down pass of a front of at most MAXE <= 64 eliminated rows, lane p
// holding row p: y = its four right-hand sides less the outline's part, w[r] = W(r, p).
template <int MAXE>
__device__ __forceinline__ void back_rows(double (&w)[MAXE], int ne, int lane, double (&y)[kDirectRhs])
{
#pragma unroll
  for (int r = 0; r < MAXE; ++r)
    w[r] = (lane >> 2) < (r >> 2) ? w[r] : 0.0; // (a row's own pivot block: in W already)
#pragma unroll
  for (int r = MAXE - 1; r > 0; --r)
    if (r < ne)
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        y[i] -= w[r] * readlane_f64(y[i], r);
}

// Values of a larger front's eliminated nodes: one wave, lane l holds rows l, l + 64, ...
// xo(i, r): value of outline row r; put(i, r, x): stores one.
template <int Q, typename Xo, typename Put>
__device__ __forceinline__ void back_substitute(const double *W, int ldw, int ne, int nb, int lane, Xo xo, Put put)
{
  double y[Q][kDirectRhs];
#pragma unroll
  for (int q = 0; q < Q; ++q)
    {
      const int p = lane + 64 * q;
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        y[q][i] = p < ne ? W[(size_t)(ne + nb + i) * ldw + p] : 0.0;
    }
#pragma unroll 8
  for (int r = ne; r < ne + nb; ++r)
    {
      double x[kDirectRhs];
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        x[i] = xo(i, r - ne);
#pragma unroll
      for (int q = 0; q < Q; ++q)
        {
          const double w = lane + 64 * q < ne ? W[(size_t)r * ldw + lane + 64 * q] : 0.0;
#pragma unroll
          for (int i = 0; i < kDirectRhs; ++i)
            y[q][i] -= w * x[i];
        }
    }
#pragma unroll
  for (int qr = Q - 1; qr >= 0; --qr)
    {
      const int top = ne - 64 * qr < 64 ? ne - 64 * qr : 64;
#pragma unroll 8
      for (int rr = top - 1; rr >= 0; --rr)
        {
          const int r = 64 * qr + rr;
          double x[kDirectRhs];
#pragma unroll
          for (int i = 0; i < kDirectRhs; ++i)
            x[i] = readlane_f64(y[qr][i], rr);
#pragma unroll
          for (int q = 0; q <= qr; ++q)
            {
              const int p = lane + 64 * q;
              const double w = (p >> 2) < (r >> 2) ? W[(size_t)r * ldw + p] : 0.0;
#pragma unroll
              for (int i = 0; i < kDirectRhs; ++i)
                y[q][i] -= w * x[i];
            }
        }
    }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (lane + 64 * q < ne)
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        put(i, lane + 64 * q, y[q][i]);
}

// Top-down pass of one front of level a.level.
template <int Q>
__global__ void __launch_bounds__(64) direct_front_back(DirectArgs a)
{
  __shared__ double xs[256 * kDirectRhs];
  const int nblk = a.n_fronts[a.level];
  const int slot = blockIdx.x / nblk;
  if (a.need && !a.need[slot])
    return;
  const int lane = threadIdx.x, np = a.nf + 1;
  const DirectFront &f = a.fronts[a.level][blockIdx.x % nblk];
  double *x = a.x_of(slot, a.cells[slot]);
  const uint32_t *nodes = a.tables + f.nodes;
  for (int r = lane; r < f.nb; r += 64)
#pragma unroll
    for (int i = 0; i < kDirectRhs; ++i)
      xs[r * kDirectRhs + i] = x[(size_t)i * np * np + nodes[f.ne + r]];
  __syncthreads();
  back_substitute<Q>(
    a.scratch + (size_t)slot * a.cell_doubles + f.w_off, f.ldw, f.ne, f.nb, lane,
    [&](int i, int r) { return xs[r * kDirectRhs + i]; },
    [&](int i, int r, double v) { x[(size_t)i * np * np + nodes[r]] = v; });
}

// Top-down pass of one block of the last front level: its own lines, its leaves, the patch
// centres.  The leaves are solved with their whole outline given: 29 rows instead of the 61 of
// the bottom-up front, so forming them again costs less than storing their W.  Bound by the LDS
// (10k of the 17k cycles a block); 16304 blocks: 432 us, against 812 with two workgroups a CU, each
// of the block's rows loaded behind a branch and 2 x 2 patches alone eliminated in closed form.
template <int CELLS>
__global__ void __launch_bounds__(kTpb, 3) direct_leaf_back(DirectArgs a)
{
  constexpr int NP = kNp, NX = kNx;
  __shared__ double X[kDirectRhs * NP * NX]; // the block's node values, 0 where not known yet
  __shared__ double pool[4 * kLeafDoubles];  // fine cells, the outline's part of the block's lines; patches; each
                                             // leaf's W and pivot columns
  __shared__ int at[96];                     // place in X of every row (<= 93) of the block's front
  constexpr int kLeafW = (kLeafElim + kDirectRhs) * (kLeafElim + kDirectRhs + 1) / 2;
  double *work = pool + 6 * kElemCells;
  static_assert(6 * kElemCells + 8 * kDirectRhs * 32 <= 4 * kLeafDoubles &&
                  kLeafW + 16 * kLeafBackTiles * 4 <= kLeafDoubles &&
                  sizeof(X) + sizeof(pool) + sizeof(at) <= kLdsThird, "shared regions");
  const int nblk = a.n_fronts[a.depth - 1];
  const int slot = blockIdx.x / nblk;
  if (a.need && !a.need[slot])
    return;
  const int cell = a.cells[slot], lane = threadIdx.x & 63, np = a.nf + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DirectFront &f = a.fronts[a.depth - 1][blockIdx.x % nblk];
  double *x = a.x_of(slot, cell);
  const double *R = a.loads ? a.loads + (size_t)slot * kDirectRhs * np * np : nullptr;
  const double *W = a.scratch + (size_t)slot * a.cell_doubles + f.w_off;
  // Everything this launch reads is asked for here, without a branch around a load (places beyond
  // a row or a side read a neighbour's and drop it): a load waited for where it is used costs
  // ~1000 cycles, and the block's lines alone take 29 of them one after the other.
  // The outline's part of the block's lines: thread (p, g) takes row p and outline rows g, g + 8, ...
  const int p = threadIdx.x & 31, g = threadIdx.x >> 5, pw = min(p, f.ldw - 1);
  double wo[8], wl[kBlockElim], wb[kDirectRhs], xo[2];
  int xat[2];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    wo[k] = W[(size_t)min(f.ne + g + 8 * k, f.ne + f.nb) * f.ldw + pw];
  if (wave == 0)
    {
#pragma unroll
      for (int r = 0; r < kBlockElim; ++r)
        wl[r] = W[(size_t)min(r, f.ne) * f.ldw + pw];
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        wb[i] = W[(size_t)(f.ne + f.nb + i) * f.ldw + pw];
    }
#pragma unroll
  for (int k = 0; k < 2; ++k)
    {
      const int e = min((int)threadIdx.x + k * kTpb, kDirectRhs * 4 * NP - 1), i = e / (4 * NP);
      int X0, Y0;
      const bool ok = outline_node(f, e / NP & 3, e % NP, X0, Y0);
      X0 = min(X0, f.w), Y0 = min(Y0, f.h);
      xo[k] = x[((size_t)i * np + f.y0 + Y0) * np + f.x0 + X0];
      xat[k] = ok ? (i * NP + Y0) * NX + X0 : -1;
    }
  const int node = a.tables[f.nodes + min((int)threadIdx.x, f.ne + f.nb - 1)];
  const DirectLeafType &t = a.types[a.leaves[f.child[wave]].back];
  LeafTables<kLeafBackTiles> tab;
  tab.load(a.tables, t, lane);
  for (int k = threadIdx.x; k < kDirectRhs * NP * NX; k += kTpb)
    X[k] = 0;
  block_conductances<CELLS>(a, slot, cell, f, pool);
  if (threadIdx.x < f.ne + f.nb)
    at[threadIdx.x] = (node / np - f.y0) * NX + node % np - f.x0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (xat[k] >= 0)
      X[xat[k]] = xo[k];
  __syncthreads();
  {
    double s[kDirectRhs] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (g + 8 * k < f.nb)
        {
          const int o = at[f.ne + g + 8 * k];
#pragma unroll
          for (int i = 0; i < kDirectRhs; ++i)
            s[i] += wo[k] * X[i * NP * NX + o];
        }
#pragma unroll
    for (int i = 0; i < kDirectRhs; ++i)
      work[(g * kDirectRhs + i) * 32 + p] = s[i];
  }
  __syncthreads();
  if (wave == 0)
    {
      double y[kDirectRhs];
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        {
          double s = 0;
#pragma unroll
          for (int k = 0; k < 8; ++k)
            s += work[(k * kDirectRhs + i) * 32 + (lane & 31)];
          y[i] = lane < f.ne ? wb[i] - s : 0.0;
        }
      back_rows<kBlockElim>(wl, f.ne, lane, y);
      if (lane < f.ne)
#pragma unroll
        for (int i = 0; i < kDirectRhs; ++i)
          X[i * NP * NX + at[lane]] = y[i];
    }
  __syncthreads();
  double cc[9], cm[9], invm; // what the nodes eliminated in closed form need
  {
    const DirectLeaf &lf = a.leaves[f.child[lane >> 4]];
    const int px = lane & 3, py = (lane >> 2) & 3;
    const int X0 = min(lf.x0 - f.x0 + 2 * px, NP - 3), Y0 = min(lf.y0 - f.y0 + 2 * py, NP - 3);
    Patch q;
    q.form(lf, px, py, pool + elem_at(lane >> 4, 0, 0), true, X + (wave * NP + Y0) * NX + X0, R != nullptr,
           [&](int lx, int ly) { return R[((size_t)wave * np + lf.y0 + ly) * np + lf.x0 + lx]; });
#pragma unroll
    for (int k = 0; k < 9; ++k)
      cc[k] = k == 4 ? q.inv : q.S[tri(k, 4)];
    q.middle(lf, px, py);
#pragma unroll
    for (int k = 0; k < 9; ++k)
      cm[k] = k % 6 == 0 && (px & 1) ? 0.0 : q.s[k]; // (shared nodes: in the left patch's sum)
    invm = q.invm;
    __syncthreads(); // fine cells read by all
    q.store(pool + (lane >> 4) * kLeafDoubles, lane & 15, wave, wave == 0);
  }
  __syncthreads();
  {
    const DirectLeaf &lf = a.leaves[f.child[wave]];
    double *mine = pool + wave * kLeafDoubles;
    const int lm = t.ne + kDirectRhs;
    d4 acc[kLeafBackTiles * (kLeafBackTiles + 1) / 2];
    tab.front(a.tables, t, mine, lane, acc);
    wave_lds_fence();
    eliminate_wave<kLeafBackTiles, kLeafElim, true>(acc, t.ne, lm, mine + kLeafW, mine, lane);
    double y[kDirectRhs];
#pragma unroll
    for (int i = 0; i < kDirectRhs; ++i)
      y[i] = lane < t.ne ? mine[(t.ne + i) * (t.ne + i + 1) / 2 + lane] : 0.0;
    double w[kLeafElim];
#pragma unroll
    for (int r = 0; r < kLeafElim; ++r)
      w[r] = mine[r * (r + 1) / 2 + min(lane, r)];
    back_rows<kLeafElim>(w, t.ne, lane, y);
    if (lane < t.ne)
      {
        const uint32_t xy = a.tables[t.nodes + lane];
        const int o = (lf.y0 - f.y0 + (int)(xy >> 8)) * NX + lf.x0 - f.x0 + (int)(xy & 255);
#pragma unroll
        for (int i = 0; i < kDirectRhs; ++i)
          X[i * NP * NX + o] = y[i];
      }
  }
  __syncthreads();
  {
    // middle nodes of the pairs, then patch centres: thread = (patch, basis)
    const DirectLeaf &lf = a.leaves[f.child[lane >> 4]];
    const int px = lane & 3, py = (lane >> 2) & 3;
    const bool odd = px & 1, centre = 2 * px + 2 <= lf.w && 2 * py + 2 <= lf.h;
    const int X0 = min(lf.x0 - f.x0 + 2 * px, NP - 3), Y0 = min(lf.y0 - f.y0 + 2 * py, NP - 3);
    double *o = X + (wave * NP + Y0) * NX + X0;
    const double *Rc = R ? R + ((size_t)wave * np + f.y0 + Y0 + 1) * np + f.x0 + X0 + 1 : nullptr; // the centre's load
    const double rc = centre && R ? *Rc : 0.0;
    double s = invm != 0.0 && R && !odd ? Rc[1] : 0.0; // the middle node's
    if (centre)
      s -= (odd ? cc[3] : cc[5]) * cc[4] * rc;
#pragma unroll
    for (int k = 0; k < 9; ++k)
      s -= (k == (odd ? 3 : 5) ? 0.0 : cm[k]) * o[k / 3 * NX + k % 3];
    s = (s + Patch::partner(s)) * invm;
    if (invm != 0.0 && !odd)
      o[NX + 2] = s;
    wave_lds_fence();
    if (centre)
      {
        s = rc;
#pragma unroll
        for (int k = 0; k < 9; ++k)
          if (k != 4)
            s -= cc[k] * o[k / 3 * NX + k % 3];
        o[NX + 1] = s * cc[4];
      }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kDirectRhs * 16 * 16; k += kTpb)
    {
      const int i = k >> 8, X0 = k & 15, Y0 = (k >> 4) & 15;
      if (X0 > 0 && Y0 > 0 && X0 < f.w && Y0 < f.h)
        x[((size_t)i * np + f.y0 + Y0) * np + f.x0 + X0] = X[(i * NP + Y0) * NX + X0];
    }
}

// ---- residuals --------------------------------------------------------------------------------

// A cell's interior nodes in tasks of a wave: 63 node columns x kStripRows node rows.
constexpr int kStripRows = 16;
__host__ __device__ constexpr int sweep_segs(int nf) { return (nf - 1 + 62) / 63; }
__host__ __device__ constexpr int sweep_tasks(int nf)
{
  return sweep_segs(nf) * ((nf - 1 + kStripRows - 1) / kStripRows);
}

// Residuals r = -(K x)_I of the four bases at the nodes of task `task`: the wave sweeps the
// fine-cell rows, a lane per fine-cell column, and passes the right-hand nodes' part to the next
// lane, so a fine cell is formed once per task.  value(i, X, Y): nodal value; emit(i, X, Y, r).
template <int CELLS, typename Value, typename Emit>
__device__ __forceinline__ void sweep(const DirectArgs &a, int slot, int cell, int task, Value value, Emit emit)
{
  const int lane = threadIdx.x & 63, nf = a.nf, segs = sweep_segs(nf);
  const int X = 63 * (task % segs) + lane, Y0 = 1 + kStripRows * (task / segs), Y1 = min(Y0 + kStripRows, nf);
  const bool cellok = X < nf;
  double b0[kDirectRhs], b1[kDirectRhs], up[kDirectRhs], upr[kDirectRhs];
#pragma unroll
  for (int i = 0; i < kDirectRhs; ++i)
    {
      b0[i] = cellok ? value(i, X, Y0 - 1) : 0.0;
      b1[i] = cellok ? value(i, X + 1, Y0 - 1) : 0.0;
      up[i] = upr[i] = 0;
    }
#pragma unroll 2
  for (int cy = Y0 - 1; cy < Y1; ++cy)
    {
      double c[6] = {0, 0, 0, 0, 0, 0}, t0[kDirectRhs], t1[kDirectRhs];
      if (cellok)
        fine_conductances<CELLS>(a, slot, cell, X, cy, c);
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        {
          t0[i] = cellok ? value(i, X, cy + 1) : 0.0;
          t1[i] = cellok ? value(i, X + 1, cy + 1) : 0.0;
        }
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        {
          const double e01 = c[0] * (b0[i] - b1[i]), e23 = c[1] * (t0[i] - t1[i]), e02 = c[2] * (b0[i] - t0[i]),
                       e13 = c[3] * (b1[i] - t1[i]), e03 = c[4] * (b0[i] - t1[i]), e12 = c[5] * (b1[i] - t0[i]);
          const double right = upr[i] + ((e13 - e01) + e12);
          const double r = -((up[i] + ((e01 + e02) + e03)) + __shfl_up(right, 1));
          if (cy >= Y0 && lane > 0 && cellok)
            emit(i, X, cy, r);
          up[i] = (e23 - e02) - e12;
          upr[i] = -((e23 + e13) + e03);
          b0[i] = t0[i];
          b1[i] = t1[i];
        }
    }
}

// Before the solve: boundary values of box cells and, per task, the sums of squares of b = K_IB g
// (a.part[slot][task][0..3]) and of the Q1 interpolant's residual ([4..7]).
template <int CELLS>
__global__ void __launch_bounds__(kTpb) direct_start(DirectArgs a)
{
  const int tasks = sweep_tasks(a.nf), wgs = (tasks + 3) / 4, slot = blockIdx.x / wgs, cell = a.cells[slot];
  const int task = (blockIdx.x % wgs) * 4 + (threadIdx.x >> 6), nf = a.nf, np = nf + 1;
  double *x = a.bases + a.bas_off[cell];
  const bool boxes = !a.verts;
  if (boxes && blockIdx.x % wgs == 0)
    for (int k = threadIdx.x; k < 4 * nf * kDirectRhs; k += kTpb)
      {
        const int i = k / (4 * nf), e = k % (4 * nf), s = e / nf, t = e % nf;
        const int X = s == 0 ? t : s == 1 ? nf : s == 2 ? nf - t : 0, Y = s == 0 ? 0 : s == 1 ? t : s == 2 ? nf : nf - t;
        x[((size_t)i * np + Y) * np + X] = nodal_q1(i, 2, X, Y, 0, nf);
      }
  if (task >= tasks)
    return;
  double sb[kDirectRhs] = {0, 0, 0, 0}, sq[kDirectRhs] = {0, 0, 0, 0};
  const double inv = 1.0 / nf;
  auto q1 = [&](int i, int X, int Y) { // the box cell's nodal functions
    const double tx = X * inv, ty = Y * inv;
    return ((i & 1) ? tx : 1.0 - tx) * ((i & 2) ? ty : 1.0 - ty);
  };
  if (!a.ptol)
    sweep<CELLS>(
      a, slot, cell, task,
      [&](int i, int X, int Y) {
        const bool edge = X == 0 || Y == 0 || X == nf || Y == nf;
        return !edge ? 0.0 : boxes ? q1(i, X, Y) : x[((size_t)i * np + Y) * np + X];
      },
      [&](int i, int, int, double r) { sb[i] += r * r; });
  if (boxes && a.q1_start)
    sweep<CELLS>(a, slot, cell, task, q1, [&](int i, int, int, double r) { sq[i] += r * r; });
#pragma unroll
  for (int i = 0; i < kDirectRhs; ++i)
    {
      const double tb = group_sum_dpp<64>(sb[i]), tq = group_sum_dpp<64>(sq[i]);
      if ((threadIdx.x & 63) == 0)
        {
          a.part[((size_t)slot * tasks + task) * 12 + i] = tb;
          a.part[((size_t)slot * tasks + task) * 12 + 4 + i] = tq;
        }
    }
}

// After a pass: sums of squares of the true residuals per task (a.part[..][8..11]); the second
// time of x + correction, for the cells that were corrected.
template <int CELLS>
__global__ void __launch_bounds__(kTpb) direct_residual(DirectArgs a)
{
  const int tasks = sweep_tasks(a.nf), wgs = (tasks + 3) / 4, slot = blockIdx.x / wgs;
  if (a.need && !a.need[slot])
    return;
  const int cell = a.cells[slot], task = (blockIdx.x % wgs) * 4 + (threadIdx.x >> 6), np = a.nf + 1;
  if (task >= tasks)
    return;
  const double *x = a.bases + a.bas_off[cell];
  const double *e = a.need ? a.corr + (size_t)slot * kDirectRhs * np * np : nullptr;
  double s[kDirectRhs] = {0, 0, 0, 0};
  auto sum = [&](int i, int, int, double r) { s[i] += r * r; };
  if (e)
    sweep<CELLS>(
      a, slot, cell, task,
      [&](int i, int X, int Y) {
        const size_t k = ((size_t)i * np + Y) * np + X;
        return x[k] + e[k];
      },
      sum);
  else
    sweep<CELLS>(a, slot, cell, task, [&](int i, int X, int Y) { return x[((size_t)i * np + Y) * np + X]; }, sum);
#pragma unroll
  for (int i = 0; i < kDirectRhs; ++i)
    {
      const double t = group_sum_dpp<64>(s[i]);
      if ((threadIdx.x & 63) == 0)
        a.part[((size_t)slot * tasks + task) * 12 + 8 + i] = t;
    }
}

// Settles a pass: every basis's residual norm against its tolerance.  A basis that the Q1
// interpolant already solves keeps the interpolant (no iteration); a cell that misses a
// tolerance has its residuals stored as the loads of a correction (need[slot] = 1).  After the
// correction (a.need): x += correction.
template <int CELLS>
__global__ void __launch_bounds__(kTpb) direct_settle(DirectArgs a, double *loads, int *need)
{
  const int slot = blockIdx.x;
  if (a.need && !a.need[slot])
    return;
  const int cell = a.cells[slot], nf = a.nf, np = nf + 1, nn = np * np, tasks = sweep_tasks(nf);
  const bool corrected = a.need != nullptr;
  double t[12];
#pragma unroll
  for (int k = 0; k < 12; ++k)
    t[k] = 0;
  for (int s = 0; s < tasks; ++s)
#pragma unroll
    for (int k = 0; k < 12; ++k)
      t[k] += a.part[((size_t)slot * tasks + s) * 12 + k];
  bool taken[kDirectRhs], miss = false, any = corrected;
  double tol[kDirectRhs], rn[kDirectRhs];
#pragma unroll
  for (int i = 0; i < kDirectRhs; ++i)
    {
      tol[i] = a.ptol ? a.ptol[(size_t)cell * a.nb + i] : fmax(a.rel_tol * sqrt(t[i]), a.abs_tol);
      const double q = sqrt(t[4 + i]), r = sqrt(t[8 + i]);
      taken[i] = !a.verts && a.q1_start && q <= tol[i];
      rn[i] = taken[i] ? q : r;
      miss = miss || (i < a.nb_solve && !(rn[i] <= tol[i]));
      any = any || taken[i];
    }
  if (threadIdx.x == 0)
    {
#pragma unroll
      for (int i = 0; i < kDirectRhs; ++i)
        if (i < a.nb_solve)
          {
            const size_t k = (size_t)cell * a.nb + i;
            if (a.iters)
              a.iters[k] = taken[i] ? 0 : corrected ? 2 : 1;
            if (a.status)
              a.status[k] = rn[i] <= tol[i] ? 0 : 1;
            if (a.resid)
              a.resid[k] = rn[i];
          }
      if (!corrected)
        need[slot] = miss ? 1 : 0;
    }
  double *x = a.bases + a.bas_off[cell];
  double *E = a.corr + (size_t)slot * kDirectRhs * nn;
  if (any)
    {
      for (int k = threadIdx.x; k < kDirectRhs * nn; k += kTpb)
        {
          const int i = k / nn, X = k % np, Y = k % nn / np;
          if (X == 0 || Y == 0 || X == nf || Y == nf)
            continue;
          const bool ti = i == 0 ? taken[0] : i == 1 ? taken[1] : i == 2 ? taken[2] : taken[3];
          if (ti)
            x[k] = nodal_q1(i, 2, X, Y, 0, nf);
          else if (corrected)
            x[k] += E[k];
        }
      __syncthreads();
    }
  if (miss && !corrected)
    {
      double *R = loads + (size_t)slot * kDirectRhs * nn;
      for (int s = threadIdx.x >> 6; s < tasks; s += kTpb / 64)
        sweep<CELLS>(a, slot, cell, s, [&](int i, int X, int Y) { return x[((size_t)i * np + Y) * np + X]; },
                     [&](int i, int X, int Y, double r) { R[((size_t)i * np + Y) * np + X] = r; });
      // the outline carries neither load nor correction
      for (int k = threadIdx.x; k < kDirectRhs * nn; k += kTpb)
        {
          const int X = k % np, Y = k % nn / np;
          if (X == 0 || Y == 0 || X == nf || Y == nf)
            R[k] = E[k] = 0.0;
        }
    }
}

// Front kernels by tile rows: the smallest that holds a level's largest front.  Up to 8 tile
// rows four waves share a front, beyond eight do (20 tiles of 8 registers each at 16 rows).
hipError_t launch_front(const DirectArgs &a, int rows, int grid, hipStream_t st)
{
  const int t = (rows + 15) / 16;
  if (t <= 6)
    hipLaunchKernelGGL((direct_front<6, 2, 2>), dim3(grid), dim3(256), 0, st, a);
  else if (t <= 8)
    hipLaunchKernelGGL((direct_front<8, 2, 2>), dim3(grid), dim3(256), 0, st, a);
  else if (t <= 9)
    hipLaunchKernelGGL((direct_front<9, 2, 2>), dim3(grid), dim3(256), 0, st, a);
  else if (t <= 13)
    hipLaunchKernelGGL((direct_front<13, 4, 2>), dim3(grid), dim3(512), 0, st, a);
  else if (t <= 16)
    hipLaunchKernelGGL((direct_front<16, 4, 2>), dim3(grid), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((direct_front<17, 2, 4>), dim3(grid), dim3(512), 0, st, a);
  return hipGetLastError();
}

template <int CELLS>
hipError_t launch_pass(DirectArgs a, const DirectHost &h, int n, hipStream_t st)
{
  const int D = h.depth, nblk = h.n_fronts[D - 1];
  hipLaunchKernelGGL(direct_leaf_forward<CELLS>, dim3(n * nblk), dim3(kTpb), 0, st, a);
  hipError_t e = hipGetLastError();
  for (int l = D - 2; l >= 0 && e == hipSuccess; --l)
    {
      a.level = l;
      e = launch_front(a, h.max_rows[l], n * h.n_fronts[l], st);
    }
  for (int l = 0; l <= D - 2 && e == hipSuccess; ++l)
    {
      a.level = l;
      const dim3 grid(n * h.n_fronts[l]);
      if (h.max_elim[l] <= 64)
        hipLaunchKernelGGL(direct_front_back<1>, grid, dim3(64), 0, st, a);
      else if (h.max_elim[l] <= 128)
        hipLaunchKernelGGL(direct_front_back<2>, grid, dim3(64), 0, st, a);
      else
        hipLaunchKernelGGL(direct_front_back<4>, grid, dim3(64), 0, st, a);
      e = hipGetLastError();
    }
  if (e == hipSuccess)
    {
      hipLaunchKernelGGL(direct_leaf_back<CELLS>, dim3(n * nblk), dim3(kTpb), 0, st, a);
      e = hipGetLastError();
    }
  return e;
}

template <int CELLS>
hipError_t solve_chunk(DirectArgs a, const DirectHost &h, int n, hipStream_t st)
{
  int *need = a.need_out;
  double *loads = a.loads_out;
  const dim3 sweeps(n * ((sweep_tasks(h.nf) + 3) / 4));
  hipError_t e = hipSuccess;
  if (CELLS == kStored)
    {
      hipLaunchKernelGGL(direct_conductances, dim3(n * ((h.nf * h.nf + kTpb - 1) / kTpb)), dim3(kTpb), 0, st, a);
      e = hipGetLastError();
    }
  if (e == hipSuccess)
    {
      hipLaunchKernelGGL(direct_start<CELLS>, sweeps, dim3(kTpb), 0, st, a);
      e = hipGetLastError();
    }
  for (int pass = 0; pass < 2 && e == hipSuccess; ++pass)
    {
      a.second = pass;
      a.need = pass ? need : nullptr;
      a.loads = pass ? loads : nullptr;
      e = launch_pass<CELLS>(a, h, n, st);
      if (e != hipSuccess)
        break;
      hipLaunchKernelGGL(direct_residual<CELLS>, sweeps, dim3(kTpb), 0, st, a);
      hipLaunchKernelGGL(direct_settle<CELLS>, dim3(n), dim3(kTpb), 0, st, a, loads, need);
      e = hipGetLastError();
    }
  return e;
}

} // namespace

bool direct_supported(int dim, int nf) { return dim == 2 && nf >= kDirectMinNf && nf <= kDirectMaxNf; }

void direct_host_plan(int nf, DirectHost &h, std::vector<char> &blob)
{
  const DirectPlan p = DirectPlanBuilder(nf).build();
  h.nf = nf;
  h.depth = p.depth;
  h.cell_doubles = p.cell_doubles;
  size_t off = 0;
  auto add = [&](const void *src, size_t bytes) {
    off = (off + 15) & ~(size_t)15;
    blob.resize(off + bytes);
    std::copy((const char *)src, (const char *)src + bytes, blob.data() + off);
    const size_t at = off;
    off += bytes;
    return at;
  };
  for (int l = 0; l < p.depth; ++l)
    {
      h.n_fronts[l] = (int)p.fronts[l].size();
      h.max_rows[l] = p.max_rows[l];
      h.max_elim[l] = 0;
      for (const DirectFront &f : p.fronts[l])
        h.max_elim[l] = std::max(h.max_elim[l], f.ne);
      h.fronts_at[l] = add(p.fronts[l].data(), p.fronts[l].size() * sizeof(DirectFront));
    }
  h.leaves_at = add(p.leaves.data(), p.leaves.size() * sizeof(DirectLeaf));
  h.types_at = add(p.types.data(), p.types.size() * sizeof(DirectLeafType));
  h.tables_at = add(p.pool.data(), p.pool.size() * sizeof(uint32_t));
}

// Doubles of scratch per cell: factors, loads and corrections, residual sums, flags, and the
// stored fine cells where a class needs them.
static size_t direct_cell_doubles(const DirectHost &h, bool stored)
{
  const size_t nn = (size_t)(h.nf + 1) * (h.nf + 1);
  return h.cell_doubles + 2 * kDirectRhs * nn + 12 * sweep_tasks(h.nf) + 2 + (stored ? 6 * (size_t)h.nf * h.nf : 0);
}

// Whether a class reads stored fine cells (see kStored).
static bool direct_stored(int coef_kind, bool general) { return general || coef_kind > 1; }

// Cells solved together: as many as keep their scratch within 4.5 GB of the 288, so that a batch of
// any size needs no more.  A chunk is ~20 launches, whose upper levels have 1, 4, 16 fronts a cell
// and end in partly empty waves of workgroups, so fewer are better: 4096 cells of 64^2 take 13.5 ms
// with 0.25 GB, 9.28 with 1.5, 8.81 with 4.5 and 8.61 with 6.4.
constexpr size_t kChunkDoubles = 560000000;
static int direct_chunk(const DirectHost &h, int n_cells, bool stored)
{
  return (int)std::min<size_t>(n_cells, std::max<size_t>(16, kChunkDoubles / direct_cell_doubles(h, stored)));
}

size_t direct_scratch_doubles(const DirectHost &h, int n_cells, int coef_kind, bool general)
{
  const bool stored = direct_stored(coef_kind, general);
  return (size_t)direct_chunk(h, n_cells, stored) * direct_cell_doubles(h, stored);
}

hipError_t launch_direct_solve(const DirectHost &h, const char *blob, const LocalArgs &in, int n_cells, int coef_kind,
                               double *scratch, hipStream_t st)
{
  const bool stored = direct_stored(coef_kind, in.verts != nullptr);
  const size_t chunk = (size_t)direct_chunk(h, n_cells, stored), nn = (size_t)(h.nf + 1) * (h.nf + 1);
  DirectArgs a = {};
  a.nf = h.nf;
  a.depth = h.depth;
  a.nb = in.nb;
  a.nb_solve = in.nb_solve;
  a.coef_kind = coef_kind;
  a.box = in.box;
  a.verts = in.verts;
  a.coef = in.coef;
  a.coef_off = in.coef_off;
  a.bases = in.bases;
  a.bas_off = in.bas_off;
  for (int l = 0; l < h.depth; ++l)
    {
      a.n_fronts[l] = h.n_fronts[l];
      a.fronts[l] = (const DirectFront *)(blob + h.fronts_at[l]);
    }
  a.leaves = (const DirectLeaf *)(blob + h.leaves_at);
  a.types = (const DirectLeafType *)(blob + h.types_at);
  a.tables = (const uint32_t *)(blob + h.tables_at);
  a.cell_doubles = h.cell_doubles;
  a.scratch = scratch;
  a.loads_out = scratch + chunk * h.cell_doubles;
  a.corr = a.loads_out + chunk * kDirectRhs * nn;
  a.cond = a.corr + chunk * kDirectRhs * nn;
  a.part = a.cond + (stored ? chunk * 6 * h.nf * h.nf : 0);
  a.need_out = (int *)(a.part + chunk * 12 * sweep_tasks(h.nf));
  a.ptol = in.ptol;
  a.rel_tol = in.rel_tol;
  a.abs_tol = in.abs_tol;
  a.q1_start = in.q1_start;
  a.iters = in.iters;
  a.status = in.status;
  a.resid = in.resid;
  hipError_t e = hipSuccess;
  for (int c = 0; c < n_cells && e == hipSuccess; c += (int)chunk)
    {
      a.cells = in.cells + c;
      const int n = (int)std::min<size_t>(chunk, n_cells - c);
      e = stored ? solve_chunk<kStored>(a, h, n, st) : solve_chunk<kFormed>(a, h, n, st);
    }
  return e;
}

} // namespace msfem
