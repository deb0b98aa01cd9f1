// Symbolic side of the direct local solves (direct.hip): the nested dissection
// of one nf x nf fine grid, the same for every cell of a resolution class, so it
// is laid out once per resolution on the host and kept in device memory.
//
// The grid is cut in half along both axes `depth` times: level l has 4^l blocks,
// the blocks of level `depth` are the leaves (4..8 fine cells per side).  A block
// of level l < depth has a front: the nodes on the lines between its four
// children, which it eliminates, then the nodes of its own outline that other
// blocks share (Dirichlet nodes of the grid are never in a front), then the four
// right-hand sides as four more rows.  A leaf is made of 2 x 2-cell patches whose
// centre nodes are eliminated by closed formulas, and so is the node in the middle
// of the side that the two patches of a pair (side by side) share; its front holds
// its other interior nodes and its outline.
#pragma once

#include <algorithm>
#include <cstdint>
#include <map>
#include <vector>

namespace msfem {

constexpr int kDirectMinNf = 9, kDirectMaxNf = 128; // resolutions with at least one cut and at most 17 tile rows
constexpr int kDirectRhs = 4;                      // bases of a 2D cell
constexpr int kPatchDoubles = 81;                  // 3 x 3-node patch: 45 lower entries, then 4 x 9 right-hand sides
constexpr int kLeafDoubles = 1328; // 16 patches and a last zero (what table entries without a source read), padded so
                                   // that two leaves' patches are in different LDS banks (1328 = 16 mod 32)
static_assert(16 * kPatchDoubles < kLeafDoubles);
constexpr int kLeafElim = 25;                        // most rows that a leaf's front eliminates
constexpr int kLeafTiles = 4, kLeafBackTiles = 2;    // tile rows of a leaf's front: 25 + 32 + 4 and 25 + 4 rows
constexpr int kLeafLd = 36;                          // leading dimension of a leaf's Schur complement (32 + 4)

// Row of a 16 x 16 FP64 accumulator tile that entry v of lane l holds (its column is l % 16).
constexpr int mfma_row(int lane, int v) { return (lane >> 4) + 4 * v; }

// A pair's middle node (node 5 of the left patch, 3 of the right one) couples the nodes kPairLeft
// of the left patch to the nodes kPairRight of the right one, neither of which the other has
// (node 5, or node 4 where the right patch is one cell wide).  These 25 entries take the place of
// the entries of the eliminated nodes: the first kPairSlotsLeft in the left patch, the others in
// the right one.
constexpr int kPairLeft[5] = {0, 1, 3, 6, 7}, kPairRight[5] = {1, 2, 5, 7, 8};
constexpr int kPairSlotsLeft = 17;
constexpr int kPairSlot[25] = {10, 11, 12, 13, 14, 19, 25, 32, 40, 15, 16, 17, 18, 20, 26, 33, 41, // (4, .), (5, .)
                               6,  7,  8,  9,  18, 24, 31, 39};                                 // (3, .)

struct DirectFront {
  int ne, nb;               // eliminated rows, outline rows (then kDirectRhs rows)
  int lds, ldw;             // leading dimensions of its Schur complement and of its W
  int nodes;                // pool offset: grid node of every row < ne + nb
  int codes;                // pool offset: byte k of row r = its row in child k's Schur complement, 255 = none
  int child[4];             // index of child k in the next level (leaf index on the last front level)
  int x0, y0, w, h;         // block, fine cells
  int tab, tabx;            // (last front level) pool offsets: per (tile, lane, v) two 16-bit sources, bytes from
                            // the four leaves' Schur complements; two more for the tiles in `extra`, in order
  unsigned extra;
  uint8_t kids[20];         // bit k of tile row i: some of rows 16 i .. 16 i + 15 are in child k
  long long s_off, w_off;   // doubles from the cell's scratch
};

struct DirectLeaf {
  int x0, y0, w, h, fwd, back; // fwd, back: types of the forward front and of the leaf with its whole outline given
};

struct DirectLeafType {
  int ne, nb;
  int nodes;                // pool offset: x | y << 8 (leaf coordinates) of every row < ne + nb
  int tab, tabx;            // pool offsets: per (tile, lane, v) two 16-bit sources (bytes from the leaf's
                            // patches); two more for the tiles in `extra`
  unsigned extra;
};

struct DirectPlan {
  int nf = 0, depth = 0;
  std::vector<std::vector<DirectFront>> fronts; // [level][block]
  std::vector<int> max_rows;                    // per level: largest front
  std::vector<DirectLeaf> leaves;
  std::vector<DirectLeafType> types;
  std::vector<uint32_t> pool;
  long long cell_doubles = 0;                   // scratch of one cell
};

inline int direct_depth(int nf)
{
  int d = 1;
  while ((8 << d) < nf)
    ++d;
  return d;
}

class DirectPlanBuilder {
public:
  explicit DirectPlanBuilder(int nf) { p.nf = nf, p.depth = direct_depth(nf); }

  DirectPlan build()
  {
    const int D = p.depth, nl = 1 << D, np = p.nf + 1;
    cut.resize(nl + 1);
    for (int i = 0; i <= nl; ++i)
      cut[i] = (int)((long long)i * p.nf / nl);
    p.fronts.resize(D);
    p.max_rows.assign(D, 0);
    std::vector<std::vector<std::vector<int>>> outline(D); // [level][block]: outline nodes in front order
    for (int l = 0; l < D; ++l)
      {
        const int n = 1 << l;
        outline[l].resize(n * n);
        for (int by = 0; by < n; ++by)
          for (int bx = 0; bx < n; ++bx)
            {
              DirectFront f = {};
              block(l, bx, by, f.x0, f.y0, f.w, f.h);
              const int xm = at(l + 1, 2 * bx + 1), ym = at(l + 1, 2 * by + 1);
              std::vector<int> rows;
              for (int y = f.y0 + 1; y < f.y0 + f.h; ++y)
                if (y != ym)
                  rows.push_back(y * np + xm);
              for (int x = f.x0 + 1; x < f.x0 + f.w; ++x)
                rows.push_back(ym * np + x);
              f.ne = (int)rows.size();
              if (l > 0)
                {
                  // in the parent's row order, so that a child's rows ascend with the parent's
                  const std::vector<int> &up = parent_rows[l - 1][(by / 2) * (n / 2) + bx / 2];
                  for (int node : up)
                    if (on_outline(f.x0, f.y0, f.w, f.h, node % np, node / np))
                      outline[l][by * n + bx].push_back(node);
                }
              const std::vector<int> &out = outline[l][by * n + bx];
              f.nb = (int)out.size();
              rows.insert(rows.end(), out.begin(), out.end());
              f.lds = f.nb + kDirectRhs;
              f.ldw = (f.ne + 15) & ~15;
              f.nodes = (int)p.pool.size();
              for (int node : rows)
                p.pool.push_back((uint32_t)node);
              for (int k = 0; k < 4; ++k)
                f.child[k] = (2 * by + (k >> 1)) * 2 * n + 2 * bx + (k & 1);
              if (l > 0)
                {
                  f.s_off = p.cell_doubles;
                  p.cell_doubles += (long long)f.lds * f.lds;
                }
              f.w_off = p.cell_doubles;
              const int m = f.ne + f.nb + kDirectRhs;
              p.cell_doubles += (long long)m * f.ldw;
              p.cell_doubles = (p.cell_doubles + 1) & ~1LL;
              p.max_rows[l] = std::max(p.max_rows[l], m);
              p.fronts[l].push_back(f);
              if ((int)parent_rows.size() <= l)
                parent_rows.resize(l + 1);
              parent_rows[l].push_back(rows);
            }
      }
    for (int by = 0; by < nl; ++by)
      for (int bx = 0; bx < nl; ++bx)
        {
          DirectLeaf q;
          block(D, bx, by, q.x0, q.y0, q.w, q.h);
          const int sides = (q.x0 == 0 ? 1 : 0) | (q.x0 + q.w == p.nf ? 2 : 0) | (q.y0 == 0 ? 4 : 0) |
                            (q.y0 + q.h == p.nf ? 8 : 0);
          q.fwd = leaf_type(q.w, q.h, sides, kLeafTiles);
          q.back = leaf_type(q.w, q.h, 15, kLeafBackTiles);
          p.leaves.push_back(q);
        }
    for (int l = 0; l < D; ++l)
      for (size_t b = 0; b < p.fronts[l].size(); ++b)
        {
          DirectFront &f = p.fronts[l][b];
          const std::vector<int> &rows = parent_rows[l][b];
          std::vector<uint32_t> code(f.ne + f.nb + kDirectRhs, 0xFFFFFFFFu);
          for (int k = 0; k < 4; ++k)
            {
              std::map<int, int> pos;
              int nbk;
              if (l + 1 < D)
                {
                  const std::vector<int> &c = outline[l + 1][f.child[k]];
                  for (size_t i = 0; i < c.size(); ++i)
                    pos[c[i]] = (int)i;
                  nbk = (int)c.size();
                }
              else
                {
                  const DirectLeaf &q = p.leaves[f.child[k]];
                  const DirectLeafType &t = p.types[q.fwd];
                  for (int i = 0; i < t.nb; ++i)
                    {
                      const uint32_t xy = p.pool[t.nodes + t.ne + i];
                      pos[(q.y0 + (int)(xy >> 8)) * np + q.x0 + (int)(xy & 255)] = i;
                    }
                  nbk = t.nb;
                }
              auto put = [&](size_t r, int v) { code[r] = (code[r] & ~(255u << (8 * k))) | ((uint32_t)v << (8 * k)); };
              for (size_t r = 0; r < rows.size(); ++r)
                {
                  auto it = pos.find(rows[r]);
                  if (it != pos.end())
                    put(r, it->second);
                }
              for (int i = 0; i < kDirectRhs; ++i)
                put(rows.size() + i, nbk + i);
            }
          for (size_t r = 0; r < code.size(); ++r)
            for (int k = 0; k < 4; ++k)
              if (((code[r] >> (8 * k)) & 255) != 255)
                f.kids[r / 16] |= 1 << k;
          f.codes = (int)p.pool.size();
          p.pool.insert(p.pool.end(), code.begin(), code.end());
          if (l + 1 == D)
            block_tables(f, code);
        }
    return p;
  }

private:
  DirectPlan p;
  std::vector<int> cut; // leaf boundaries along an axis
  std::vector<std::vector<std::vector<int>>> parent_rows;
  std::map<int, int> type_of;
  std::map<std::vector<uint32_t>, DirectFront> block_of;

  int at(int level, int i) const { return cut[i << (p.depth - level)]; }
  void block(int level, int bx, int by, int &x0, int &y0, int &w, int &h) const
  {
    x0 = at(level, bx), y0 = at(level, by);
    w = at(level, bx + 1) - x0, h = at(level, by + 1) - y0;
  }
  // Assembly tables of a last-level front; fronts with the same rows share them.
  void block_tables(DirectFront &f, const std::vector<uint32_t> &code)
  {
    auto it = block_of.find(code);
    if (it != block_of.end())
      {
        f.tab = it->second.tab, f.tabx = it->second.tabx, f.extra = it->second.extra;
        return;
      }
    const int m = (int)code.size(), tiles = (m + 15) / 16;
    std::vector<uint32_t> tab, tabx;
    for (int i = 0, q = 0; i < tiles; ++i)
      for (int j = 0; j <= i; ++j, ++q)
        {
          std::vector<uint32_t> more;
          bool any = false;
          for (int lane = 0; lane < 64; ++lane)
            for (int v = 0; v < 4; ++v)
              {
                uint32_t s[4];
                s[0] = s[1] = s[2] = s[3] = 4 * kLeafDoubles - 1;
                const int r = 16 * i + mfma_row(lane, v), c = 16 * j + lane % 16;
                if (r < m && c < m)
                  for (int k = 0, n = 0; k < 4; ++k)
                    {
                      const uint32_t a = (code[r] >> (8 * k)) & 255, b = (code[c] >> (8 * k)) & 255;
                      if (a != 255 && b != 255)
                        s[n++] = k * kLeafDoubles + std::max(a, b) * kLeafLd + std::min(a, b);
                    }
                tab.push_back(8 * s[0] | 8 * s[1] << 16);
                more.push_back(8 * s[2] | 8 * s[3] << 16);
                any = any || s[2] != 4 * kLeafDoubles - 1;
              }
          if (any)
            {
              f.extra |= 1u << q;
              tabx.insert(tabx.end(), more.begin(), more.end());
            }
        }
    p.pool.resize((p.pool.size() + 3) & ~(size_t)3); // (read four at a time)
    f.tab = (int)p.pool.size();
    p.pool.insert(p.pool.end(), tab.begin(), tab.end());
    f.tabx = (int)p.pool.size();
    p.pool.insert(p.pool.end(), tabx.begin(), tabx.end());
    block_of[code] = f;
  }
  bool on_outline(int x0, int y0, int w, int h, int x, int y) const
  {
    return x >= x0 && x <= x0 + w && y >= y0 && y <= y0 + h && (x == x0 || x == x0 + w || y == y0 || y == y0 + h);
  }

  // Front of a w x h leaf whose sides in `sides` (1 x = 0, 2 x = w, 4 y = 0, 8 y = h) hold given values.
  int leaf_type(int w, int h, int sides, int tiles)
  {
    const int key = ((w * 16 + h) * 16 + sides) * 8 + tiles;
    auto it = type_of.find(key);
    if (it != type_of.end())
      return it->second;
    DirectLeafType t = {};
    std::vector<int> row_x, row_y;
    for (int pass = 0; pass < 2; ++pass)
      {
        for (int y = 0; y <= h; ++y)
          for (int x = 0; x <= w; ++x)
            {
              const bool edge = x == 0 || x == w || y == 0 || y == h;
              const bool given = (x == 0 && (sides & 1)) || (x == w && (sides & 2)) || (y == 0 && (sides & 4)) ||
                                 (y == h && (sides & 8));
              const bool centre = (x & 1) && (y & 1) && !edge; // of a full patch: an odd node inside is followed by a cell
              const bool middle = x % 4 == 2 && (y & 1) && !edge; // of a pair, likewise
              if (given || (pass == 0 ? edge || centre || middle : !edge))
                continue;
              row_x.push_back(x), row_y.push_back(y);
            }
        (pass == 0 ? t.ne : t.nb) = (int)row_x.size() - (pass == 0 ? 0 : t.ne);
      }
    t.nodes = (int)p.pool.size();
    for (size_t r = 0; r < row_x.size(); ++r)
      p.pool.push_back((uint32_t)(row_x[r] | row_y[r] << 8));
    const int n = (int)row_x.size(), m = n + kDirectRhs, pw = (w + 1) / 2, ph = (h + 1) / 2;
    const uint32_t none = kLeafDoubles - 1;
    auto sources = [&](int r, int c, uint32_t (&s)[4]) {
      s[0] = s[1] = s[2] = s[3] = none;
      if (r < c)
        std::swap(r, c);
      if (r >= m || c >= n)
        return;
      int k = 0;
      for (int py = 0; py < ph; ++py)
        for (int px = 0; px < pw; ++px)
          {
            const int cx = row_x[c] - 2 * px, cy = row_y[c] - 2 * py;
            if (cx < 0 || cx > 2 || cy < 0 || cy > 2)
              continue;
            const int b = cx + 3 * cy, base = (py * 4 + px) * kPatchDoubles;
            if (r >= n)
              {
                s[k++] = base + 45 + (r - n) * 9 + b;
                continue;
              }
            const int rx = row_x[r] - 2 * px, ry = row_y[r] - 2 * py;
            if (rx < 0 || rx > 2 || ry < 0 || ry > 2)
              continue;
            const int a = rx + 3 * ry, hi = std::max(a, b), lo = std::min(a, b);
            s[k++] = base + hi * (hi + 1) / 2 + lo;
          }
      if (r < n) // coupled through a pair's middle node
        for (int py = 0; py < ph; ++py)
          for (int px = 0; px + 1 < pw; px += 2)
            {
              if (2 * py + 2 > h)
                continue;
              const int left = row_x[r] < row_x[c] ? r : c, right = r + c - left;
              const int lx = row_x[left] - 2 * px, ly = row_y[left] - 2 * py;
              const int rx = row_x[right] - 2 * px - 2, ry = row_y[right] - 2 * py;
              if (lx < 0 || lx > 1 || rx < 1 || rx > 2 || ly < 0 || ly > 2 || ry < 0 || ry > 2)
                continue;
              int li = 0, ri = 0;
              while (kPairLeft[li] != lx + 3 * ly)
                ++li;
              const int rn = rx + 3 * ry;
              while (kPairRight[ri] != (rn == 4 ? 5 : rn))
                ++ri;
              const int e = li * 5 + ri;
              s[k++] = (py * 4 + px + (e < kPairSlotsLeft ? 0 : 1)) * kPatchDoubles + kPairSlot[e];
            }
    };
    std::vector<uint32_t> tab, tabx;
    for (int i = 0, q = 0; i < tiles; ++i)
      for (int j = 0; j <= i; ++j, ++q)
        for (int lane = 0; lane < 64; ++lane)
          for (int v = 0; v < 4; ++v)
            {
              uint32_t s[4];
              sources(16 * i + mfma_row(lane, v), 16 * j + lane % 16, s);
              tab.push_back(8 * s[0] | 8 * s[1] << 16);
              tabx.push_back(8 * s[2] | 8 * s[3] << 16);
              if (s[2] != none)
                t.extra |= 1u << q;
            }
    p.pool.resize((p.pool.size() + 3) & ~(size_t)3); // (read four at a time)
    t.tab = (int)p.pool.size();
    p.pool.insert(p.pool.end(), tab.begin(), tab.end());
    t.tabx = (int)p.pool.size();
    p.pool.insert(p.pool.end(), tabx.begin(), tabx.end());
    p.types.push_back(t);
    return type_of[key] = (int)p.types.size() - 1;
  }
};

} // namespace msfem
