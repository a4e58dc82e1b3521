// Host check of the SpMV row tiles (xyst_amd/csrc/xg_tiles.cpp) on a seeded
// random matrix with empty rows and rows longer than a tile:
// tiles_check NROW NCOL MEAN_NNZ NLONG SEED [ROWS] (default: as the CG).  Prints "ok" or the
// first mismatch.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>

#include "../../xyst_amd/csrc/xg_tiles.hpp"

int main(int argc, char** argv) {
  if (argc != 6 && argc != 7) return 2;
  const long nrow = atol(argv[1]), ncol = atol(argv[2]), mean = atol(argv[3]);
  const long nlong = atol(argv[4]);
  std::mt19937 g(atoi(argv[5]));
  std::vector<int64_t> ia(1, 0);
  std::vector<int32_t> ja;
  for (long r = 0; r < nrow; ++r) {
    long n = mean ? (long)(g() % (2 * mean + 1)) : 0;
    if (nlong && r % (nrow / nlong) == nrow / nlong - 1)
      n = xg::kTileNnz + (r % 2 ? 1 : 0);   // a full tile, or one more
    std::set<int32_t> c;
    n = std::min(n, ncol);
    while ((long)c.size() < n) c.insert((int32_t)(g() % ncol));
    ja.insert(ja.end(), c.begin(), c.end());
    ia.push_back((int64_t)ja.size());
  }
  const int64_t nnz = (int64_t)ja.size();
  const int maxr = argc == 7 ? atoi(argv[6]) : xg::tile_rows(nrow, nnz);
  // at least three quarters of a tile's nonzeros or the most rows
  if (argc != 7 && maxr != xg::kTileRowsMax &&
      4 * maxr * nnz < 3 * xg::kTileNnz * nrow)
    return printf("rows\n"), 1;
  xg::TileSet t;
  xg::build_tiles(nrow, ncol, ia.data(), ja.data(), t, maxr);
  long next = 0;
  size_t u0 = 0;
  int64_t nwide = 0;
  for (const xg::Tile& w : t.tile) {
    if (w.row0 != next || w.row1 <= w.row0 || w.k0 != ia[w.row0] ||
        w.nz != ia[w.row1] - ia[w.row0])
      return printf("tile of row %ld\n", next), 1;
    next = w.row1;
    if (w.row1 - w.row0 > maxr) return printf("too many rows\n"), 1;
    if (w.nz > xg::kTileNnz) {
      if (!t.has_long) return printf("has_long\n"), 1;
      if (w.row1 - w.row0 != 1 || w.nu) return printf("long row %d\n", w.row0), 1;
      continue;
    }
    if ((size_t)w.u0 != u0 || w.nu > w.nz) return printf("list of row %d\n", w.row0), 1;
    u0 += w.nu;
    nwide += w.nu > xg::kTileCols;
    std::set<int32_t> used;
    for (int k = 0; k < w.nz; ++k) {
      if (t.lidx[w.k0 + k] >= w.nu || t.ucol[w.u0 + t.lidx[w.k0 + k]] != ja[w.k0 + k])
        return printf("entry %d\n", w.k0 + k), 1;
      used.insert(ja[w.k0 + k]);
    }
    if ((int)used.size() != w.nu) return printf("unused columns\n"), 1;
    for (int k = 1; k < w.nu; ++k)
      if (t.ucol[w.u0 + k] <= t.ucol[w.u0 + k - 1]) return printf("order\n"), 1;
  }
  if (nwide != t.nwide) return printf("nwide\n"), 1;
  if (next != nrow || u0 != t.ucol.size() || t.lidx.size() != ja.size())
    return printf("sizes\n"), 1;
  printf("ok\n");
  return 0;
}
