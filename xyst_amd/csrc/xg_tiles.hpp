// Row tiles of a CSR matrix for SpMV on the device (xg_cg.hip, xg_amg.hip).
//
// A tile is a run of consecutive rows with at most kTileNnz nonzeros and
// kTileRows or kTileRowsMax rows (a longer row is a tile of its own, without a
// column list).
// Neighbouring rows share most of their columns: the matrix of a tet mesh
// has some 560 different ones among a tile's 2048 nonzeros.  So a tile lists
// its columns once, ascending, and its nonzeros hold 16-bit positions in
// that list: a workgroup reads every source value once, with neighbouring
// lanes on neighbouring addresses, into LDS, where the nonzeros find it, and
// a nonzero costs 2 bytes of index instead of 4 (with the lists 3.1; 2.8 in
// compact cells, 3.5 in band order at 160^3).
#pragma once
#include <cstdint>
#include <memory>
#include <new>
#include <utility>
#include <vector>

namespace xg {

constexpr int kTileNnz = 2048;
constexpr int kTileRows = 128;     // two lanes a row in the V-cycle's kernels
constexpr int kTileRowsMax = 256;  // a thread a row
constexpr int kTileCols = 768;   // columns that a workgroup loads a tile ahead

struct alignas(32) Tile {
  int row0, row1;   // rows
  int k0, nz;       // first nonzero, nonzeros
  int u0, nu;       // column list
  int pad0, pad1;
};

// on the device, with the matrix' row offsets
struct TileMat {
  int ntile = 0;
  const Tile* tile = nullptr;
  const int* ia = nullptr;
  const int* ja = nullptr;   // columns (only of rows longer than a tile)
  const int* ucol = nullptr;
  const uint16_t* lidx = nullptr;
};

// std::vector whose new elements are left as they are: they are written by
// several threads, which then touch the pages first
template <class T>
struct NoInit : std::allocator<T> {
  template <class U>
  struct rebind {
    using other = NoInit<U>;
  };
  template <class U>
  void construct(U* p) noexcept { ::new ((void*)p) U; }
  template <class U, class... A>
  void construct(U* p, A&&... a) { ::new ((void*)p) U(std::forward<A>(a)...); }
};
template <class T>
using RawVector = std::vector<T, NoInit<T>>;

struct TileSet {
  bool has_long = false;        // a row is longer than a tile
  int64_t nwide = 0;            // tiles with more than kTileCols columns
  std::vector<Tile> tile;
  RawVector<int32_t> ucol;      // the tiles' columns
  RawVector<uint16_t> lidx;   // per nonzero: position in its tile's list
};

// Tiles of the matrix with row offsets ia (nrow + 1, from 0) and columns ja
// below ncol, of at most `rows` rows.  Threads work on runs of tiles; the
// result does not depend on their number.
void build_tiles(int64_t nrow, int64_t ncol, const int64_t* ia, const int32_t* ja, TileSet& t,
                 int rows = kTileRows);

// Rows of a tile where one thread sums a row (the CG recurrences): twice
// kTileRows where these would leave a quarter of a tile's nonzeros unused, as
// below 12 entries a row.  An iteration on 10^6 rows with 128 and 256 rows a
// tile: 7 entries a row 56.1 and 49.8 us in FP64, 43.3 and 35.4 in FP32; 3
// entries 53.7 and 41.6, 41.2 and 30.7.  The matrix of a tet mesh has 15.
inline int tile_rows(int64_t nrow, int64_t nnz) {
  return 4 * kTileRows * nnz < 3 * kTileNnz * nrow ? kTileRowsMax : kTileRows;
}

}  // namespace xg
