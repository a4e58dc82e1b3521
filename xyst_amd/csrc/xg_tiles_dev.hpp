// SpMV over row tiles on the device (see xg_tiles.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "xg_tiles.hpp"

namespace {

constexpr int kTileThreads = 256;
// workgroups of a SpMV launch: four per CU, so that a launch of more than
// 1024 tiles walks them evenly with the next tile's loads in flight
constexpr int kSpmvGrid = 1024;

// LDS of a workgroup: the tile's source values and its products
template <class T>
struct TileLds {
  T src[xg::kTileNnz];
  T prod[xg::kTileNnz];
  double sm[4][kTileThreads / 64];
};

// For the rows of this workgroup's tiles (ti = blockIdx.x, + gridDim.x, ...)
// row.apply(r, row.load(r), sum_k a_k v(ja_k)), once per row:
//   src.load(c), src.value(raw): the source value v(c), loaded and formed in
//     two steps, so that coef() -- scalars that value() needs, themselves
//     sums over the last kernel's partials -- runs while the loads of the
//     first tile are in flight.  coef() false: nothing to do.
//   row.load(r): what the row's result needs, loaded ahead of its sum.
// LANES false: one thread per row, its products in CSR order; true: as many
// lanes per row (a power of two, at most 64) as the tile's rows leave room
// for, strided partial sums and a fixed butterfly -- for matrices whose rows
// are long or whose tiles have few.  Fixed order in both.  Every thread of
// the workgroup calls this (it holds barriers).
//
// What bounds it: bytes from some 600,000 rows on, below that the chain of
// dependent loads of one or two tiles per workgroup.  So the loads of the
// next tile are in flight during the current one: its source values from the
// start (their columns were loaded a tile before), the rest from the
// products on.
// COLS: columns a thread loads ahead (3: lists of up to kTileCols columns; a
// longer list costs its tile a chain of two loads).
template <class T, bool LANES, int COLS, class Src, class Row, class Coef>
__device__ inline bool tiles_spmv(const xg::TileMat& M, const T* __restrict__ a, Src& src,
                                  Row& row, Coef coef, TileLds<T>& lds) {
  constexpr int kShare = xg::kTileNnz / kTileThreads;   // nonzeros of a thread
  constexpr int kCols = COLS;
  // in FP64 the row's own data a tile ahead would take the registers of a
  // fourth wave per SIMD (148; 64^3: 20.4 us a launch instead of 16.5; in
  // FP32 19.7 instead of 21.0 at 80^3)
  constexpr bool kRowsAhead = sizeof(T) == 4;
  const unsigned t = threadIdx.x;
  const int G = gridDim.x;
  typename Src::Raw raw[kCols];
  unsigned li[kShare] = {}, uc[kCols];
  T av[kShare] = {};
  int e0 = 0, e1 = 0, sh = 0;
  typename Row::Raw own = {};
  // Loads past the end of a list are of its last entry: no branch between
  // the loads.  A long row's tile has an empty list and is not prefetched.
  auto columns = [&](const xg::Tile& W) {
    if (W.nu == 0) return;
    const int* u = M.ucol + W.u0;
#pragma unroll
    for (int k = 0; k < kCols; ++k)
      uc[k] = (unsigned)u[min(t + k * kTileThreads, (unsigned)W.nu - 1)];
  };
  auto gather = [&](const xg::Tile& W) {
    if (W.nu == 0) return;
#pragma unroll
    for (int k = 0; k < kCols; ++k) raw[k] = src.load(uc[k]);
  };
  auto entries = [&](const xg::Tile& W) {
    if (W.nu == 0) return;
    const uint16_t* l = M.lidx + W.k0;
    const T* v = a + W.k0;
#pragma unroll
    for (int k = 0; k < kShare; ++k) {
      const unsigned kk = min(t + k * kTileThreads, (unsigned)W.nz - 1);
      li[k] = l[kk];
      av[k] = v[kk];
    }
  };
  // lanes per row (1 << sh), this thread's row and what its result needs
  auto rows = [&](const xg::Tile& W) {
    if (W.nu == 0) return;
    if (LANES) {
      sh = 0;
      while (sh < 6 && ((W.row1 - W.row0) << (sh + 1)) <= kTileThreads) ++sh;
    }
    const int r = min(W.row0 + (int)(t >> sh), W.row1 - 1);
    e0 = M.ia[r] - W.k0;
    e1 = M.ia[r + 1] - W.k0;
    own = row.load(r);
  };
  const xg::Tile none = {};
  auto record = [&](int ti) { return ti < M.ntile ? M.tile[ti] : none; };
  xg::Tile W = record(blockIdx.x), W1 = record(blockIdx.x + G);
  columns(W);
  entries(W);
  if (kRowsAhead) rows(W);
  gather(W);
  columns(W1);
  if (!coef()) return false;
  for (int ti = blockIdx.x; ti < M.ntile; ti += G) {
    const xg::Tile W2 = record(ti + 2 * G);
    if (W.nu) {
      if (!kRowsAhead) rows(W);
#pragma unroll
      for (int k = 0; k < kCols; ++k)
        if (t + k * kTileThreads < (unsigned)W.nu)
          lds.src[t + k * kTileThreads] = src.value(raw[k]);
      for (unsigned k = t + kCols * kTileThreads; k < (unsigned)W.nu; k += kTileThreads)
        lds.src[k] = src.value(src.load((unsigned)M.ucol[W.u0 + k]));
      gather(W1);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kShare; ++k) lds.prod[t + k * kTileThreads] = av[k] * lds.src[li[k]];
      const int r = W.row0 + (int)(t >> sh), lane = (int)t & ((1 << sh) - 1);
      const int f0 = e0, f1 = e1, s = sh;
      const typename Row::Raw mine = own;
      entries(W1);
      if (kRowsAhead) rows(W1);
      columns(W2);
      __syncthreads();        // src is the next tile's
      if (!LANES) {
        if (r < W.row1) {
          T acc = T(0);
          for (int k = f0; k < f1; k += 8) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = lds.prod[min(k + u, xg::kTileNnz - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (k + u < f1) acc += v[u];
          }
          row.apply(r, mine, acc);
        }
      } else {
        T acc = T(0);
        if (r < W.row1)
          for (int k = f0 + lane; k < f1; k += 4 << s) {
            T v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = lds.prod[min(k + (u << s), xg::kTileNnz - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (k + (u << s) < f1) acc += v[u];
          }
        for (int o = 1; o < 1 << s; o <<= 1) acc += __shfl_xor(acc, o, 64);
        if (r < W.row1 && lane == 0) row.apply(r, mine, acc);
      }
    } else if (W.nz == 0) {
      // rows without nonzeros
      const int r = W.row0 + (int)t;
      if (r < W.row1) row.apply(r, row.load(r), T(0));
      gather(W1);
      entries(W1);
      if (kRowsAhead) rows(W1);
      columns(W2);
    } else {
      // one row longer than a tile: strided partial sums, fixed-order tree
      T acc = T(0);
      for (int k = (int)t; k < W.nz; k += kTileThreads)
        acc += a[W.k0 + k] * src.value(src.load((unsigned)M.ja[W.k0 + k]));
      double s = (double)acc;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      __syncthreads();        // sm free from a previous use
      if ((t & 63) == 0) lds.sm[3][t >> 6] = s;
      __syncthreads();
      if (t == 0) {
        s = 0.0;
        for (int k = 0; k < kTileThreads / 64; ++k) s += lds.sm[3][k];
        row.apply(W.row0, row.load(W.row0), (T)s);
      }
      gather(W1);
      entries(W1);
      if (kRowsAhead) rows(W1);
      columns(W2);
    }
    W = W1;
    W1 = W2;
  }
  return true;
}

}  // namespace
