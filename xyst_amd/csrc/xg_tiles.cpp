// Host side of the SpMV row tiles (see xg_tiles.hpp).
#include "xg_tiles.hpp"

#include <algorithm>
#include <atomic>
#include <exception>
#include <system_error>
#include <thread>

namespace xg {

namespace {

// work() on up to nth threads, the caller's among them: as many as can be
// created.  What one of them throws is thrown again here.
template <class Work>
void on_threads(int64_t nth, Work work) {
  std::vector<std::exception_ptr> bad(std::max<int64_t>(nth, 1));
  auto guarded = [&](int64_t k) {
    try {
      work();
    } catch (...) {
      bad[k] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(bad.size());
  try {
    for (int64_t k = 1; k < nth; ++k) th.emplace_back(guarded, k);
  } catch (const std::system_error&) {   // no more threads: those there are
  }
  guarded(0);
  for (auto& x : th) x.join();
  for (const auto& e : bad)
    if (e) std::rethrow_exception(e);
}

}  // namespace

void build_tiles(int64_t nrow, int64_t ncol, const int64_t* ia, const int32_t* ja, TileSet& t,
                 int rows) {
  t = TileSet();
  for (int64_t r = 0; r < nrow;) {
    int64_t r1 = r;
    while (r1 < nrow && r1 - r < rows && ia[r1 + 1] - ia[r] <= kTileNnz) ++r1;
    if (r1 == r) r1 = r + 1;
    Tile w{};
    w.row0 = (int)r;
    w.row1 = (int)r1;
    w.k0 = (int)ia[r];
    w.nz = (int)(ia[r1] - ia[r]);
    t.tile.push_back(w);
    if (w.nz > kTileNnz) t.has_long = true;
    r = r1;
  }
  t.lidx.assign((size_t)ia[nrow], 0);
  const int64_t nt = (int64_t)t.tile.size();
  const int64_t per = 512;   // tiles a piece of work: some million nonzeros
  const int64_t npiece = (nt + per - 1) / per;
  std::vector<std::vector<int32_t>> cols((size_t)npiece);
  std::atomic<int64_t> next{0};
  auto work = [&] {
    std::vector<int32_t> at((size_t)ncol, -1);
    std::vector<int32_t> u;
    for (int64_t p; (p = next++) < npiece;) {
      for (int64_t i = p * per; i < std::min(nt, (p + 1) * per); ++i) {
        Tile& w = t.tile[i];
        if (w.nz > kTileNnz) continue;
        u.clear();
        for (int64_t k = w.k0; k < (int64_t)w.k0 + w.nz; ++k)
          if (at[ja[k]] < 0) {
            at[ja[k]] = 0;
            u.push_back(ja[k]);
          }
        std::sort(u.begin(), u.end());
        for (size_t k = 0; k < u.size(); ++k) at[u[k]] = (int32_t)k;
        for (int64_t k = w.k0; k < (int64_t)w.k0 + w.nz; ++k) t.lidx[k] = (uint16_t)at[ja[k]];
        for (int32_t c : u) at[c] = -1;
        w.u0 = (int)cols[p].size();
        w.nu = (int)u.size();
        cols[p].insert(cols[p].end(), u.begin(), u.end());
      }
    }
  };
  const int64_t nth = std::min<int64_t>(
      npiece, std::min(8u, std::max(1u, std::thread::hardware_concurrency())));
  on_threads(nth, work);
  for (int64_t p = 0; p < npiece; ++p) {
    const int base = (int)t.ucol.size();
    for (int64_t i = p * per; i < std::min(nt, (p + 1) * per); ++i) {
      t.tile[i].u0 += base;
      t.nwide += t.tile[i].nu > kTileCols;
    }
    t.ucol.insert(t.ucol.end(), cols[p].begin(), cols[p].end());
  }
}

}  // namespace xg
