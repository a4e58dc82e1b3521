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

// Set of columns as two levels of bits: bit c of `bits`, and bit w of `top`
// where word w of `bits` is not empty, so that the set is read in order, and
// emptied, in time of its size and its range / 4096.
struct ColumnSet {
  std::vector<uint64_t> bits, top;
  std::vector<uint16_t> before;   // columns of the set before a word's
  explicit ColumnSet(int64_t ncol)
      : bits(ncol / 64 + 1, 0), top(ncol / 4096 + 1, 0), before(ncol / 64 + 1, 0) {}
  // lidx[k] = position of ja[k] in the ascending list of the nz columns ja,
  // which is appended to out; returns its length
  int list(const int32_t* ja, int nz, uint16_t* lidx, std::vector<int32_t>& out) {
    uint32_t t0 = UINT32_MAX, t1 = 0;
    for (int k = 0; k < nz; ++k) {
      const uint32_t c = (uint32_t)ja[k], w = c >> 6, t = w >> 6;
      bits[w] |= 1ull << (c & 63);
      top[t] |= 1ull << (w & 63);
      t0 = std::min(t0, t);
      t1 = std::max(t1, t);
    }
    int n = 0;
    each_word(t0, t1, [&](uint32_t w) {
      before[w] = (uint16_t)n;
      for (uint64_t y = bits[w]; y; y &= y - 1) {
        out.push_back((int32_t)(w * 64 + (uint32_t)__builtin_ctzll(y)));
        ++n;
      }
    });
    for (int k = 0; k < nz; ++k) {
      const uint32_t c = (uint32_t)ja[k], w = c >> 6;
      const uint64_t lower = bits[w] & ((1ull << (c & 63)) - 1);
      lidx[k] = (uint16_t)(before[w] + __builtin_popcountll(lower));
    }
    each_word(t0, t1, [&](uint32_t w) { bits[w] = 0; });
    for (uint32_t t = t0; nz && t <= t1; ++t) top[t] = 0;
    return n;
  }
  template <class F>
  void each_word(uint32_t t0, uint32_t t1, F f) const {
    if (t0 > t1) return;
    for (uint32_t t = t0; t <= t1; ++t)
      for (uint64_t x = top[t]; x; x &= x - 1) f(t * 64 + (uint32_t)__builtin_ctzll(x));
  }
};

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
  t.lidx.resize((size_t)ia[nrow]);
  const int64_t nt = (int64_t)t.tile.size();
  const int64_t per = 64;   // tiles a piece of work: some hundred thousand nonzeros
  const int64_t npiece = (nt + per - 1) / per;
  const int64_t nth = std::min<int64_t>(
      npiece, std::min(16u, std::max(1u, std::thread::hardware_concurrency())));
  std::vector<std::vector<int32_t>> cols((size_t)npiece);
  std::atomic<int64_t> next{0};
  on_threads(nth, [&] {
    ColumnSet set(ncol);
    for (int64_t p; (p = next++) < npiece;)
      for (int64_t i = p * per; i < std::min(nt, (p + 1) * per); ++i) {
        Tile& w = t.tile[i];
        uint16_t* l = t.lidx.data() + w.k0;
        if (w.nz > kTileNnz) {
          std::fill(l, l + w.nz, (uint16_t)0);
          continue;
        }
        w.u0 = (int)cols[p].size();
        w.nu = set.list(ja + w.k0, w.nz, l, cols[p]);
      }
  });
  // the pieces' lists after one another
  std::vector<int64_t> base((size_t)npiece + 1, 0);
  for (int64_t p = 0; p < npiece; ++p) base[p + 1] = base[p] + (int64_t)cols[p].size();
  t.ucol.resize((size_t)base[npiece]);
  next = 0;
  on_threads(nth, [&] {
    for (int64_t p; (p = next++) < npiece;) {
      std::copy(cols[p].begin(), cols[p].end(), t.ucol.begin() + base[p]);
      for (int64_t i = p * per; i < std::min(nt, (p + 1) * per); ++i) t.tile[i].u0 += (int)base[p];
    }
  });
  for (const Tile& w : t.tile) t.nwide += w.nu > kTileCols;
}

}  // namespace xg
