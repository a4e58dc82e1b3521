// Rounding error of the node sums of D (u_p + u_q) in the order of the node
// rows (xyst_amd/csrc/xg_layout.cpp, build_rows) and in input order, against
// sums with 11 more bits, for several fields.
// Input file: int64 npoin, ne, nfield; int32 p[ne], q[ne]; double d[3 ne],
// u[nfield npoin].  Argument: FILE LANES.  Prints the two errors, relative to
// the result (2-norms over all sums).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../xyst_amd/csrc/xg_layout.hpp"
#include "../../xyst_amd/csrc/xg_rows.hpp"

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  FILE* f = std::fopen(argv[1], "rb");
  int64_t h[3];
  if (!f || std::fread(h, 8, 3, f) != 3) return 2;
  const int npoin = (int)h[0], lanes = std::atoi(argv[2]);
  std::vector<int> p(h[1]), q(h[1]);
  std::vector<double> d(3 * h[1]), u(h[0] * h[2]);
  if (std::fread(p.data(), 4, p.size(), f) != p.size() ||
      std::fread(q.data(), 4, q.size(), f) != q.size() ||
      std::fread(d.data(), 8, d.size(), f) != d.size() ||
      std::fread(u.data(), 8, u.size(), f) != u.size())
    return 2;
  std::fclose(f);
  xg::RowLayout L;
  std::string err;
  const int nodes = lanes == 1 ? xg::kGradNodes : 16, per = 64 / lanes;
  if (xg::build_rows(npoin, p, q, d, 0, nullptr, nodes, xg::kGradCap, lanes, L, err)) return 1;
  double e[2] = {0.0, 0.0}, norm = 0.0;
  for (int64_t k = 0; k < h[2]; ++k) {
    const double* v = u.data() + k * npoin;
    for (int j = 0; j < 3; ++j) {
      std::vector<double> in(npoin, 0.0);
      std::vector<long double> exact(npoin, 0.0L);
      for (int64_t i = 0; i < h[1]; ++i) {
        const long double x = (long double)d[3 * i + j] * ((long double)v[p[i]] + v[q[i]]);
        exact[p[i]] -= x;
        exact[q[i]] += x;
        in[p[i]] = std::fma(-d[3 * i + j], v[p[i]] + v[q[i]], in[p[i]]);
        in[q[i]] = std::fma(d[3 * i + j], v[p[i]] + v[q[i]], in[q[i]]);
      }
      const std::vector<double>& D = j == 0 ? L.dx : j == 1 ? L.dy : L.dz;
      for (const auto& B : L.blk)
        for (int n = 0; n < B.nown; ++n) {
          const auto& W = L.wave[B.wave0 + n / per];
          double acc[64] = {};
          for (int l = 0; l < lanes; ++l) {
            const int lane = n % per * lanes + l;
            for (int i = 0; i < L.deg[(B.wave0 + n / per) * 64 + lane]; ++i) {
              const size_t at = W.e0 + 64 * (size_t)i + lane;
              const int m = L.nb[at];
              const int g = m < B.nown ? B.own0 + m : L.halo[B.halo_off + m - B.nown];
              acc[l] = std::fma(D[at], v[B.own0 + n] + v[g], acc[l]);
            }
          }
          for (int o = 1; o < lanes; o <<= 1)
            for (int l = 0; l < lanes; l += 2 * o) acc[l] += acc[l + o];
          const long double x = exact[B.own0 + n];
          const double a = (double)(acc[0] - x), b = (double)(in[B.own0 + n] - x);
          e[0] += a * a;
          e[1] += b * b;
          norm += (double)(x * x);
        }
    }
  }
  std::printf("%.4e %.4e\n", std::sqrt(e[0] / norm), std::sqrt(e[1] / norm));
  return 0;
}
