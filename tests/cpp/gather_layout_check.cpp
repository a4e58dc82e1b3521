// CPU check of the gather block layouts (xyst_amd/csrc/xg_layout.cpp) with
// boundary faces, and of the tet layouts, at the block sizes of small meshes:
// integer values of edges, face corners and tet corners must reach every node
// exactly once, through the owned sums alone in a gather layout, and every
// index and prefetch bound of the kernels must stay inside its list.
// Input file: int64 npoin, ne, ntri, ntet; int32 p[ne], q[ne], tri[3 ntri],
// tet[4 ntet].
// Arguments: FILE KIND(rhs|cho|tet|rows|gradrows) NODES GATHER, for rows
// (node rows, xg_rows.hpp) the lanes per node instead of GATHER, for gradrows
// (riemann::grad's) the lanes that it has to choose, NODES 0.  NODES 0 of the
// others: the operator's own choice of blocks, which has to be GATHER.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../xyst_amd/csrc/xg_layout.hpp"
#include "../../xyst_amd/csrc/xg_rows.hpp"

#define CHECK(c) do { if (!(c)) { std::fprintf(stderr, "FAIL %s:%d %s\n", __FILE__, __LINE__, #c); std::exit(1); } } while (0)

static int64_t val(int64_t item, int corner) { return (item * 7 + corner * 3) % 1009 - 500; }

// every edge at both ends with that end's sign, every face at its three nodes,
// in input order (one lane: edges from both ends inward)
static void check_rows(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                       const std::vector<int>& tri, int nodes, int lanes, bool grad) {
  std::vector<double> d(3 * p.size());
  for (size_t i = 0; i < d.size(); ++i) d[i] = 1.0 + (double)i;
  xg::RowLayout L;
  std::string err;
  int cap = 700;
  if (grad) {
    int got = 0;
    CHECK(xg::build_grad_rows(npoin, p, q, d, (int64_t)tri.size() / 3, tri.data(), L, got, err) ==
          0);
    CHECK(got == lanes);
    nodes = got == 1 ? xg::kGradNodes : 16;
    cap = got == 1 ? xg::kGradCap : xg::kGradSmallCap;
  } else {
    CHECK(xg::build_rows(npoin, p, q, d, (int64_t)tri.size() / 3, tri.data(), nodes, cap, lanes,
                         L, err) == 0);
  }
  const int per = 64 / lanes;
  std::vector<std::vector<int64_t>> edges(npoin), faces(npoin), ge(npoin), gf(npoin);
  for (size_t e = 0; e < p.size(); ++e) {
    edges[p[e]].push_back(-(int64_t)e - 1);
    edges[q[e]].push_back((int64_t)e + 1);
  }
  for (size_t k = 0; k < tri.size(); ++k) faces[tri[k]].push_back(k);
  if (lanes == 1)
    for (auto& v : edges) {
      std::vector<int64_t> w;
      for (size_t a = 0, b = v.size(); a < b;) {
        w.push_back(v[a++]);
        if (a < b) w.push_back(v[--b]);
      }
      v = w;
    }
  int next = 0;
  for (const auto& B : L.blk) {
    CHECK(B.own0 == next && B.nown > 0 && B.nown <= nodes && B.nloc <= cap);
    next += B.nown;
    CHECK(B.halo_off + B.nloc - B.nown <= (int)L.halo.size());
    auto glob = [&](int l) {
      CHECK(l >= 0 && l < B.nloc);
      return l < B.nown ? B.own0 + l : L.halo[B.halo_off + l - B.nown];
    };
    for (int w = 0; w * per < B.nown; ++w) {
      CHECK(B.wave0 + w < (int)L.wave.size());
      const auto& W = L.wave[B.wave0 + w];
      CHECK(W.e0 + 64 * W.erows <= (int)L.nb.size() && L.dx.size() == L.nb.size());
      CHECK(W.f0 + 64 * W.frows <= (int)L.fab.size());
      for (int k = w * per; k < std::min(B.nown, (w + 1) * per); ++k)
        for (int j = 0;; ++j) {
          const int lane = (k - w * per) * lanes + j % lanes, row = j / lanes;
          const int g = (B.wave0 + w) * 64 + lane;
          const bool has = row < L.deg[g], face = row < L.fdeg[g];
          if (!has && !face) break;
          CHECK((!has || row < W.erows) && (!face || row < W.frows));
          if (has) {
            const size_t at = W.e0 + 64 * (size_t)row + lane;
            const int64_t e = L.eidx[at];
            const bool first = L.dx[at] < 0.0;
            CHECK(L.dx[at] == (first ? -1 : 1) * d[3 * e] &&
                  L.dy[at] == (first ? -1 : 1) * d[3 * e + 1] &&
                  L.dz[at] == (first ? -1 : 1) * d[3 * e + 2]);
            CHECK((first ? p[e] : q[e]) == B.own0 + k);
            CHECK(glob(L.nb[at]) == (first ? q[e] : p[e]));
            ge[B.own0 + k].push_back(first ? -e - 1 : e + 1);
          }
          if (face) {
            const size_t at = W.f0 + 64 * (size_t)row + lane;
            const int64_t f = L.fidx[at];
            const int a = L.fcs[at] >> 16;
            CHECK(glob(L.fab[at] & 0xffff) == tri[3 * f] && glob(L.fab[at] >> 16) == tri[3 * f + 1] &&
                  glob(L.fcs[at] & 0xffff) == tri[3 * f + 2]);
            CHECK(a < 3 && tri[3 * f + a] == B.own0 + k);
            gf[B.own0 + k].push_back(3 * f + a);
          }
        }
    }
  }
  CHECK(next == npoin);
  CHECK(ge == edges && gf == faces);
  std::printf("ok blocks=%zu\n", L.blk.size());
}

int main(int argc, char** argv) {
  CHECK(argc == 5);
  const char* kind = argv[2];
  const int nodes = std::atoi(argv[3]);
  const bool gather = std::atoi(argv[4]) != 0;
  FILE* f = std::fopen(argv[1], "rb");
  CHECK(f);
  int64_t h[4];
  CHECK(std::fread(h, 8, 4, f) == 4);
  const int npoin = (int)h[0];
  std::vector<int> p(h[1]), q(h[1]), tri(3 * h[2]), t32(4 * h[3]);
  CHECK(std::fread(p.data(), 4, p.size(), f) == p.size());
  CHECK(std::fread(q.data(), 4, q.size(), f) == q.size());
  CHECK(std::fread(tri.data(), 4, tri.size(), f) == tri.size());
  CHECK(std::fread(t32.data(), 4, t32.size(), f) == t32.size());
  std::fclose(f);
  if (!std::strcmp(kind, "rows") || !std::strcmp(kind, "gradrows")) {
    check_rows(npoin, p, q, tri, nodes, std::atoi(argv[4]), !std::strcmp(kind, "gradrows"));
    return 0;
  }
  std::string err;
  std::vector<int64_t> want(npoin, 0), got(npoin, -1);
  const bool tets = !std::strcmp(kind, "tet");
  xg::Layout L;
  xg::TetLayout T;
  int cap, slots;
  if (tets) {
    cap = xg::kKozCap;
    slots = xg::kKozPairSlots;
    std::vector<size_t> inp(t32.begin(), t32.end());
    CHECK((nodes ? xg::build_tet_layout(npoin, h[3], inp.data(), nodes, cap, T, err,
                                        xg::kTetsPerPairChunk, gather)
                 : xg::build_kozak_layout(npoin, h[3], inp.data(), T, err)) == 0);
    for (int64_t e = 0; e < h[3]; ++e)
      for (int a = 0; a < 4; ++a) want[t32[e * 4 + a]] += val(t32[e * 4] + t32[e * 4 + 1], a);
  } else {
    const bool cho = !std::strcmp(kind, "cho");
    cap = cho ? xg::kBlockCap : xg::kRhsCap;
    slots = cho ? xg::kChunkSlots : xg::kRhsSlots;
    std::vector<double> d(3 * p.size(), 1.0);
    std::vector<uint8_t> sym(3 * h[2], 1);
    CHECK((nodes ? xg::build_layout(npoin, p, q, d, h[2], tri.data(), sym.data(), nodes, cap,
                                    slots, L, err, gather, !cho)
           : cho ? xg::build_cho_layout(npoin, p, q, d, h[2], tri.data(), L, err)
                 : xg::build_rhs_layout(npoin, p, q, d, h[2], tri.data(), sym.data(), L, err)) ==
          0);
    for (size_t e = 0; e < p.size(); ++e) {
      want[p[e]] -= val(e, 0);
      want[q[e]] += val(e, 0);
    }
    for (int64_t t = 0; t < h[2]; ++t)
      for (int a = 0; a < 3; ++a) want[tri[t * 3 + a]] += val(t, 1 + a);
  }
  const auto& blk = tets ? T.blk : L.blk;
  const auto& chunks = tets ? T.chunks : L.chunks;
  const auto& halo = tets ? T.halo : L.halo;
  const auto& tend = tets ? T.tend : L.tend;
  const auto& ents = tets ? T.entries : L.entries;
  const int nslot = tets ? T.nslot : L.nslot;
  const auto& fxn = tets ? T.fx_node : L.fx_node;
  const auto& fxo = tets ? T.fx_off : L.fx_off;
  const auto& fxs = tets ? T.fx_slot : L.fx_slot;
  if (gather) CHECK(nslot == 0 && fxn.empty());
  std::vector<int64_t> S(nslot, 0);
  for (const auto& B : blk) {
    CHECK(B.nown > 0 && (!nodes || B.nown <= nodes) && B.nloc <= cap && B.nloc <= slots);
    CHECK(gather ? B.slot0 == -1 : B.slot0 + B.nloc - B.nown <= nslot);
    std::vector<int> glob(B.nloc);
    for (int i = 0; i < B.nloc; ++i) {
      glob[i] = i < B.nown ? B.own0 + i : halo[B.halo_off + i - B.nown];
      CHECK(glob[i] >= 0 && glob[i] < npoin);
    }
    std::vector<int64_t> acc(B.nloc, 0), F(slots);
    for (int ch = B.chunk0; ch < B.chunk1; ++ch) {
      const auto& C = chunks[ch];
      const int per = C.kind == 0 ? 2 : C.kind == 1 ? 3 : 4;
      CHECK(C.count > 0 && C.count * (C.kind == 0 ? 1 : per) <= slots);
      CHECK(C.ent_off + C.count * per <= (int)ents.size());   // the prefetch
      CHECK(C.tend_off + B.nloc <= (int)tend.size());
      for (int t = 0; t < C.count; ++t) {
        const int i = C.first + t;
        if (C.kind == 0) {
          const int a = L.elpq[i] & 0xffff, b = L.elpq[i] >> 16;
          CHECK(a < B.nloc && b < B.nloc);
          CHECK(glob[a] == p[L.eidx[i]] && glob[b] == q[L.eidx[i]]);
          F[t] = val(L.eidx[i], 0);
        } else if (C.kind == 1) {
          const int N[3] = {(int)(L.fab[i] & 0xffff), (int)(L.fab[i] >> 16),
                            (int)(L.fcs[i] & 0xffff)};
          for (int a = 0; a < 3; ++a) {
            CHECK(N[a] < B.nloc && glob[N[a]] == tri[L.fidx[i] * 3 + a]);
            F[3 * t + a] = val(L.fidx[i], 1 + a);
          }
        } else {
          const int N[4] = {(int)(T.tab[i] & 0xffff), (int)(T.tab[i] >> 16),
                            (int)(T.tcd[i] & 0xffff), (int)(T.tcd[i] >> 16)};
          for (int a = 0; a < 4; ++a) CHECK(N[a] < B.nloc && glob[N[a]] == T.tglob[i * 4 + a]);
          for (int a = 0; a < 4; ++a) F[4 * t + a] = val(glob[N[0]] + glob[N[1]], a);
        }
      }
      const int filled = C.kind == 0 ? C.count : per * C.count;
      for (int n = 0; n < B.nloc; ++n) {
        const int e0 = n ? tend[C.tend_off + n - 1] : 0, e1 = tend[C.tend_off + n];
        CHECK(e0 <= e1 && e1 <= C.count * per);
        if (gather && n >= B.nown) CHECK(e0 == e1);
        for (int j = e0; j < e1; ++j) {
          const int v = ents[C.ent_off + j], s = tets ? v : v & 0x3ff;
          CHECK(s < filled);
          acc[n] += !tets && (v & 0x8000) ? -F[s] : F[s];
        }
      }
    }
    for (int n = 0; n < B.nloc; ++n) {
      if (n < B.nown) got[B.own0 + n] = acc[n];
      else if (!gather) S[B.slot0 + n - B.nown] = acc[n];
    }
  }
  for (size_t i = 0; i < fxn.size(); ++i)
    for (int k = fxo[i]; k < fxo[i + 1]; ++k) got[fxn[i]] += S[fxs[k]];
  for (int n = 0; n < npoin; ++n) CHECK(got[n] == want[n]);
  std::printf("ok blocks=%zu\n", blk.size());
  return 0;
}
