// Device layout of the edge-based operators (host side).
//
// rhs: nodes are grouped into blocks of consecutive ids; a block owns the
// edges and boundary faces whose smallest node id lies in it, and all nodes
// those touch that lie beyond the block are its halo.  One workgroup per
// block accumulates the block's nodal sums in LDS: the block's work items
// (edges, or boundary faces) are cut into chunks of at most chunk_slots
// flux slots; a chunk's fluxes go to LDS, then every node the chunk touches
// sums its slots in a fixed order.  Owned nodes are written directly; halo
// partial sums go to slots that a fix-up pass adds to their owners in block
// order.  Every sum is therefore taken in an order fixed here: results are
// bitwise reproducible, without atomics.
//
// The nodes a block touches are staged in LDS (primitive state, gradients,
// coordinates), so a chunk's flux evaluations read LDS only; a thread owns one
// local node and keeps its running sum in registers.
//
// The chorin operators use blocks of up to kBlockCap nodes with 1024-slot
// chunks (each node thread gathers the terms of the chunk edges that touch
// it); riemann::rhs builds its own layout of kRhsCap-node blocks and 512-slot
// chunks, two workgroups per CU.  On small meshes both use gather blocks (see
// build_layout): edges and faces between two blocks are evaluated in both, so
// no block leaves partial sums behind.  riemann::grad, whose per-edge work is
// small, uses node rows (build_rows).
//
// The layout is fastest when node ids are block-contiguous and spatially
// compact (xg_mesh_block_order), but is correct for any numbering.
#include "xg_layout.hpp"
#include "xg_rows.hpp"

#include <algorithm>
#include <cstring>
#include <numeric>

namespace xg {

// Node blocks of consecutive ids for the node graph given as neighbour lists
// (uoff/up: the neighbours with larger ids of every node, or all neighbours
// for a gather layout), grown while owned <= block_nodes and owned + halo <=
// block_cap; bstart receives the block starts followed by npoin.
static int partition_blocks(int npoin, const std::vector<int64_t>& uoff,
                            const std::vector<int>& up, int block_nodes,
                            int block_cap, std::vector<int>& bstart,
                            std::string& err) {
  bstart.clear();
  std::vector<int> mark(npoin, -1);   // block id that has node in its halo
  int s = 0, b = 0;
  while (s < npoin) {
    int nown = 0, nhalo = 0, end = s;
    while (end < npoin && nown < block_nodes) {
      // adding node `end`: it leaves the halo if it was there
      // (a neighbour outside [s, end] is halo: beyond end, or before s)
      int add = 0;
      for (int64_t k = uoff[end]; k < uoff[end + 1]; ++k)
        if (mark[up[k]] != b && (up[k] > end || up[k] < s)) ++add;
      int was_halo = mark[end] == b ? 1 : 0;
      if (nown > 0 && nown + 1 + nhalo - was_halo + add > block_cap) break;
      for (int64_t k = uoff[end]; k < uoff[end + 1]; ++k)
        if (mark[up[k]] != b && (up[k] > end || up[k] < s)) { mark[up[k]] = b; ++nhalo; }
      if (was_halo) { --nhalo; mark[end] = -2; }
      ++nown; ++end;
    }
    if (nown + nhalo > block_cap) {
      err = "layout: a single node has more neighbours than the block capacity";
      return XG_EUNSUPPORTED;
    }
    bstart.push_back(s);
    s = end; ++b;
  }
  bstart.push_back(npoin);
  return XG_OK;
}

// Upper-neighbour lists of the graph with edges (p[e], q[e]).
static void upper_lists(int npoin, const std::vector<int>& p,
                        const std::vector<int>& q, std::vector<int64_t>& uoff,
                        std::vector<int>& up) {
  const int64_t ne = (int64_t)p.size();
  std::vector<int> ucnt(npoin + 1, 0);
  for (int64_t e = 0; e < ne; ++e) ++ucnt[std::min(p[e], q[e]) + 1];
  uoff.assign(npoin + 1, 0);
  for (int i = 0; i < npoin; ++i) uoff[i + 1] = uoff[i] + ucnt[i + 1];
  up.resize(uoff[npoin]);
  std::vector<int64_t> pos(uoff.begin(), uoff.end() - 1);
  for (int64_t e = 0; e < ne; ++e)
    up[pos[std::min(p[e], q[e])]++] = std::max(p[e], q[e]);
}

// Neighbour lists in both directions (CSR over all nodes).
static void full_lists(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                       std::vector<int64_t>& off, std::vector<int>& nb) {
  const int64_t ne = (int64_t)p.size();
  off.assign(npoin + 1, 0);
  for (int64_t e = 0; e < ne; ++e) {
    ++off[p[e] + 1];
    ++off[q[e] + 1];
  }
  for (int i = 0; i < npoin; ++i) off[i + 1] += off[i];
  nb.resize(off[npoin]);
  std::vector<int64_t> pos(off.begin(), off.end() - 1);
  for (int64_t e = 0; e < ne; ++e) {
    nb[pos[p[e]]++] = q[e];
    nb[pos[q[e]]++] = p[e];
  }
}

// Sorts items by key(item), ties by item; the keys are formed once, in `keyed`.
template <class Key>
static void sort_by_key(std::vector<int64_t>& items,
                        std::vector<std::pair<uint64_t, int64_t>>& keyed, Key key) {
  keyed.clear();
  for (int64_t i : items) keyed.emplace_back(key(i), i);
  std::sort(keyed.begin(), keyed.end());
  for (size_t k = 0; k < items.size(); ++k) items[k] = keyed[k].second;
}

// Appends a chunk's entries (local node, slot | sign) grouped by node, each
// node's in the order given, and every local node's entry end.
static void group_entries(const std::vector<std::pair<int, uint16_t>>& ent, int nloc,
                          std::vector<uint16_t>& entries, std::vector<uint16_t>& tend) {
  const size_t e0 = entries.size(), t0 = tend.size();
  std::vector<int> pos(nloc + 1, 0);
  for (const auto& e : ent) ++pos[e.first + 1];
  for (int n = 0; n < nloc; ++n) pos[n + 1] += pos[n];
  tend.resize(t0 + nloc);
  for (int n = 0; n < nloc; ++n) tend[t0 + n] = (uint16_t)pos[n + 1];
  entries.resize(e0 + ent.size());
  for (const auto& e : ent) entries[e0 + pos[e.first]++] = e.second;
}

// Cuts a block's items (edges or tets, in local order) into chunks of at most
// `slots`, spreading the items of a node over the chunks: a chunk's node sums
// take as long as the node with the most entries in it.  In local order alone
// a node's items fall into one or two chunks (kozak::rhs on 96^3 240 us, 183
// spread; the KozCG step 1253 -> 1013; riemann::rhs on 128^3 470 -> 444).  The
// chorin operators keep local order (spread = false): chorin::rhs on 64^3 took
// 59.7 us spread instead of 62.6, but neighbours that nearly cancel were added
// apart, and the error against exact sums grew from 4.2e-15 to 5.7e-15 (the
// others' did not).
// Greedy, in item order: the chunk where the item's nodes have the fewest
// entries so far, then the emptiest.  ends(i, out): the local nodes that item
// i adds to; returns how many.  The items of a chunk keep their order.
template <class Ends>
static std::vector<std::vector<int64_t>> spread_chunks(const std::vector<int64_t>& items,
                                                       int slots, int nloc, Ends ends) {
  const size_t n = items.size();
  const size_t nch = (n + slots - 1) / slots;
  std::vector<std::vector<int64_t>> out(nch);
  if (nch <= 1) {
    if (nch) out[0] = items;
    return out;
  }
  // chunks of equal size, in whole waves
  const size_t room = std::min<size_t>(slots, ((n + nch - 1) / nch + 63) / 64 * 64);
  std::vector<uint16_t> cnt(nch * (size_t)nloc, 0);
  for (int64_t it : items) {
    int node[4];
    const int k = ends(it, node);
    size_t best = nch;
    int bmax = 0, bsum = 0;
    for (size_t c = 0; c < nch; ++c) {
      if (out[c].size() >= room) continue;
      int mx = 0, sum = 0;
      for (int a = 0; a < k; ++a) {
        const int v = cnt[c * nloc + node[a]];
        mx = std::max(mx, v);
        sum += v;
      }
      if (best == nch || mx < bmax || (mx == bmax && sum < bsum) ||
          (mx == bmax && sum == bsum && out[c].size() < out[best].size())) {
        best = c;
        bmax = mx;
        bsum = sum;
      }
    }
    out[best].push_back(it);
    for (int a = 0; a < k; ++a) ++cnt[best * nloc + node[a]];
  }
  return out;
}

int build_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                 const std::vector<double>& d, int64_t ntri, const int* tri,
                 const uint8_t* besym, int block_nodes, int block_cap,
                 int chunk_slots, Layout& L, std::string& err, bool gather, bool spread) {
  const int64_t ne = (int64_t)p.size();
  L = Layout();
  if (chunk_slots < 3 || chunk_slots > kChunkSlots) {
    err = "layout: chunk size out of range";
    return XG_EINVAL;
  }
  L.npoin = npoin;
  // neighbour lists for halo tracking: by the smaller end (a block's halo
  // lies beyond it), or both ways for a gather layout
  std::vector<int64_t> uoff;
  std::vector<int> up;
  if (gather) {
    // the faces' edges too: a block holds the nodes of every face it takes
    std::vector<int> pf(p), qf(q);
    for (int64_t f = 0; f < ntri; ++f)
      for (int a = 0; a < 3; ++a) {
        pf.push_back(tri[f * 3 + a]);
        qf.push_back(tri[f * 3 + (a + 1) % 3]);
      }
    full_lists(npoin, pf, qf, uoff, up);
  } else {
    upper_lists(npoin, p, q, uoff, up);
  }
  // (boundary faces are tet faces: their nodes are edge neighbours of the
  // face's smallest node, so the upper lists already cover them)
  std::vector<int> bstart;
  int prc = partition_blocks(npoin, uoff, up, block_nodes, block_cap, bstart, err);
  if (prc) return prc;
  const int nblk = (int)bstart.size() - 1;
  std::vector<int> blk_of(npoin);
  for (int b = 0; b < nblk; ++b)
    for (int i = bstart[b]; i < bstart[b + 1]; ++i) blk_of[i] = b;
  // work items per block (gather: an edge or face belongs to the blocks of
  // all its nodes)
  std::vector<std::vector<int64_t>> bedges(nblk), bfaces(nblk);
  for (int64_t e = 0; e < ne; ++e) {
    const int b0 = blk_of[std::min(p[e], q[e])], b1 = blk_of[std::max(p[e], q[e])];
    bedges[b0].push_back(e);
    if (gather && b1 != b0) bedges[b1].push_back(e);
  }
  for (int64_t f = 0; f < ntri; ++f) {
    const int* N = tri + f * 3;
    if (!gather) {
      bfaces[blk_of[std::min(N[0], std::min(N[1], N[2]))]].push_back(f);
      continue;
    }
    const int b[3] = {blk_of[N[0]], blk_of[N[1]], blk_of[N[2]]};
    for (int a = 0; a < 3; ++a)
      if ((a < 1 || b[a] != b[0]) && (a < 2 || b[a] != b[1])) bfaces[b[a]].push_back(f);
  }
  size_t nitem = 0, nface = 0;   // an edge of two gather blocks is in both
  for (int b = 0; b < nblk; ++b) {
    nitem += bedges[b].size();
    nface += bfaces[b].size();
  }
  for (auto* v : {&L.dx, &L.dy, &L.dz}) v->reserve(nitem);
  for (auto* v : {&L.ep, &L.eq}) v->reserve(nitem);
  L.elpq.reserve(nitem);
  L.eidx.reserve(nitem);
  L.entries.reserve(2 * nitem + 3 * nface + 3 * (size_t)chunk_slots);
  L.blk.resize(nblk);
  std::vector<std::vector<std::pair<int,int>>> fix(npoin);   // node -> (block, slot)
  int nslot = 0;
  std::vector<int> local(npoin, -1);
  std::vector<std::pair<uint64_t, int64_t>> keyed;
  for (int b = 0; b < nblk; ++b) {
    Block& B = L.blk[b];
    B.own0 = bstart[b];
    B.nown = bstart[b + 1] - bstart[b];
    // halo: nodes touched by owned items outside the block, ascending
    std::vector<int> halo;
    auto touch = [&](int m) {
      if ((m >= bstart[b + 1] || m < bstart[b]) && local[m] != -2) {
        local[m] = -2;
        halo.push_back(m);
      }
    };
    for (int64_t e : bedges[b])
      for (int m : {p[e], q[e]}) touch(m);
    for (int64_t f : bfaces[b])
      for (int a = 0; a < 3; ++a) touch(tri[f * 3 + a]);
    std::sort(halo.begin(), halo.end());
    B.nloc = B.nown + (int)halo.size();
    if (B.nloc > block_cap) {
      err = "layout: block exceeds LDS capacity";
      return XG_EUNSUPPORTED;
    }
    B.halo_off = (int)L.halo.size();
    B.slot0 = gather ? -1 : nslot;
    for (size_t h = 0; h < halo.size(); ++h) {
      L.halo.push_back(halo[h]);
      if (!gather) fix[halo[h]].emplace_back(b, nslot + (int)h);
    }
    if (!gather) nslot += (int)halo.size();
    for (int i = 0; i < B.nown; ++i) local[B.own0 + i] = i;
    for (size_t h = 0; h < halo.size(); ++h) local[halo[h]] = B.nown + (int)h;
    // edges ordered by (smaller local end, larger local end) for locality
    auto& E = bedges[b];
    sort_by_key(E, keyed, [&](int64_t e) {
      const uint64_t a = local[p[e]], c = local[q[e]];
      return (std::min(a, c) << 32) | std::max(a, c);
    });
    B.chunk0 = (int)L.chunks.size();
    // chunk builder: entries (local node, slot | sign) grouped by node, with
    // a dense table of per-node entry ends over all nloc local nodes
    auto emit = [&](int kind, int64_t first, int count,
                    const std::vector<std::pair<int, uint16_t>>& ent) {
      Chunk C;
      C.kind = kind;
      C.first = (int)first;
      C.count = count;
      C.tend_off = (int)L.tend.size();
      C.ent_off = (int)L.entries.size();
      group_entries(ent, B.nloc, L.entries, L.tend);
      L.chunks.push_back(C);
    };
    std::vector<std::vector<int64_t>> parts;
    if (spread)
      parts = spread_chunks(E, chunk_slots, B.nloc, [&](int64_t e, int* node) {
        int k = 0;
        for (int m : {local[p[e]], local[q[e]]})
          if (!gather || m < B.nown) node[k++] = m;
        return k;
      });
    else
      for (size_t i0 = 0; i0 < E.size(); i0 += (size_t)chunk_slots)
        parts.emplace_back(E.begin() + i0,
                           E.begin() + std::min(E.size(), i0 + (size_t)chunk_slots));
    for (const auto& C : parts) {
      std::vector<std::pair<int, uint16_t>> ent;
      for (size_t i = 0; i < C.size(); ++i) {
        int64_t e = C[i];
        uint16_t slot = (uint16_t)i;
        // R(p) -= f, R(q) += f (gather: owned ends only)
        if (!gather || local[p[e]] < B.nown)
          ent.emplace_back(local[p[e]], (uint16_t)(slot | 0x8000));
        if (!gather || local[q[e]] < B.nown) ent.emplace_back(local[q[e]], slot);
      }
      emit(0, (int64_t)L.elpq.size(), (int)C.size(), ent);
      for (int64_t e : C) {
        L.elpq.push_back((uint32_t)local[p[e]] | ((uint32_t)local[q[e]] << 16));
        L.ep.push_back(p[e]);
        L.eq.push_back(q[e]);
        L.eidx.push_back(e);
        L.dx.push_back(d[e * 3 + 0]);
        L.dy.push_back(d[e * 3 + 1]);
        L.dz.push_back(d[e * 3 + 2]);
      }
    }
    auto& F = bfaces[b];
    const int fmax = chunk_slots / 3;
    for (size_t i0 = 0; i0 < F.size(); i0 += fmax) {
      size_t i1 = std::min(F.size(), i0 + (size_t)fmax);
      std::vector<std::pair<int, uint16_t>> ent;
      for (size_t i = i0; i < i1; ++i) {
        int64_t f = F[i];
        for (int a = 0; a < 3; ++a)
          if (!gather || local[tri[f * 3 + a]] < B.nown)
            ent.emplace_back(local[tri[f * 3 + a]], (uint16_t)(3 * (i - i0) + a));
      }
      emit(1, (int64_t)L.fab.size(), (int)(i1 - i0), ent);
      for (size_t i = i0; i < i1; ++i) {
        int64_t f = F[i];
        uint32_t sym = (besym[f * 3] ? 1u : 0u) | (besym[f * 3 + 1] ? 2u : 0u) |
                       (besym[f * 3 + 2] ? 4u : 0u);
        L.fab.push_back((uint32_t)local[tri[f * 3]] | ((uint32_t)local[tri[f * 3 + 1]] << 16));
        L.fcs.push_back((uint32_t)local[tri[f * 3 + 2]] | (sym << 16));
        for (int a = 0; a < 3; ++a) L.fglob.push_back(tri[f * 3 + a]);
        L.fidx.push_back(f);
      }
    }
    B.chunk1 = (int)L.chunks.size();
    for (int i = 0; i < B.nown; ++i) local[B.own0 + i] = -1;
    for (size_t h = 0; h < halo.size(); ++h) local[halo[h]] = -1;
  }
  L.nslot = nslot;
  // The block kernels prefetch a chunk's entries with a bound of 2 (edges)
  // or 3 (faces) entries per item.  A gather chunk holds fewer (only owned
  // ends), so that bound can reach past the last chunk: pad the list so the
  // prefetch stays inside the buffer.  The padding is never summed.
  L.entries.resize(L.entries.size() + 3 * (size_t)chunk_slots, 0);
  // fix-up lists: nodes receiving halo partials, slots in block order
  L.fx_off.push_back(0);
  for (int n = 0; n < npoin; ++n) {
    if (fix[n].empty()) continue;
    L.fx_node.push_back(n);
    for (auto& bs : fix[n]) L.fx_slot.push_back(bs.second);
    L.fx_off.push_back((int)L.fx_slot.size());
  }
  return XG_OK;
}

int build_rows(int npoin, const std::vector<int>& p, const std::vector<int>& q,
               const std::vector<double>& d, int64_t ntri, const int* tri, int block_nodes,
               int cap, int lanes, RowLayout& L, std::string& err) {
  L = RowLayout();
  const int64_t ne = (int64_t)p.size();
  if (lanes < 1 || 64 % lanes || cap > 65535) {
    err = "rows: bad lanes or capacity";
    return XG_EINVAL;
  }
  // the edges of every node, in input order; its faces
  std::vector<int64_t> off(npoin + 1, 0), foff(npoin + 1, 0);
  for (int64_t e = 0; e < ne; ++e) {
    ++off[p[e] + 1];
    ++off[q[e] + 1];
  }
  for (int64_t k = 0; k < 3 * ntri; ++k) ++foff[tri[k] + 1];
  for (int i = 0; i < npoin; ++i) {
    off[i + 1] += off[i];
    foff[i + 1] += foff[i];
  }
  std::vector<int64_t> inc(off[npoin]), finc(foff[npoin]);
  {
    std::vector<int64_t> pos(off.begin(), off.end() - 1);
    for (int64_t e = 0; e < ne; ++e) {
      inc[pos[p[e]]++] = e;
      inc[pos[q[e]]++] = e;
    }
    pos.assign(foff.begin(), foff.end() - 1);
    for (int64_t k = 0; k < 3 * ntri; ++k) finc[pos[tri[k]]++] = k;
  }
  // neighbours of every node (of its faces too) for the partition
  std::vector<int64_t> uoff(npoin + 1, 0);
  std::vector<int> up;
  up.reserve(inc.size() + 2 * finc.size());
  for (int i = 0; i < npoin; ++i) {
    for (int64_t k = off[i]; k < off[i + 1]; ++k)
      up.push_back(p[inc[k]] == i ? q[inc[k]] : p[inc[k]]);
    for (int64_t k = foff[i]; k < foff[i + 1]; ++k) {
      const int* N = tri + finc[k] / 3 * 3;
      for (int a = 0; a < 3; ++a)
        if (N[a] != i) up.push_back(N[a]);
    }
    uoff[i + 1] = (int64_t)up.size();
  }
  std::vector<int> bstart;
  int rc = partition_blocks(npoin, uoff, up, block_nodes, cap, bstart, err);
  if (rc) return rc;
  const int nblk = (int)bstart.size() - 1;
  std::vector<int> local(npoin, -1);
  L.blk.resize(nblk);
  for (int b = 0; b < nblk; ++b) {
    RowBlock& B = L.blk[b];
    const int s = bstart[b], e = bstart[b + 1];
    B.own0 = s;
    B.nown = e - s;
    B.halo_off = (int)L.halo.size();
    std::vector<int> halo;
    for (int i = s; i < e; ++i)
      for (int64_t k = uoff[i]; k < uoff[i + 1]; ++k)
        if (up[k] < s || up[k] >= e) halo.push_back(up[k]);
    std::sort(halo.begin(), halo.end());
    halo.erase(std::unique(halo.begin(), halo.end()), halo.end());
    L.halo.insert(L.halo.end(), halo.begin(), halo.end());
    B.nloc = B.nown + (int)halo.size();
    if (B.nloc > cap) {
      err = "rows: block exceeds its capacity";
      return XG_EUNSUPPORTED;
    }
    for (int i = s; i < e; ++i) local[i] = i - s;
    for (size_t h = 0; h < halo.size(); ++h) local[halo[h]] = B.nown + (int)h;
    B.wave0 = (int)L.wave.size();
    const int per = 64 / lanes;   // nodes of a wave
    for (int w0 = 0; w0 < B.nown; w0 += per) {
      RowWave W;
      int64_t most = 0, fmost = 0;
      for (int k = w0; k < std::min(B.nown, w0 + per); ++k) {
        most = std::max(most, off[s + k + 1] - off[s + k]);
        fmost = std::max(fmost, foff[s + k + 1] - foff[s + k]);
      }
      W.erows = (int)((most + lanes - 1) / lanes);
      W.frows = (int)((fmost + lanes - 1) / lanes);
      if (W.erows > 65535 || W.frows > 65535) {
        err = "rows: too many edges at a node";
        return XG_EUNSUPPORTED;
      }
      W.e0 = (int)L.nb.size();
      W.f0 = (int)L.fab.size();
      if (L.nb.size() + 64 * (size_t)W.erows >= (1u << 31)) {
        err = "rows: too many edges";
        return XG_EUNSUPPORTED;
      }
      L.wave.push_back(W);
      L.nb.resize(W.e0 + 64 * (size_t)W.erows, 0);
      L.dx.resize(L.nb.size(), 0.0);
      L.dy.resize(L.nb.size(), 0.0);
      L.dz.resize(L.nb.size(), 0.0);
      L.eidx.resize(L.nb.size(), -1);
      L.fab.resize(W.f0 + 64 * (size_t)W.frows, 0);
      L.fcs.resize(L.fab.size(), 0);
      L.fidx.resize(L.fab.size(), -1);
      const size_t g0 = L.deg.size();
      L.deg.resize(g0 + 64, 0);
      L.fdeg.resize(g0 + 64, 0);
      for (int k = w0; k < std::min(B.nown, w0 + per); ++k) {
        const int i = s + k, l0 = (k - w0) * lanes;
        // one lane: from both ends inward (the input's edges ascend by
        // neighbour), so that opposite neighbours, whose terms nearly cancel,
        // are added one after the other: the error of the gradient's sums
        // on 49^3 is 3.5e-16 of the result, ascending 5.5e-16 (four lanes, a
        // quarter of the terms each: 4.1e-16 so, ascending 3.8e-16)
        const int64_t ndeg = off[i + 1] - off[i];
        for (int64_t j = 0; j < ndeg; ++j) {
          const int64_t o = lanes > 1 ? j : j & 1 ? ndeg - 1 - j / 2 : j / 2;
          const int64_t ed = inc[off[i] + o];
          const int lane = l0 + (int)(j % lanes);
          const size_t at = W.e0 + 64 * (size_t)(j / lanes) + lane;
          const bool first = p[ed] == i;
          const double sg = first ? -1.0 : 1.0;
          L.nb[at] = (uint16_t)local[first ? q[ed] : p[ed]];
          L.dx[at] = sg * d[ed * 3];
          L.dy[at] = sg * d[ed * 3 + 1];
          L.dz[at] = sg * d[ed * 3 + 2];
          L.eidx[at] = ed;
          ++L.deg[g0 + lane];
        }
        for (int64_t j = 0; j < foff[i + 1] - foff[i]; ++j) {
          const int64_t f = finc[foff[i] + j] / 3, a = finc[foff[i] + j] % 3;
          const int lane = l0 + (int)(j % lanes);
          const size_t at = W.f0 + 64 * (size_t)(j / lanes) + lane;
          const int* N = tri + f * 3;
          L.fab[at] = (uint32_t)local[N[0]] | ((uint32_t)local[N[1]] << 16);
          L.fcs[at] = (uint32_t)local[N[2]] | ((uint32_t)a << 16);
          L.fidx[at] = f;
          ++L.fdeg[g0 + lane];
        }
      }
    }
    for (int i = s; i < e; ++i) local[i] = -1;
    for (int h : halo) local[h] = -1;
  }
  return XG_OK;
}

int build_grad_rows(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                    const std::vector<double>& d, int64_t ntri, const int* tri, RowLayout& L,
                    int& lanes, std::string& err) {
  if (npoin <= kSmallGrad) {
    std::string why;
    lanes = 4;
    const int rc = build_rows(npoin, p, q, d, ntri, tri, 16, kGradSmallCap, lanes, L, why);
    if (rc != XG_EUNSUPPORTED) {
      if (rc) err = why;
      return rc;
    }
  }
  lanes = 1;
  return build_rows(npoin, p, q, d, ntri, tri, kGradNodes, kGradCap, lanes, L, err);
}

// kozak::rhs layout: blocks as above on the tets' node graph; a block owns the
// tets whose smallest node lies in it.  Tets are ordered by their local node
// ids and cut into chunks of tets_per_chunk; slot 4*i + a holds corner a of
// chunk tet i, and every local node sums its slots in slot order.
int build_tet_layout(int npoin, int64_t ntet, const size_t* inpoel,
                     int block_nodes, int block_cap, TetLayout& L,
                     std::string& err, int tets_per_chunk, bool gather) {
  if (tets_per_chunk < 1 || 4 * tets_per_chunk > 32768) {
    err = "kozak layout: bad chunk size";
    return XG_EINVAL;
  }
  static const int kTetEdge[6][2] = {{0,1},{1,2},{2,0},{0,3},{1,3},{2,3}};
  L = TetLayout();
  L.npoin = npoin;
  std::vector<int> p, q;
  p.reserve(ntet * 6);
  q.reserve(ntet * 6);
  for (int64_t e = 0; e < ntet; ++e)
    for (int k = 0; k < 6; ++k) {
      size_t a = inpoel[e * 4 + kTetEdge[k][0]], b = inpoel[e * 4 + kTetEdge[k][1]];
      if (a >= (size_t)npoin || b >= (size_t)npoin || a == b) {
        err = "kozak layout: bad tet connectivity";
        return XG_EINVAL;
      }
      p.push_back((int)a);
      q.push_back((int)b);
    }
  // unique edges suffice for the partition (duplicates only repeat marks)
  std::vector<int64_t> uoff;
  std::vector<int> up;
  if (gather)
    full_lists(npoin, p, q, uoff, up);
  else
    upper_lists(npoin, p, q, uoff, up);
  {  // compact duplicates
    std::vector<int64_t> o2(npoin + 1, 0);
    std::vector<int> u2, seen(npoin, -1);
    u2.reserve(up.size() / 2);
    for (int i = 0; i < npoin; ++i) {
      for (int64_t k = uoff[i]; k < uoff[i + 1]; ++k)
        if (seen[up[k]] != i) {
          seen[up[k]] = i;
          u2.push_back(up[k]);
        }
      o2[i + 1] = (int64_t)u2.size();
    }
    uoff.swap(o2);
    up.swap(u2);
  }
  std::vector<int>().swap(p);
  std::vector<int>().swap(q);
  std::vector<int> bstart;
  int prc = partition_blocks(npoin, uoff, up, block_nodes, block_cap, bstart, err);
  if (prc) return prc;
  const int nblk = (int)bstart.size() - 1;
  std::vector<int> blk_of(npoin);
  for (int b = 0; b < nblk; ++b)
    for (int i = bstart[b]; i < bstart[b + 1]; ++i) blk_of[i] = b;
  std::vector<std::vector<int64_t>> btets(nblk);
  for (int64_t e = 0; e < ntet; ++e) {
    const size_t* N = inpoel + e * 4;
    if (!gather) {
      btets[blk_of[std::min(std::min(N[0], N[1]), std::min(N[2], N[3]))]].push_back(e);
      continue;
    }
    for (int a = 0; a < 4; ++a) {
      bool first = true;
      for (int c = 0; c < a; ++c) first = first && blk_of[N[c]] != blk_of[N[a]];
      if (first) btets[blk_of[N[a]]].push_back(e);
    }
  }
  L.blk.resize(nblk);
  std::vector<std::vector<std::pair<int,int>>> fix(npoin);
  int nslot = 0;
  std::vector<int> local(npoin, -1);
  std::vector<std::pair<uint64_t, int64_t>> keyed;
  for (int b = 0; b < nblk; ++b) {
    Block& B = L.blk[b];
    B.own0 = bstart[b];
    B.nown = bstart[b + 1] - bstart[b];
    std::vector<int> halo;
    for (int64_t e : btets[b])
      for (int a = 0; a < 4; ++a) {
        const int m = (int)inpoel[e * 4 + a];
        if ((m >= bstart[b + 1] || m < bstart[b]) && local[m] != -2) {
          local[m] = -2;
          halo.push_back(m);
        }
      }
    std::sort(halo.begin(), halo.end());
    B.nloc = B.nown + (int)halo.size();
    if (B.nloc > block_cap) {
      err = "kozak layout: block exceeds LDS capacity";
      return XG_EUNSUPPORTED;
    }
    B.halo_off = (int)L.halo.size();
    B.slot0 = gather ? -1 : nslot;
    for (size_t h = 0; h < halo.size(); ++h) {
      L.halo.push_back(halo[h]);
      if (!gather) fix[halo[h]].emplace_back(b, nslot + (int)h);
    }
    if (!gather) nslot += (int)halo.size();
    for (int i = 0; i < B.nown; ++i) local[B.own0 + i] = i;
    for (size_t h = 0; h < halo.size(); ++h) local[halo[h]] = B.nown + (int)h;
    auto& T = btets[b];
    sort_by_key(T, keyed, [&](int64_t e) {
      int l[4];
      for (int a = 0; a < 4; ++a) l[a] = local[inpoel[e * 4 + a]];
      for (auto o : {std::pair<int, int>{0, 1}, {2, 3}, {0, 2}, {1, 3}, {1, 2}})
        if (l[o.first] > l[o.second]) std::swap(l[o.first], l[o.second]);
      return ((uint64_t)l[0] << 48) | ((uint64_t)l[1] << 32) | ((uint64_t)l[2] << 16) |
             (uint64_t)l[3];
    });
    B.chunk0 = (int)L.chunks.size();
    const auto parts = spread_chunks(T, tets_per_chunk, B.nloc, [&](int64_t e, int* node) {
      int k = 0;
      for (int a = 0; a < 4; ++a) {
        const int m = local[inpoel[e * 4 + a]];
        if (!gather || m < B.nown) node[k++] = m;
      }
      return k;
    });
    for (const auto& P : parts) {
      std::vector<std::pair<int, uint16_t>> ent;
      for (size_t i = 0; i < P.size(); ++i)
        for (int a = 0; a < 4; ++a)
          if (!gather || local[inpoel[P[i] * 4 + a]] < B.nown)
            ent.emplace_back(local[inpoel[P[i] * 4 + a]], (uint16_t)(4 * i + a));
      Chunk C;
      C.kind = 2;
      C.first = (int)L.tab.size();
      C.count = (int)P.size();
      C.tend_off = (int)L.tend.size();
      C.ent_off = (int)L.entries.size();
      group_entries(ent, B.nloc, L.entries, L.tend);
      L.chunks.push_back(C);
      for (int64_t e : P) {
        const size_t* N = inpoel + e * 4;
        L.tab.push_back((uint32_t)local[N[0]] | ((uint32_t)local[N[1]] << 16));
        L.tcd.push_back((uint32_t)local[N[2]] | ((uint32_t)local[N[3]] << 16));
        for (int a = 0; a < 4; ++a) L.tglob.push_back((int)N[a]);
      }
    }
    B.chunk1 = (int)L.chunks.size();
    for (int i = 0; i < B.nown; ++i) local[B.own0 + i] = -1;
    for (size_t h = 0; h < halo.size(); ++h) local[halo[h]] = -1;
  }
  // the kernels prefetch 4 entries per tet; a gather chunk holds fewer (see
  // build_layout)
  if (gather) L.entries.resize(L.entries.size() + 4 * (size_t)tets_per_chunk, 0);
  L.nslot = nslot;
  L.fx_off.push_back(0);
  for (int n = 0; n < npoin; ++n) {
    if (fix[n].empty()) continue;
    L.fx_node.push_back(n);
    for (auto& bs : fix[n]) L.fx_slot.push_back(bs.second);
    L.fx_off.push_back((int)L.fx_slot.size());
  }
  return XG_OK;
}

// build(plan) with the size's plan and, where its gather blocks cannot hold a
// node's neighbours, with the full scatter blocks.
template <class Build>
static int by_plan(const BlockPlan& plan, int full_nodes, std::string& err, Build build) {
  if (!plan.gather) return build(plan, err);
  std::string why;
  const int rc = build(plan, why);
  if (rc == XG_EUNSUPPORTED) return build(BlockPlan{full_nodes, false}, err);
  if (rc) err = why;
  return rc;
}

int build_rhs_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                     const std::vector<double>& d, int64_t ntri, const int* tri,
                     const uint8_t* besym, Layout& L, std::string& err) {
  return by_plan(rhs_blocks(npoin), kRhsNodes, err, [&](const BlockPlan& b, std::string& e) {
    return build_layout(npoin, p, q, d, ntri, tri, besym, b.nodes, kRhsCap, kRhsSlots, L, e,
                        b.gather);
  });
}

int build_kozak_layout(int npoin, int64_t ntet, const size_t* inpoel, TetLayout& L,
                       std::string& err) {
  return by_plan(tet_blocks(npoin), kKozNodes, err, [&](const BlockPlan& b, std::string& e) {
    return build_tet_layout(npoin, ntet, inpoel, b.nodes, kKozCap, L, e, kTetsPerPairChunk,
                            b.gather);
  });
}

int build_cho_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                     const std::vector<double>& d, int64_t ntri, const int* tri, Layout& L,
                     std::string& err) {
  const std::vector<uint8_t> nosym(ntri * 3 + 1, 0);
  return by_plan(cho_blocks(npoin), kBlockNodes, err, [&](const BlockPlan& b, std::string& e) {
    return build_layout(npoin, p, q, d, ntri, tri, nosym.data(), b.nodes, kBlockCap, kChunkSlots,
                        L, e, b.gather, false);
  });
}

// Recursive coordinate bisection into cells of at most `leaf` nodes; the
// order of nodes inside a cell is their original order.
static void rcb(std::vector<int>& ids, size_t lo, size_t hi, const double* x,
                const double* y, const double* z, int leaf) {
  if (hi - lo <= (size_t)leaf) {
    std::sort(ids.begin() + lo, ids.begin() + hi);
    return;
  }
  double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
  const double* X[3] = {x, y, z};
  for (size_t i = lo; i < hi; ++i)
    for (int a = 0; a < 3; ++a) {
      mn[a] = std::min(mn[a], X[a][ids[i]]);
      mx[a] = std::max(mx[a], X[a][ids[i]]);
    }
  int ax = 0;
  for (int a = 1; a < 3; ++a)
    if (mx[a] - mn[a] > mx[ax] - mn[ax]) ax = a;
  // split so that the left part holds a whole number of leaves
  size_t n = hi - lo;
  size_t nleaf = (n + leaf - 1) / leaf;
  size_t mid = lo + ((nleaf / 2) * n) / nleaf;
  const double* C = X[ax];
  std::nth_element(ids.begin() + lo, ids.begin() + mid, ids.begin() + hi,
                   [&](int a, int b) { return C[a] < C[b] || (C[a] == C[b] && a < b); });
  rcb(ids, lo, mid, x, y, z, leaf);
  rcb(ids, mid, hi, x, y, z, leaf);
}

int block_order(int64_t npoin, const double* x, const double* y,
                const double* z, int leaf, size_t* perm) {
  std::vector<int> ids(npoin);
  std::iota(ids.begin(), ids.end(), 0);
  rcb(ids, 0, ids.size(), x, y, z, leaf);
  for (int64_t i = 0; i < npoin; ++i) perm[ids[i]] = (size_t)i;
  return XG_OK;
}

}  // namespace xg

extern "C" int xg_mesh_block_order(int64_t npoin, const double* x,
                                   const double* y, const double* z,
                                   int64_t cell_nodes, size_t* perm) {
  if (npoin <= 0 || npoin >= (1ll << 31) || !x || !y || !z || !perm ||
      cell_nodes < 1)
    return XG_EINVAL;
  return xg::block_order(npoin, x, y, z, (int)cell_nodes, perm);
}
