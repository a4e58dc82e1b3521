// Host-side description of the device layout (see xg_layout.cpp).
#pragma once
#include <cstdint>
#include <string>
#include <vector>

#include "xg_internal.hpp"

namespace xg {

// ChoCG edge blocks: slots per chunk = threads per workgroup (also the
// largest chunk any layout may use: slot ids are 10-bit)
constexpr int kChunkSlots = 1024;
// nodes (owned + halo) a ChoCG block may touch; its operators stage their
// node fields for these in LDS beside one chunk of edge terms
constexpr int kBlockCap = 616;
// owned nodes per block (a block also stops growing at kBlockCap)
constexpr int kBlockNodes = 432;
// riemann::grad blocks (node rows, xg_rows.hpp): one thread per owned node,
// the primitive state of the local ones in LDS (30,720 bytes: five
// workgroups share a CU); small meshes: 16 nodes, four lanes each.
constexpr int kGradNodes = 384;
constexpr int kGradCap = 768;
constexpr int kGradSmallCap = 256;
// riemann::rhs has blocks of its own, small enough that two 512-thread
// workgroups share a CU: 23 doubles per local node, 512 flux slots of 5
// doubles and the entry lists take 80,560 of the 81,920 bytes of LDS each
constexpr int kRhsSlots = 512;
constexpr int kRhsCap = 312;
constexpr int kRhsNodes = 312;

struct Block {
  int own0 = 0, nown = 0, nloc = 0;  // owned ids [own0, own0+nown); local ids
  int halo_off = 0;                  // halo node ids at halo[halo_off ...]
  int slot0 = 0;                     // first halo output slot (-1: none)
  int chunk0 = 0, chunk1 = 0;        // chunks [chunk0, chunk1)
};

struct Chunk {
  int kind = 0;       // 0 edges, 1 boundary faces
  int first = 0;      // first edge / face of the chunk in layout order
  int count = 0;      // number of edges / faces
  int tend_off = 0;   // dense per-local-node entry ends (nloc of them)
  int ent_off = 0;    // entry list offset
};

struct Layout {
  int npoin = 0;
  // edges and faces in block/chunk order, end nodes as block-local ids
  std::vector<uint32_t> elpq;      // local p | local q << 16
  std::vector<double> dx, dy, dz;
  std::vector<int> ep, eq;         // global end nodes (grad stream, checks)
  std::vector<int64_t> eidx;       // input index of each layout edge
  std::vector<int64_t> fidx;       // input index of each layout face
  std::vector<uint32_t> fab;       // local a | local b << 16
  std::vector<uint32_t> fcs;       // local c | symmetry bits << 16
  std::vector<int> fglob;          // global face nodes (checks)
  std::vector<Block> blk;
  std::vector<Chunk> chunks;
  std::vector<int> halo;
  std::vector<uint16_t> tend;      // per chunk: nloc cumulative entry ends
  std::vector<uint16_t> entries;   // slot | 0x8000 for a negative sign
  int nslot = 0;
  std::vector<int> fx_node, fx_off, fx_slot;
};

// KozCG blocks: a block stages U (5) and coordinates (3) of up to kKozCap
// nodes in LDS beside one chunk's corner values (5 doubles per slot); a
// chunk holds kKozPairSlots / 4 tets, two threads per tet.  At 1024 slots
// and 512 nodes the largest of the KozCG block kernels takes 80,896 bytes of
// LDS, so two share a CU.
constexpr int kKozCap = 512;
constexpr int kKozNodes = 384;
constexpr int kKozPairSlots = 1024;
constexpr int kTetsPerPairChunk = kKozPairSlots / 4;

struct TetLayout {
  int npoin = 0;
  std::vector<uint32_t> tab, tcd;  // tets in block/chunk order: local a|b<<16, c|d<<16
  std::vector<int> tglob;          // their global nodes (4 per tet)
  std::vector<Block> blk;
  std::vector<Chunk> chunks;       // kind 2
  std::vector<int> halo;
  std::vector<uint16_t> tend, entries;   // entry = slot 4*i+a
  int nslot = 0;
  std::vector<int> fx_node, fx_off, fx_slot;
};

// gather: a block takes every tet that touches one of its nodes and its
// entries reach its owned corners only (as for the edge layouts below)
int build_tet_layout(int npoin, int64_t ntet, const size_t* inpoel,
                     int block_nodes, int block_cap, TetLayout& L,
                     std::string& err,
                     int tets_per_chunk = kTetsPerPairChunk, bool gather = false);

// chunk_slots: flux slots per edge chunk (<= kChunkSlots; boundary-face
// chunks hold chunk_slots / 3 faces).
// gather: a block takes every edge that touches one of its nodes (edges
// between two blocks are in both), its halo is every outside end of those,
// and its entries add each edge to its owned ends only, so every owned sum
// is complete in its block: no halo slots (Block::slot0 is -1) and no
// fix-up lists.  Likewise every boundary face that touches one of its nodes.
// spread: a node's edges over the chunks of its block (spread_chunks).
int build_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                 const std::vector<double>& d, int64_t ntri, const int* tri,
                 const uint8_t* besym, int block_nodes, int block_cap,
                 int chunk_slots, Layout& L, std::string& err, bool gather = false,
                 bool spread = true);

// Blocks of small meshes.  At the full block sizes a mesh of a few thousand
// nodes fills a few of the 256 CUs, and each block walks its chunks alone: so
// they are cut into about as many blocks as run at once, and where that is
// the faster, into gather blocks, which need no halo fix-up.  Times of the
// full blocks and of these when the lines were drawn (chunks not yet spread,
// the tet kernels' arithmetic heavier), in us:
//  riemann::grad: sixteen nodes, four lanes each (its waves are independent);
//  riemann::rhs (two workgroups per CU: at most 512 blocks): 12^3 20.6 ->
//    6.9, 24^3 21.1 -> 9.9, 29^3 (27,000 nodes) 23.7 -> 14.5, with 6
//    components (one workgroup per CU) 23.9 -> 20.5; on 31^3 (32,768) 22.4 ->
//    20.4, but 22.7 -> 27.9 with 6;
//  the tet operators, KozCG step: 12^3 201 -> 84, 20^3 (9,261) 201 -> 104, as
//    scatter blocks 117; 24^3 (15,625) 203 -> 140 and 125 as scatter blocks,
//    36^3 216 -> 178, 39^3 (64,000) 216 -> 197, 42^3 equal;
//  the chorin operators (one workgroup per CU: at most 256 blocks),
//    chorin::rhs: 12^3 20.0 -> 6.2, 20^3 20.6 -> 8.3, 28^3 (24,389) 20.7 ->
//    11.6, as scatter blocks 14.5; 33^3 22.2 -> 23.3.
constexpr int64_t kSmallGrad = 49152;
constexpr int64_t kSmallRhs = 28672;
constexpr int64_t kSmallTetGather = 10240;
constexpr int64_t kSmallTet = 65536;
constexpr int64_t kSmallCho = 28672;

struct BlockPlan {
  int nodes;     // owned nodes per block, at most
  bool gather;   // a gather layout
};

inline int small_nodes(int64_t npoin, int64_t nblk) {
  return (int)(npoin < 16 * nblk ? 16 : (npoin + nblk - 1) / nblk);
}
inline BlockPlan rhs_blocks(int64_t npoin) {
  if (npoin <= kSmallRhs) return {small_nodes(npoin, 512), true};
  return {kRhsNodes, false};
}
inline BlockPlan tet_blocks(int64_t npoin) {
  if (npoin <= kSmallTetGather) return {small_nodes(npoin, 320), true};
  return {npoin <= kSmallTet ? small_nodes(npoin, 768) : kKozNodes, false};
}
inline BlockPlan cho_blocks(int64_t npoin) {
  if (npoin <= kSmallCho) return {small_nodes(npoin, 224), true};
  return {kBlockNodes, false};
}

// The layouts of riemann::rhs, the tet operators and the chorin operators by
// these plans.  A gather block holds all neighbours of its nodes, a scatter
// block those with larger ids only (for tets: the nodes of the tets whose
// smallest node it owns), so a mesh with a node of too many neighbours for
// gather blocks takes the full scatter blocks whatever its size.
int build_rhs_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                     const std::vector<double>& d, int64_t ntri, const int* tri,
                     const uint8_t* besym, Layout& L, std::string& err);
int build_kozak_layout(int npoin, int64_t ntet, const size_t* inpoel, TetLayout& L,
                       std::string& err);
int build_cho_layout(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                     const std::vector<double>& d, int64_t ntri, const int* tri, Layout& L,
                     std::string& err);

int block_order(int64_t npoin, const double* x, const double* y,
                const double* z, int leaf, size_t* perm);

}  // namespace xg
