// Node rows: the layout of edge operators whose edge terms are cheap enough
// to be evaluated at both ends (xg_rows_dev.hpp).
//
// Blocks of consecutive owned nodes as in xg_layout.hpp, with every outside
// neighbour as halo.  The edges of a node are taken in the order of the input,
// with one lane per node from both ends inward, each as the neighbour's
// block-local id and the edge integral with the sign of this end (R(p) -= f,
// R(q) += f), interleaved over the 64 lanes of a wave, so that a wave reads
// consecutive addresses and a lane sums its node in registers: no edge records
// in LDS, no barrier after the block's nodes are staged.  `lanes` lanes share a
// node (entry k goes to lane k % lanes) where one per node would leave too few
// waves.  Boundary faces likewise, at each of their nodes, in input order.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

#include "xg_internal.hpp"

namespace xg {

struct RowBlock {
  int own0 = 0, nown = 0, nloc = 0, halo_off = 0;
  int wave0 = 0;                 // first wave record
};
struct RowWave {
  int e0 = 0, erows = 0;         // entry (row j, lane l) at e0 + 64 j + l
  int f0 = 0, frows = 0;
};
struct RowLayout {
  std::vector<RowBlock> blk;
  std::vector<RowWave> wave;
  std::vector<int> halo;
  std::vector<uint16_t> deg, fdeg;  // per wave and lane: its entries, faces
  std::vector<uint16_t> nb;         // neighbour, block-local
  std::vector<double> dx, dy, dz;   // signed integrals
  std::vector<int64_t> eidx;        // input edge of each entry (-1: padding)
  std::vector<uint32_t> fab, fcs;   // a | b << 16; c | this corner << 16 (checks)
  std::vector<int64_t> fidx;        // input face of each face entry (-1: padding)
};

// XG_EUNSUPPORTED when a node and its neighbours are more than cap nodes, or
// it has more than 65535 entries or faces per lane
int build_rows(int npoin, const std::vector<int>& p, const std::vector<int>& q,
               const std::vector<double>& d, int64_t ntri, const int* tri, int block_nodes,
               int cap, int lanes, RowLayout& L, std::string& err);

// riemann::grad's rows (xg_layout.hpp, kGrad*) and their lanes per node: four
// on small meshes, unless a node has more neighbours than their blocks hold.
int build_grad_rows(int npoin, const std::vector<int>& p, const std::vector<int>& q,
                    const std::vector<double>& d, int64_t ntri, const int* tri, RowLayout& L,
                    int& lanes, std::string& err);

}  // namespace xg
