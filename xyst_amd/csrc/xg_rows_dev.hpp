// Device side of the node rows (see xg_rows.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "xg_ctx.hpp"
#include "xg_rows.hpp"

// an xg::RowLayout on the device
struct RowsDev {
  int nblk = 0;
  int lanes = 1;
  int4* blk = nullptr;      // own0, nown, nloc, halo_off
  int* wave0 = nullptr;
  int4* wave = nullptr;     // e0, erows, f0, frows
  int* halo = nullptr;
  uint16_t *deg = nullptr, *fdeg = nullptr, *nb = nullptr;
  double *dx = nullptr, *dy = nullptr, *dz = nullptr;
  uint32_t *fab = nullptr, *fcs = nullptr;
  double* fn = nullptr;     // normals of the face entries, 3 each
};

namespace {

// fn: a normal per face entry (padding: 0), scaled as the operator needs it
inline int upload_rows(xg_ctx* c, std::vector<DevArr>& M, const xg::RowLayout& L,
                       const std::vector<double>& fn, int lanes, RowsDev& R) {
  using namespace xgd;
  std::vector<int4> b(L.blk.size()), w(L.wave.size());
  std::vector<int> w0(L.blk.size());
  for (size_t i = 0; i < L.blk.size(); ++i) {
    const auto& B = L.blk[i];
    b[i] = make_int4(B.own0, B.nown, B.nloc, B.halo_off);
    w0[i] = B.wave0;
  }
  for (size_t i = 0; i < L.wave.size(); ++i) {
    const auto& W = L.wave[i];
    w[i] = make_int4(W.e0, W.erows, W.f0, W.frows);
  }
  int rc;
  if ((rc = upload(c, M, &R.blk, b)) || (rc = upload(c, M, &R.wave0, w0)) ||
      (rc = upload(c, M, &R.wave, w)) || (rc = upload(c, M, &R.halo, L.halo)) ||
      (rc = upload(c, M, &R.deg, L.deg)) || (rc = upload(c, M, &R.fdeg, L.fdeg)) ||
      (rc = upload(c, M, &R.nb, L.nb)) || (rc = upload(c, M, &R.dx, L.dx)) ||
      (rc = upload(c, M, &R.dy, L.dy)) || (rc = upload(c, M, &R.dz, L.dz)) ||
      (rc = upload(c, M, &R.fab, L.fab)) || (rc = upload(c, M, &R.fcs, L.fcs)) ||
      (rc = upload(c, M, &R.fn, fn)))
    return rc;
  R.nblk = (int)L.blk.size();
  R.lanes = lanes;
  return XG_OK;
}

// sum over the LPN neighbouring lanes of a node (a power of two), the same in
// all of them
template <int LPN>
__device__ inline double node_sum(double v) {
#pragma unroll
  for (int o = 1; o < LPN; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Writes K values of each node of a wave (one lane per node) to
// out[node * K ...], `nodes` (<= 64) consecutive ones: through `buf`, 32 K
// doubles of LDS of the wave's own, so that the stores are consecutive
// (stores of 8 bytes at a stride of 8 K take the memory path a lane at a
// time).  Half the wave's nodes at a time; lockstep within the wave.
template <int K>
__device__ inline void store_nodes(const double v[K], double* buf, double* __restrict__ out,
                                   int nodes, int lane) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if ((lane >> 5) == h) {
#pragma unroll
      for (int k = 0; k < K; ++k) buf[(lane & 31) * K + k] = v[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n = min(32, nodes - 32 * h) * K;
    for (int i = lane; i < n; i += 64) out[(size_t)32 * h * K + i] = buf[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

}  // namespace
