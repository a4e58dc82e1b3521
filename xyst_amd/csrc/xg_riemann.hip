// MI355X (gfx950) device path of the RieCG edge-based Riemann/MUSCL scheme:
// context, device mesh layout, riemann::grad/rhs kernels, RK stage, CFL
// minimum.  All FP64.  Deterministic: no atomics, every nodal sum is taken in
// an order fixed by the layout (xg_layout.cpp).
//
//   rhs:  k_rhs_blocks -- one 512-thread workgroup per node block (two per
//         CU); the block's node data staged in LDS, one node sum per thread;
//         k_fixup<5> adds halo partials.
//   grad: k_grad_rows -- node rows (xg_rows.hpp): each edge evaluated at both
//         ends, a lane per node.
// Small meshes use gather blocks for the rhs (xg::rhs_blocks) and four lanes
// per node for the gradient.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "xg_flux.hpp"
#include "xg_layout.hpp"
#include "xg_problems.hpp"

using xg::Cfg;

#include "xg_blocks.hpp"
#include "xg_rows_dev.hpp"
#include "xg_amg.hpp"
#include "xg_ctx.hpp"
#include "xg_gnn.hpp"

namespace {

using namespace xgd;
constexpr int kRhsThreads = xg::kRhsSlots;

// ----------------------------------------------------------------- kernels --

// riemann::grad (Riemann.cpp:229-367) on node rows (xg_rows.hpp): the block's
// primitive states are staged in LDS, then each node's lane (or LPN lanes)
// adds D (u + u_neighbour) over its edges (:263-328), reading neighbour ids
// and integrals with consecutive addresses across the wave, and over its
// boundary faces (:332-359) the faces' values, which as in the reference go
// to every node of a face alike: g[j] n[j] for direction j, with g[j] the
// 4:1:1-weighted value belonging to the face's j-th node.
// What bounds it: the bytes, 26 per entry (two entries an edge), 40 of U (about
// twice, with the halo) and 120 of G per node: 0.51 GB on 96^3 (912,673
// nodes), 128 us, 4.0 TB/s.  A block kernel that evaluated an edge once or
// twice into LDS and summed it per node between barriers took 207 us.  Two rows
// in flight instead of four: 131 us; six waves per SIMD (spills): 135 us.
// DIV: divided by the nodal volume (RieCG.cpp:935-939).  NC components per
// node (5 + transported scalars).
template <bool DIV, int NC, int LPN, int NT, int CAP>
__global__ __launch_bounds__(NT) void k_grad_rows(RowsDev L, const double* __restrict__ U,
                                                 double* __restrict__ G,
                                                 const double* __restrict__ vol) {
  constexpr int K = 3 * NC;
  constexpr int AHEAD = 4;     // rows in flight
  __shared__ double sP[NC * CAP];
  static_assert(NT / 64 * 32 * K <= NC * CAP || LPN > 1, "the stores' buffers reuse sP");
  const int t = threadIdx.x, lane = t & 63;
  const int b = xcd_block(blockIdx.x, L.nblk);
  const int4 B = L.blk[b];     // own0, nown, nloc, halo_off
  const int w0 = L.wave0[b];
  const int own0 = B.x, nown = B.y, nloc = B.z;
  for (int i = t; i < nloc; i += NT) {
    const int g = i < nown ? own0 + i : L.halo[B.w + i - nown];
    double s[NC], u[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) s[c] = U[(size_t)g * NC + c];
    xg::primitive_fast(s, u);
#pragma unroll
    for (int c = 5; c < NC; ++c) u[c] = s[c];
#pragma unroll
    for (int c = 0; c < NC; ++c) sP[c * CAP + i] = u[c];
  }
  const int n = t / LPN;       // local node
  const bool any = (t & ~63) / LPN < nown;   // the wave has nodes
  int4 W = make_int4(0, 0, 0, 0);
  int deg = 0, fdeg = 0;
  if (any) {
    W = L.wave[w0 + (t >> 6)];
    deg = L.deg[(w0 + (t >> 6)) * 64 + lane];
    fdeg = L.fdeg[(w0 + (t >> 6)) * 64 + lane];
  }
  int nb[AHEAD];
  double D[AHEAD][3];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (j0 + u < W.y) {      // the same for the wave
        const int e = W.x + (j0 + u) * 64 + lane;
        nb[u] = L.nb[e];
        D[u][0] = L.dx[e];
        D[u][1] = L.dy[e];
        D[u][2] = L.dz[e];
      }
  };
  fetch(0);
  __syncthreads();             // the block's nodes are staged
  double own[NC], acc[K];
#pragma unroll
  for (int c = 0; c < NC; ++c) own[c] = sP[c * CAP + min(n, nloc - 1)];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.0;
  for (int j0 = 0; j0 < W.y; j0 += AHEAD) {
    int m[AHEAD];
    double d[AHEAD][3];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      m[u] = nb[u];
#pragma unroll
      for (int k = 0; k < 3; ++k) d[u][k] = D[u][k];
    }
    fetch(j0 + AHEAD);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (j0 + u < deg) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const double f = own[c] + sP[c * CAP + m[u]];
          acc[c * 3 + 0] += d[u][0] * f;
          acc[c * 3 + 1] += d[u][1] * f;
          acc[c * 3 + 2] += d[u][2] * f;
        }
      }
  }
  for (int j = 0; j < W.w; ++j) {
    if (j >= fdeg) continue;
    const size_t e = (size_t)W.z + j * 64 + lane;
    const uint32_t ab = L.fab[e], cs = L.fcs[e];
    const int a = ab & 0xffff, bb = ab >> 16, cc = cs & 0xffff;
    const double n0 = L.fn[e * 3], n1 = L.fn[e * 3 + 1], n2 = L.fn[e * 3 + 2];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const double ua = sP[c * CAP + a], ub = sP[c * CAP + bb], uc = sP[c * CAP + cc];
      const double uab = (ua + ub) * 0.25, ubc = (ub + uc) * 0.25, uca = (uc + ua) * 0.25;
      acc[c * 3 + 0] += (uab + uca + ua) * n0;
      acc[c * 3 + 1] += (uab + ubc + ub) * n1;
      acc[c * 3 + 2] += (ubc + uca + uc) * n2;
    }
  }
  if (LPN > 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = node_sum<LPN>(acc[k]);
  }
  if (DIV && n < nown) {
    const double v = vol[own0 + n];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] /= v;
  }
  if constexpr (LPN > 1) {
    if (n < nown) {
      double* o = G + (size_t)(own0 + n) * K;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if ((k & (LPN - 1)) == (t & (LPN - 1))) o[k] = acc[k];
    }
  } else {
    __syncthreads();           // sP is read no more
    const int left = nown - (t & ~63);
    if (left > 0)
      store_nodes<K>(acc, sP + (t >> 6) * 32 * K, G + (size_t)(own0 + (t & ~63)) * K,
                     min(left, 64), lane);
  }
}

// Per-chunk bookkeeping shared by the block kernels: the chunk's entry list
// (slot | sign bit, grouped by local node) and each local node's entry end
// are prefetched into registers one chunk ahead with coalesced loads, then
// placed in LDS, so the per-node accumulation loop reads LDS only.
// (NT threads, chunks of at most NT edges: up to 2 NT entries)
template <int NT>
struct ChunkPrefetch {
  uint16_t e0 = 0, e1 = 0, te = 0;
  __device__ inline void load(const int4& C, int ent_off, int nloc, int t,
                              const uint16_t* __restrict__ tend,
                              const uint16_t* __restrict__ entries) {
    int nent = C.z * (C.x == 0 ? 2 : 3);
    if (t < nent) e0 = entries[ent_off + t];
    if (t + NT < nent) e1 = entries[ent_off + NT + t];
    if (t < nloc) te = tend[C.w + t];
  }
  __device__ inline void store(const int4& C, int nloc, int t, uint16_t* sE,
                               uint16_t* sT) const {
    int nent = C.z * (C.x == 0 ? 2 : 3);
    if (t < nent) sE[t] = e0;
    if (t + NT < nent) sE[NT + t] = e1;
    if (t < nloc) sT[t] = te;
  }
};

// advbnd (Riemann.cpp:768-878) for one boundary face from the staged
// primitive states: the three corner contributions (fab + fca + f_a style
// weights).  The conserved values are rebuilt from the primitive ones; a
// transported scalar's corner flux is its value times the normal velocity.
template <int NC>
__device__ inline void face_flux_lds(int la, int lb, int lc, int sym,
                                     const double* __restrict__ sP,
                                     const double* __restrict__ sX,
                                     double gm1, double out[3][NC]) {
  constexpr int CAP = xg::kRhsCap;   // the rhs blocks' LDS stride
  int N[3] = {la, lb, lc};
  double ba[3], ca[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    ba[j] = sX[j * CAP + lb] - sX[j * CAP + la];
    ca[j] = sX[j * CAP + lc] - sX[j * CAP + la];
  }
  double nx = (ba[1] * ca[2] - ca[1] * ba[2]) / 12.0;
  double ny = (ba[2] * ca[0] - ca[2] * ba[0]) / 12.0;
  double nz = (ba[0] * ca[1] - ca[0] * ba[1]) / 12.0;
  double fl[NC][3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double r = sP[0 * CAP + N[a]], u = sP[1 * CAP + N[a]], v = sP[2 * CAP + N[a]];
    double w = sP[3 * CAP + N[a]], e = sP[4 * CAP + N[a]];
    double p = (r * e) * gm1;
    double vn = ((sym >> a) & 1) ? 0.0 : (nx * u + ny * v + nz * w);
    double re = r * (e + 0.5 * (u * u + v * v + w * w));
    fl[0][a] = r * vn;
    fl[1][a] = r * u * vn + p * nx;
    fl[2][a] = r * v * vn + p * ny;
    fl[3][a] = r * w * vn + p * nz;
    fl[4][a] = (re + p) * vn;
#pragma unroll
    for (int c = 5; c < NC; ++c) fl[c][a] = sP[c * CAP + N[a]] * vn;
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    double fab = (fl[c][0] + fl[c][1]) / 4.0;
    double fbc = (fl[c][1] + fl[c][2]) / 4.0;
    double fca = (fl[c][2] + fl[c][0]) / 4.0;
    out[0][c] = fab + fca + fl[c][0];
    out[1][c] = fab + fbc + fl[c][1];
    out[2][c] = fbc + fca + fl[c][2];
  }
}

// riemann::rhs (advdom + advbnd, Riemann.cpp:652-878) for one node block.
// The block's nodes (owned range + halo) are staged in LDS as primitive
// state, gradient and coordinates.  Thread t owns local node t and keeps its
// nodal sum in registers.  Per chunk: each thread evaluates one edge flux (or
// one face's three corner terms) into LDS, then every node thread adds the
// chunk's slots that touch it, in slot order.  NC components per node
// (5 + transported scalars; with scalars the LDS of one workgroup exceeds
// half a CU's, so one workgroup runs per CU).
template <int FLUX, int NC>
__global__ __launch_bounds__(kRhsThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_rhs_blocks(
    int nblk, const int4* __restrict__ blk0, const int4* __restrict__ blk1,
    const int* __restrict__ halo, const int4* __restrict__ chk,
    const int* __restrict__ chk_ent, const uint16_t* __restrict__ tend,
    const uint16_t* __restrict__ entries, const uint32_t* __restrict__ elpq,
    const double* __restrict__ dx, const double* __restrict__ dy,
    const double* __restrict__ dz, const uint32_t* __restrict__ fab,
    const uint32_t* __restrict__ fcs, const double* __restrict__ x,
    const double* __restrict__ y, const double* __restrict__ z,
    const double* __restrict__ G, const double* __restrict__ U,
    double* __restrict__ R, double* __restrict__ S, Cfg cfg) {
  constexpr int CAP = xg::kRhsCap;
  __shared__ double sN[(4 * NC + 3) * CAP];
  double* const sP = sN;                  // primitive state, NC x CAP
  double* const sG = sN + NC * CAP;       // gradients, 3 NC x CAP
  double* const sX = sN + 4 * NC * CAP;   // coordinates, 3 x CAP
  __shared__ double F[kRhsThreads * NC];
  __shared__ uint16_t sE[2 * kRhsThreads];
  __shared__ uint16_t sT[CAP];
  const int t = threadIdx.x;
  const int b = xcd_block(blockIdx.x, nblk);
  const int4 B0 = blk0[b];   // own0, nown, nloc, halo_off
  const int4 B1 = blk1[b];   // slot0, chunk0, chunk1
  const int own0 = B0.x, nown = B0.y, nloc = B0.z;
  // stage the block's nodes (one per thread, nloc <= threads): all 4 NC + 3
  // loads of a node are issued before the first is used
  if (t < nloc) {
    int g = t < nown ? own0 + t : halo[B0.w + t - nown];
    double s[NC], u[NC], gg[3 * NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) s[c] = U[(size_t)g * NC + c];
#pragma unroll
    for (int c = 0; c < 3 * NC; ++c) gg[c] = G[(size_t)g * (3 * NC) + c];
    double xg_ = x[g], yg = y[g], zg = z[g];
    xg::primitive_fast(s, u);
#pragma unroll
    for (int c = 5; c < NC; ++c) u[c] = s[c];
#pragma unroll
    for (int c = 0; c < NC; ++c) sP[c * CAP + t] = u[c];
#pragma unroll
    for (int c = 0; c < 3 * NC; ++c) sG[c * CAP + t] = gg[c];
    sX[0 * CAP + t] = xg_;
    sX[1 * CAP + t] = yg;
    sX[2 * CAP + t] = zg;
  }
  // the next chunk's edge record and entry lists are loaded while the
  // current chunk computes
  ChunkPrefetch<kRhsThreads> pf;
  uint32_t pq_n = 0;
  double dx_n = 0.0, dy_n = 0.0, dz_n = 0.0;
  auto fetch = [&](int c, int tl) {
    if (c < B1.z) {
      const int4 C = chk[c];
      pf.load(C, chk_ent[c], nloc, tl, tend, entries);
      if (C.x == 0 && tl < C.z) {
        int e = C.y + tl;
        pq_n = elpq[e];
        dx_n = dx[e];
        dy_n = dy[e];
        dz_n = dz[e];
      }
    }
  };
  fetch(B1.y, t);
  double acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0.0;
  for (int ch = B1.y; ch < B1.z; ++ch) {
    // the thread index, opaque to the optimizer: thread-dependent LDS
    // addresses are recomputed per chunk instead of being held (and spilled)
    // across the whole loop
    int tl = t;
    asm volatile("" : "+v"(tl));
    const int4 C = chk[ch];   // kind, first, count, tend_off
    const uint32_t pq = pq_n;
    double d[3] = {dx_n, dy_n, dz_n};
    __syncthreads();          // staging done / previous chunk's F consumed
    pf.store(C, nloc, tl, sE, sT);
    if (tl < C.z) {
      if (C.x == 0) {
        int lp = pq & 0xffff, lq = pq >> 16;
        double l[NC], r[NC], f[NC], g1[NC], g2[NC];
        double vw[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) vw[j] = sX[j * CAP + lq] - sX[j * CAP + lp];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          l[c] = sP[c * CAP + lp];
          r[c] = sP[c * CAP + lq];
          g1[c] = sG[(c * 3 + 0) * CAP + lp] * vw[0] + sG[(c * 3 + 1) * CAP + lp] * vw[1] +
                  sG[(c * 3 + 2) * CAP + lp] * vw[2];
          g2[c] = sG[(c * 3 + 0) * CAP + lq] * vw[0] + sG[(c * 3 + 1) * CAP + lq] * vw[1] +
                  sG[(c * 3 + 2) * CAP + lq] * vw[2];
        }
        xg::muscl_fast(g1, g2, l, r);
        xg::ScalarFlux sf;
        if (FLUX == 0)
          xg::rusanov_fast(cfg, d, l, r, f, sf);
        else
          xg::hllc_fast(cfg, d, l, r, f, sf);
        if constexpr (NC > 5) {
          xg::muscl_scalars<NC>(g1, g2, l, r);
#pragma unroll
          for (int c = 5; c < NC; ++c)
            f[c] = (l[c] * sf.a + r[c] * sf.b) * sf.m + sf.sw * (r[c] - l[c]);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) F[tl * NC + c] = f[c];
      } else {
        int f = C.y + tl;
        uint32_t ab = fab[f], cs = fcs[f];
        double o[3][NC];
        face_flux_lds<NC>(ab & 0xffff, ab >> 16, cs & 0xffff, cs >> 16, sP, sX, cfg.gm1, o);
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
          for (int c = 0; c < NC; ++c) F[(3 * tl + a) * NC + c] = o[a][c];
      }
    }
    fetch(ch + 1, tl);        // in flight during the accumulation below
    __syncthreads();          // F, sE, sT complete
    if (tl < nloc) {
      int e0 = tl ? sT[tl - 1] : 0, e1 = sT[tl];
      for (int j = e0; j < e1; ++j) {
        int v = sE[j];
        const double* fs = F + (v & 0x3ff) * NC;
        double sg = (v & 0x8000) ? -1.0 : 1.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = fma(sg, fs[c], acc[c]);
      }
    }
  }
  if (t < nown) {
    double* o = R + (size_t)(own0 + t) * NC;
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] = acc[c];
  } else if (t < nloc && B1.x >= 0) {
    double* o = S + (size_t)(B1.x + t - nown) * NC;
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] = acc[c];
  }
}

// U = Un - rkcoef*dt*R/vol (RieCG.cpp:1016-1021); STAGE0 first saves
// Un = U (RieCG.cpp:1000-1003); NC components per node
template <bool STAGE0, int NC>
__global__ void k_update(int npoin, double coef_dt, double* __restrict__ U,
                         double* __restrict__ Un, const double* __restrict__ R,
                         const double* __restrict__ vol) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)npoin * NC) return;
  double un;
  if (STAGE0) {
    un = U[i];
    Un[i] = un;
  } else {
    un = Un[i];
  }
  U[i] = un - coef_dt * R[i] / vol[i / NC];
}

// U = Un - rkcoef*dtp[i]*R/vol with per-node time steps (steady runs,
// RieCG.cpp:1017-1018)
template <bool STAGE0, int NC>
__global__ void k_update_steady(int npoin, double rk, const double* __restrict__ dtp,
                                double* __restrict__ U, double* __restrict__ Un,
                                const double* __restrict__ R,
                                const double* __restrict__ vol) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)npoin * NC) return;
  double un;
  if (STAGE0) {
    un = U[i];
    Un[i] = un;
  } else {
    un = Un[i];
  }
  U[i] = un - rk * dtp[i / NC] * R[i] / vol[i / NC];
}

// F(i, :) /= vol[i] for NC components (RieCG.cpp:935-939)
template <int NC>
__global__ void k_div_vol(int npoin, double* __restrict__ F, const double* __restrict__ vol) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)npoin * NC) return;
  F[i] /= vol[i / NC];
}

// riemann::src (Riemann.cpp:880-907): R(p,c) -= s_c(x_p) v[p] for the flow
// components of the nc per node (the scalars have no source)
__global__ void k_src(int npoin, int nc, xg::Prob P, const double* __restrict__ x,
                      const double* __restrict__ y, const double* __restrict__ z,
                      const double* __restrict__ v, double* __restrict__ R) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npoin) return;
  double s[5];
  xg::source(P, x[p], y[p], z[p], s);
  double* r = R + (size_t)p * nc;
  const double vp = v[p];
#pragma unroll
  for (int c = 0; c < 5; ++c) r[c] -= s[c] * vp;
}

// physics::dirbc (BC.cpp:29-72) as the RieCG chare calls it: components
// with mask 1 take the node's initial-condition value (nc per node)
__global__ void k_dirbc_ic(int nd, int nc, const int* __restrict__ node,
                           const uint8_t* __restrict__ mask,
                           const double* __restrict__ val, double* __restrict__ U) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nd) return;
  double* u = U + (size_t)node[i] * nc;
  for (int c = 0; c < nc; ++c)
    if (mask[i * nc + c] == 1) u[c] = val[i * nc + c];
}

// physics::farbc (BC.cpp:152-221), the (node, normal) pairs of a node in
// list order
__global__ void k_farbc(int nf, int nc, const int* __restrict__ node,
                        const int* __restrict__ off, const double* __restrict__ nrm,
                        double fr, double fu, double fv, double fw, double fp, double g,
                        double* __restrict__ U) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nf) return;
  double* s = U + (size_t)node[i] * nc;
  double r = s[0], ru = s[1], rv = s[2], rw = s[3], re = s[4];
  const double a = sqrt(g * fp / fr);
  for (int k = off[i]; k < off[i + 1]; ++k) {
    const double* n = nrm + (size_t)k * 3;
    const double M = (fu * n[0] + fv * n[1] + fw * n[2]) / a;
    if (M <= -1.0) {              // supersonic inflow
      r = fr; ru = fr * fu; rv = fr * fv; rw = fr * fw;
      re = xg::total_energy(g, fr, fu, fv, fw, fp);
    } else if (M > -1.0 && M < 0.0) {   // subsonic inflow: inside pressure
      const double pr = (re - 0.5 * (ru * ru + rv * rv + rw * rw) / r) * (g - 1.0);
      r = fr; ru = fr * fu; rv = fr * fv; rw = fr * fw;
      re = xg::total_energy(g, fr, fu, fv, fw, pr);
    } else if (M >= 0.0 && M < 1.0) {   // subsonic outflow: outside pressure
      re = xg::total_energy(g, r, ru / r, rv / r, rw / r, fp);
    }
  }
  s[0] = r; s[1] = ru; s[2] = rv; s[3] = rw; s[4] = re;
}

// physics::prebc (BC.cpp:223-241), a node's (density, pressure) records in
// list order
__global__ void k_prebc(int np, int nc, const int* __restrict__ node,
                        const int* __restrict__ off, const double* __restrict__ val,
                        double g, double* __restrict__ U) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  double* s = U + (size_t)node[i] * nc;
  for (int k = off[i]; k < off[i + 1]; ++k) {
    s[0] = val[k * 2 + 0];
    s[4] = xg::total_energy(g, s[0], s[1] / s[0], s[2] / s[0], s[3] / s[0], val[k * 2 + 1]);
  }
}

// ------------------------------------------------------------- launchers --

int check_ncomp(xg_ctx* c, int ncomp) {
  if (ncomp < 5 || ncomp > XG_MAX_NCOMP)
    return fail(c, XG_EUNSUPPORTED,
                "device path supports ncomp = 5 + at most " +
                    std::to_string(XG_MAX_NCOMP - 5) + " transported scalars");
  return XG_OK;
}

int check_mesh(xg_ctx* c, int ncomp) {
  if (!c) return XG_EINVAL;
  if (!c->have_mesh) return fail(c, XG_ENOMESH, "no mesh uploaded");
  return check_ncomp(c, ncomp);
}

template <int NC>
void launch_grad_nc(xg_ctx* c, const double* U, double* G, bool div) {
  const RowsDev& L = *c->grows;
  if (L.lanes == 1) {
    auto kern = div ? k_grad_rows<true, NC, 1, xg::kGradNodes, xg::kGradCap>
                    : k_grad_rows<false, NC, 1, xg::kGradNodes, xg::kGradCap>;
    hipLaunchKernelGGL(kern, dim3(L.nblk), dim3(xg::kGradNodes), 0, c->stream, L, U, G, c->vol);
  } else {
    auto kern = div ? k_grad_rows<true, NC, 4, 64, xg::kGradSmallCap>
                    : k_grad_rows<false, NC, 4, 64, xg::kGradSmallCap>;
    hipLaunchKernelGGL(kern, dim3(L.nblk), dim3(64), 0, c->stream, L, U, G, c->vol);
  }
}

// div: G = grad(U)/vol (the RK stage; needs xg_riecg_setup).
// nc components per node (checked by the caller).
int launch_grad(xg_ctx* c, int nc, const double* U, double* G, bool div = false) {
  static_assert(XG_MAX_NCOMP == 7, "one instantiation per component count");
  if (nc == 5) launch_grad_nc<5>(c, U, G, div);
  else if (nc == 6) launch_grad_nc<6>(c, U, G, div);
  else launch_grad_nc<7>(c, U, G, div);
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

xg::Prob prob_of(const xg_ctx* c) {
  return xg::Prob{c->problem.kind, c->problem.alpha, c->problem.kappa, c->problem.p0,
                  c->cfg.gamma};
}

template <int NC>
void launch_rhs_nc(xg_ctx* c, const double* G, const double* U, double* R) {
  const double g = c->cfg.gamma;
  Cfg cfg{g, c->cfg.stab2, c->cfg.stab2coef, g - 1.0, g * (g - 1.0)};
  auto kern = c->cfg.flux == 0 ? k_rhs_blocks<0, NC> : k_rhs_blocks<1, NC>;
  const auto& B = c->rb;
  if (B.nblk)
    hipLaunchKernelGGL(kern, dim3(B.nblk), dim3(kRhsThreads), 0, c->stream,
                       B.nblk, B.blk0, B.blk1, B.halo, B.chk, B.chk_ent, B.tend,
                       B.entries, B.elpq, B.dx, B.dy, B.dz, B.fab, B.fcs, c->x, c->y,
                       c->z, G, U, R, B.slots, cfg);
  if (B.nfx)
    hipLaunchKernelGGL(k_fixup<NC>, dim3(nblocks(B.nfx)), dim3(kBlock), 0,
                       c->stream, B.nfx, B.fx_node, B.fx_off, B.fx_slot, B.slots, R);
}

// riemann::rhs with nc components per node (checked by the caller), then
// the problem's source on the flow components
int launch_rhs(xg_ctx* c, int nc, const double* G, const double* U, double* R,
               const double* v) {
  if (c->cfg.flux != 0 && c->cfg.flux != 1)
    return fail(c, XG_EINVAL, "Flux not configured");
  if (nc == 5) launch_rhs_nc<5>(c, G, U, R);
  else if (nc == 6) launch_rhs_nc<6>(c, G, U, R);
  else launch_rhs_nc<7>(c, G, U, R);
  const xg::Prob P = prob_of(c);
  if (xg::has_source(P))
    hipLaunchKernelGGL(k_src, dim3(nblocks(c->npoin)), dim3(kBlock), 0, c->stream,
                       c->npoin, nc, P, c->x, c->y, c->z, v, R);
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

// RieCG::BC (RieCG.cpp:764-785): dirbc, symbc, farbc, prebc
int launch_bc(xg_ctx* c, double* U) {
  const int nc = c->ncomp;
  if (c->ndirnode)
    hipLaunchKernelGGL(k_dirbc_ic, dim3(nblocks(c->ndirnode)), dim3(kBlock), 0,
                       c->stream, c->ndirnode, nc, c->dirnode, c->dirmask, c->dirval, U);
  if (c->nsymnode)
    hipLaunchKernelGGL(k_symbc, dim3(nblocks(c->nsymnode)), dim3(kBlock), 0,
                       c->stream, c->nsymnode, c->symnode, c->symoff,
                       c->symnorm, U, nc, 1);
  if (c->nfarnode)
    hipLaunchKernelGGL(k_farbc, dim3(nblocks(c->nfarnode)), dim3(kBlock), 0,
                       c->stream, c->nfarnode, nc, c->farnode, c->faroff, c->farnorm,
                       c->far[0], c->far[1], c->far[2], c->far[3], c->far[4],
                       c->cfg.gamma, U);
  if (c->nprenode)
    hipLaunchKernelGGL(k_prebc, dim3(nblocks(c->nprenode)), dim3(kBlock), 0,
                       c->stream, c->nprenode, nc, c->prenode, c->preoff, c->preval,
                       c->cfg.gamma, U);
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

template <int NC>
void launch_update_nc(xg_ctx* c, int stage, double rk, double dt, const double* dtp,
                      double* U, double* Un, const double* R) {
  const int64_t n = (int64_t)c->npoin * NC;
  if (dtp) {
    if (stage == 0)
      hipLaunchKernelGGL((k_update_steady<true, NC>), dim3(nblocks(n)), dim3(kBlock), 0,
                         c->stream, c->npoin, rk, dtp, U, Un, R, c->vol);
    else
      hipLaunchKernelGGL((k_update_steady<false, NC>), dim3(nblocks(n)), dim3(kBlock), 0,
                         c->stream, c->npoin, rk, dtp, U, Un, R, c->vol);
  } else if (stage == 0) {
    hipLaunchKernelGGL((k_update<true, NC>), dim3(nblocks(n)), dim3(kBlock), 0, c->stream,
                       c->npoin, rk * dt, U, Un, R, c->vol);
  } else {
    hipLaunchKernelGGL((k_update<false, NC>), dim3(nblocks(n)), dim3(kBlock), 0, c->stream,
                       c->npoin, rk * dt, U, Un, R, c->vol);
  }
}

// RieCG::solve (RieCG.cpp:992-1057) after the rhs is complete
int launch_solve(xg_ctx* c, int stage, double dt, const double* dtp, double* tp,
                 double* U, double* Un, const double* R) {
  static const double rkcoef[3] = {1.0 / 3.0, 1.0 / 2.0, 1.0};
  const double rk = rkcoef[stage];
  if (c->ncomp == 5) launch_update_nc<5>(c, stage, rk, dt, dtp, U, Un, R);
  else if (c->ncomp == 6) launch_update_nc<6>(c, stage, rk, dt, dtp, U, Un, R);
  else launch_update_nc<7>(c, stage, rk, dt, dtp, U, Un, R);
  int rc = launch_bc(c, U);
  if (rc) return rc;
  if (dtp && stage == 2)
    hipLaunchKernelGGL(k_axpy1, dim3(nblocks(c->npoin)), dim3(kBlock), 0, c->stream,
                       (int64_t)c->npoin, dtp, tp);
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

// (node, record) lists grouped by node, records of a node in list order
template <int W>
int group_by_node(xg_ctx* c, int64_t n, const size_t* nodes, const double* rec,
                  std::vector<int>& node, std::vector<int>& off,
                  std::vector<double>& out, const char* what) {
  std::vector<int64_t> order(n);
  for (int64_t i = 0; i < n; ++i) {
    if (nodes[i] >= (size_t)c->npoin)
      return fail(c, XG_EINVAL, std::string("xg_riecg_bc: ") + what + " node out of range");
    order[i] = i;
  }
  std::stable_sort(order.begin(), order.end(),
                   [&](int64_t a, int64_t b) { return nodes[a] < nodes[b]; });
  off.assign(1, 0);
  node.clear();
  out.clear();
  for (int64_t k = 0; k < n; ++k) {
    int64_t i = order[k];
    if (k == 0 || nodes[order[k - 1]] != nodes[i]) {
      if (k) off.push_back((int)(out.size() / W));
      node.push_back((int)nodes[i]);
    }
    out.insert(out.end(), rec + i * W, rec + i * W + W);
  }
  if (n) off.push_back((int)(out.size() / W));
  return XG_OK;
}

// uploads the riemann::rhs layout (its block tables, edge records, chunk
// entry lists, boundary faces, halo slots and fix-up lists)
int upload_blocks(xg_ctx* c, std::vector<DevArr>& M, const xg::Layout& L,
                  xg_ctx::EdgeBlocks& B) {
  std::vector<int4> b0(L.blk.size()), b1(L.blk.size());
  for (size_t b = 0; b < L.blk.size(); ++b) {
    const auto& K = L.blk[b];
    b0[b] = make_int4(K.own0, K.nown, K.nloc, K.halo_off);
    b1[b] = make_int4(K.slot0, K.chunk0, K.chunk1, 0);
  }
  std::vector<int4> c0(L.chunks.size());
  std::vector<int> c1(L.chunks.size());
  for (size_t i = 0; i < L.chunks.size(); ++i) {
    const auto& C = L.chunks[i];
    c0[i] = make_int4(C.kind, C.first, C.count, C.tend_off);
    c1[i] = C.ent_off;
  }
  int rc;
  if ((rc = upload(c, M, &B.blk0, b0)) || (rc = upload(c, M, &B.blk1, b1)) ||
      (rc = upload(c, M, &B.halo, L.halo)) || (rc = upload(c, M, &B.chk, c0)) ||
      (rc = upload(c, M, &B.chk_ent, c1)) || (rc = upload(c, M, &B.tend, L.tend)) ||
      (rc = upload(c, M, &B.entries, L.entries)) || (rc = upload(c, M, &B.elpq, L.elpq)) ||
      (rc = upload(c, M, &B.dx, L.dx)) || (rc = upload(c, M, &B.dy, L.dy)) ||
      (rc = upload(c, M, &B.dz, L.dz)) || (rc = upload(c, M, &B.fab, L.fab)) ||
      (rc = upload(c, M, &B.fcs, L.fcs)) ||
      (rc = dev_alloc(c, M, (void**)&B.slots,
                      (size_t)L.nslot * XG_MAX_NCOMP * sizeof(double))) ||
      (rc = upload(c, M, &B.fx_node, L.fx_node)) || (rc = upload(c, M, &B.fx_off, L.fx_off)) ||
      (rc = upload(c, M, &B.fx_slot, L.fx_slot)))
    return rc;
  B.nblk = (int)L.blk.size();
  B.nfx = (int)L.fx_node.size();
  return XG_OK;
}

// device staging of the host-pointer entries for nc components per node
int stage_buffers(xg_ctx* c, int nc) {
  size_t need = (size_t)c->npoin * 8;
  if (c->sbytes >= need && c->snc >= nc) return XG_OK;
  if (c->sU) { (void)hipFree(c->sU); (void)hipFree(c->sG); (void)hipFree(c->sR); }
  c->sU = c->sG = c->sR = nullptr; c->sbytes = 0; c->snc = 0;
  XG_HIP(c, hipMalloc((void**)&c->sU, need * nc));
  XG_HIP(c, hipMalloc((void**)&c->sG, need * (3 * nc + 1)));   // G and, after it, v
  XG_HIP(c, hipMalloc((void**)&c->sR, need * nc));
  c->sbytes = need;
  c->snc = nc;
  return XG_OK;
}

}  // namespace

// =================================================================== C-ABI ==

extern "C" {

int xg_ctx_create(int device, xg_ctx** out) {
  if (!out) return XG_EINVAL;
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return XG_EHIP;
  if (device < 0 || device >= n) return XG_EINVAL;
  if (hipSetDevice(device) != hipSuccess) return XG_EHIP;
  if (xg_diag_scratch_init(device) != XG_OK) return XG_EHIP;
  xg_ctx* c = new xg_ctx;
  c->device = device;
  *out = c;
  return XG_OK;
}

int xg_ctx_destroy(xg_ctx* c) {
  if (!c) return XG_EINVAL;
  (void)hipSetDevice(c->device);
  (void)hipStreamSynchronize(c->stream);
  dev_free_all(c->mesh_allocs);
  dev_free_all(c->riecg_allocs);
  dev_free_all(c->bc_allocs);
  if (c->sU) { (void)hipFree(c->sU); (void)hipFree(c->sG); (void)hipFree(c->sR); }
  if (c->cg) (void)xg_cg_destroy(c);
  if (c->koz) xg_kozak_free(c);
  if (c->cho) xg_chocg_free(c);
  if (c->gnn) xg_gnn_free(c);
  if (c->diagbuf.p) (void)hipFree(c->diagbuf.p);
  if (c->amg) xg_amg_free(c);
  delete c->grows;
  delete c;
  return XG_OK;
}

const char* xg_last_error(const xg_ctx* c) {
  return c ? c->err.c_str() : "null context";
}

int xg_set_stream(xg_ctx* c, void* s) {
  if (!c) return XG_EINVAL;
  c->stream = (hipStream_t)s;
  return XG_OK;
}

int xg_set_config(xg_ctx* c, const xg_config* cfg) {
  if (!c || !cfg) return XG_EINVAL;
  if (cfg->flux != 0 && cfg->flux != 1)
    return fail(c, XG_EINVAL, "Flux not configured");
  if (!(cfg->gamma > 1.0)) return fail(c, XG_EINVAL, "gamma must exceed 1");
  c->cfg = *cfg;
  return XG_OK;
}

int xg_mesh_upload(xg_ctx* c, int64_t npoin, const double* x, const double* y,
                   const double* z, const int64_t nsup[3],
                   const size_t* s0, const double* i0, const size_t* s1,
                   const double* i1, const size_t* s2, const double* i2,
                   int64_t ntri, const size_t* tri, const uint8_t* besym) {
  if (!c) return XG_EINVAL;
  if (npoin <= 0 || npoin >= (1ll << 31) || !x || !y || !z || !nsup)
    return fail(c, XG_EINVAL, "xg_mesh_upload: bad mesh size or coordinates");
  if (nsup[0] < 0 || nsup[1] < 0 || nsup[2] < 0 || ntri < 0 ||
      (nsup[0] && (!s0 || !i0)) || (nsup[1] && (!s1 || !i1)) ||
      (nsup[2] && (!s2 || !i2)) || (ntri && (!tri || !besym)))
    return fail(c, XG_EINVAL, "xg_mesh_upload: missing superedge/face arrays");
  XG_HIP(c, hipSetDevice(c->device));
  // expand superedges into oriented edges, in the reference's loop order
  static const int lpoed[6][2] = {{0,1},{1,2},{2,0},{0,3},{1,3},{2,3}};
  static const int lpoet[3][2] = {{0,1},{1,2},{2,0}};
  int64_t ne = nsup[0] * 6 + nsup[1] * 3 + nsup[2];
  if (ne >= (1ll << 31))
    return fail(c, XG_EINVAL, "xg_mesh_upload: too many edges");
  std::vector<int> p(ne), q(ne);
  std::vector<double> d(ne * 3);
  int64_t k = 0;
  auto push = [&](size_t a, size_t b, const double* D) {
    p[k] = (int)std::min<size_t>(a, (size_t)INT32_MAX);
    q[k] = (int)std::min<size_t>(b, (size_t)INT32_MAX);
    d[k * 3 + 0] = D[0]; d[k * 3 + 1] = D[1]; d[k * 3 + 2] = D[2];
    ++k;
  };
  for (int64_t e = 0; e < nsup[0]; ++e)
    for (int j = 0; j < 6; ++j)
      push(s0[e * 4 + lpoed[j][0]], s0[e * 4 + lpoed[j][1]], i0 + (e * 6 + j) * 3);
  for (int64_t e = 0; e < nsup[1]; ++e)
    for (int j = 0; j < 3; ++j)
      push(s1[e * 3 + lpoet[j][0]], s1[e * 3 + lpoet[j][1]], i1 + (e * 3 + j) * 3);
  for (int64_t e = 0; e < nsup[2]; ++e) push(s2[e * 2], s2[e * 2 + 1], i2 + e * 3);
  for (int64_t e = 0; e < ne; ++e)
    if (p[e] < 0 || q[e] < 0 || p[e] >= npoin || q[e] >= npoin || p[e] == q[e])
      return fail(c, XG_EINVAL, "xg_mesh_upload: superedge node id out of range");
  for (int64_t f = 0; f < ntri * 3; ++f)
    if (tri[f] >= (size_t)npoin)
      return fail(c, XG_EINVAL, "xg_mesh_upload: boundary face node out of range");
  std::vector<int> tri32(ntri * 3);
  for (int64_t f = 0; f < ntri * 3; ++f) tri32[f] = (int)tri[f];
  xg::RowLayout L;
  xg::Layout LR;
  int lanes = 1;
  int rc = xg::build_grad_rows((int)npoin, p, q, d, ntri, tri32.data(), L, lanes, c->err);
  if (rc) return rc;
  rc = xg::build_rhs_layout((int)npoin, p, q, d, ntri, tri32.data(), besym, LR, c->err);
  if (rc) return rc;
  // normals of the rows' boundary faces, (b - a) x (c - a) / 12
  std::vector<double> fn(L.fidx.size() * 3, 0.0);
  for (size_t i = 0; i < L.fidx.size(); ++i) {
    if (L.fidx[i] < 0) continue;
    const size_t* N = tri + L.fidx[i] * 3;
    const double ax = x[N[1]] - x[N[0]], ay = y[N[1]] - y[N[0]], az = z[N[1]] - z[N[0]];
    const double bx = x[N[2]] - x[N[0]], by = y[N[2]] - y[N[0]], bz = z[N[2]] - z[N[0]];
    fn[i * 3 + 0] = (ay * bz - by * az) / 12.0;
    fn[i * 3 + 1] = (az * bx - bz * ax) / 12.0;
    fn[i * 3 + 2] = (ax * by - bx * ay) / 12.0;
  }
  // device arrays
  (void)hipStreamSynchronize(c->stream);
  dev_free_all(c->mesh_allocs);
  c->have_mesh = false;
  auto& M = c->mesh_allocs;
  if ((rc = upload(c, M, &c->x, x, npoin)) || (rc = upload(c, M, &c->y, y, npoin)) ||
      (rc = upload(c, M, &c->z, z, npoin)))
    return rc;
  if (!c->grows) c->grows = new RowsDev;
  if ((rc = upload_rows(c, M, L, fn, lanes, *c->grows))) return rc;
  if ((rc = upload_blocks(c, M, LR, c->rb))) return rc;
  c->npoin = (int)npoin;
  c->nedge = ne;
  c->have_mesh = true;
  c->have_riecg = false;
  return XG_OK;
}

int xg_mesh_device_bytes(const xg_ctx* c, int64_t* bytes) {
  if (!c || !bytes) return XG_EINVAL;
  int64_t b = 0;
  for (auto& a : c->mesh_allocs) b += (int64_t)a.bytes;
  *bytes = b;
  return XG_OK;
}

int xg_riemann_grad_dev(xg_ctx* c, int ncomp, const double* U, double* G) {
  int rc = check_mesh(c, ncomp);
  if (rc) return rc;
  if (!U || !G) return fail(c, XG_EINVAL, "xg_riemann_grad: null field");
  XG_HIP(c, hipSetDevice(c->device));
  return launch_grad(c, ncomp, U, G);
}

int xg_riemann_rhs_dev(xg_ctx* c, int ncomp, const double* G, const double* U,
                       const double* v, double t, const double* tp, double* R) {
  (void)t;   // the sources served do not depend on time
  (void)tp;
  int rc = check_mesh(c, ncomp);
  if (rc) return rc;
  if (!U || !G || !R) return fail(c, XG_EINVAL, "xg_riemann_rhs: null field");
  if (xg::has_source(prob_of(c)) && !v)
    return fail(c, XG_EINVAL, "xg_riemann_rhs: the problem's source needs the nodal volumes v");
  XG_HIP(c, hipSetDevice(c->device));
  return launch_rhs(c, ncomp, G, U, R, v);
}

int xg_riemann_grad(xg_ctx* c, int ncomp, const double* U, double* G) {
  int rc = check_mesh(c, ncomp);
  if (rc) return rc;
  if (!U || !G) return fail(c, XG_EINVAL, "xg_riemann_grad: null field");
  XG_HIP(c, hipSetDevice(c->device));
  if ((rc = stage_buffers(c, ncomp))) return rc;
  size_t n = (size_t)c->npoin * 8;
  XG_HIP(c, hipMemcpyAsync(c->sU, U, n * ncomp, hipMemcpyHostToDevice, c->stream));
  if ((rc = launch_grad(c, ncomp, c->sU, c->sG))) return rc;
  XG_HIP(c, hipMemcpyAsync(G, c->sG, n * 3 * ncomp, hipMemcpyDeviceToHost, c->stream));
  XG_HIP(c, hipStreamSynchronize(c->stream));
  return XG_OK;
}

int xg_riemann_rhs(xg_ctx* c, int ncomp, const double* G, const double* U,
                   const double* v, double t, const double* tp, double* R) {
  (void)t;   // the sources served do not depend on time
  (void)tp;
  int rc = check_mesh(c, ncomp);
  if (rc) return rc;
  if (!U || !G || !R) return fail(c, XG_EINVAL, "xg_riemann_rhs: null field");
  const bool src = xg::has_source(prob_of(c));
  if (src && !v)
    return fail(c, XG_EINVAL, "xg_riemann_rhs: the problem's source needs the nodal volumes v");
  XG_HIP(c, hipSetDevice(c->device));
  if ((rc = stage_buffers(c, ncomp))) return rc;
  size_t n = (size_t)c->npoin;
  XG_HIP(c, hipMemcpyAsync(c->sU, U, n * 8 * ncomp, hipMemcpyHostToDevice, c->stream));
  XG_HIP(c, hipMemcpyAsync(c->sG, G, n * 24 * ncomp, hipMemcpyHostToDevice, c->stream));
  // the volumes are staged after G in the G staging buffer (3 ncomp + 1
  // doubles per node)
  double* sv = nullptr;
  if (src) {
    sv = c->sG + n * 3 * ncomp;
    XG_HIP(c, hipMemcpyAsync(sv, v, n * 8, hipMemcpyHostToDevice, c->stream));
  }
  if ((rc = launch_rhs(c, ncomp, c->sG, c->sU, c->sR, sv))) return rc;
  XG_HIP(c, hipMemcpyAsync(R, c->sR, n * 8 * ncomp, hipMemcpyDeviceToHost, c->stream));
  XG_HIP(c, hipStreamSynchronize(c->stream));
  return XG_OK;
}

int xg_riecg_setup(xg_ctx* c, const double* vol, int64_t nsym,
                   const size_t* symnodes, const double* symnorms) {
  if (!c) return XG_EINVAL;
  if (!c->have_mesh) return fail(c, XG_ENOMESH, "no mesh uploaded");
  if (!vol || nsym < 0 || (nsym && (!symnodes || !symnorms)))
    return fail(c, XG_EINVAL, "xg_riecg_setup: bad arguments");
  for (int64_t i = 0; i < c->npoin; ++i)
    if (!(vol[i] > 0)) return fail(c, XG_EINVAL, "xg_riecg_setup: non-positive nodal volume");
  // group the (node, normal) pairs by node, keeping list order per node
  std::vector<int> node, off(1, 0);
  std::vector<double> nrm;
  {
    std::vector<int64_t> order(nsym);
    for (int64_t i = 0; i < nsym; ++i) {
      if (symnodes[i] >= (size_t)c->npoin)
        return fail(c, XG_EINVAL, "xg_riecg_setup: symmetry node out of range");
      order[i] = i;
    }
    std::stable_sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
      return symnodes[a] < symnodes[b];
    });
    for (int64_t k = 0; k < nsym; ++k) {
      int64_t i = order[k];
      if (k == 0 || symnodes[order[k - 1]] != symnodes[i]) {
        if (k) off.push_back((int)(nrm.size() / 3));
        node.push_back((int)symnodes[i]);
      }
      nrm.insert(nrm.end(), symnorms + i * 3, symnorms + i * 3 + 3);
    }
    if (nsym) off.push_back((int)(nrm.size() / 3));
  }
  XG_HIP(c, hipSetDevice(c->device));
  (void)hipStreamSynchronize(c->stream);
  dev_free_all(c->riecg_allocs);
  dev_free_all(c->bc_allocs);
  c->ndirnode = c->nfarnode = c->nprenode = 0;
  c->have_riecg = false;
  c->ncomp = 5;
  int rc;
  auto& L = c->riecg_allocs;
  if ((rc = upload(c, L, &c->vol, vol, (size_t)c->npoin)) ||
      (rc = upload(c, L, &c->symnode, node)) || (rc = upload(c, L, &c->symoff, off)) ||
      (rc = upload(c, L, &c->symnorm, nrm)) ||
      (rc = dev_alloc(c, L, (void**)&c->red, sizeof(double) * (kRedBlocks + 1))))
    return rc;
  c->nsymnode = (int)node.size();
  c->have_riecg = true;
  return XG_OK;
}

int xg_riecg_set_ncomp(xg_ctx* c, int ncomp) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  int rc = check_ncomp(c, ncomp);
  if (rc) return rc;
  if (ncomp != c->ncomp) {
    // the Dirichlet masks and values are per component: drop the lists
    XG_HIP(c, hipSetDevice(c->device));
    (void)hipStreamSynchronize(c->stream);
    dev_free_all(c->bc_allocs);
    c->ndirnode = c->nfarnode = c->nprenode = 0;
  }
  c->ncomp = ncomp;
  return XG_OK;
}

int xg_riecg_dt_dev(xg_ctx* c, const double* U, double cfl, double* dt) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (!U || !dt) return fail(c, XG_EINVAL, "xg_riecg_dt: null argument");
  XG_HIP(c, hipSetDevice(c->device));
  int nb = (int)std::min<int64_t>(kRedBlocks, std::max<int64_t>(1, nblocks(c->npoin)));
  hipLaunchKernelGGL(k_dt_partial, dim3(nb), dim3(kBlock), 0, c->stream,
                     c->npoin, c->ncomp, U, c->vol, c->cfg.gamma, c->red);
  hipLaunchKernelGGL(k_min_final, dim3(1), dim3(kRedBlocks), 0, c->stream, nb,
                     c->red, cfl, c->red + kRedBlocks);
  XG_HIP(c, hipGetLastError());
  XG_HIP(c, hipMemcpyAsync(dt, c->red + kRedBlocks, sizeof(double),
                           hipMemcpyDeviceToHost, c->stream));
  XG_HIP(c, hipStreamSynchronize(c->stream));
  if (*dt < 2.220446049250313e-16)
    return fail(c, XG_EBLOWUP, "time step below machine epsilon");
  return XG_OK;
}

int xg_riecg_dt_steady_dev(xg_ctx* c, const double* U, double cfl, double* dtp,
                           double* dt) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (!U || !dtp || !dt) return fail(c, XG_EINVAL, "xg_riecg_dt_steady: null argument");
  XG_HIP(c, hipSetDevice(c->device));
  int nb = (int)std::min<int64_t>(kRedBlocks, std::max<int64_t>(1, nblocks(c->npoin)));
  hipLaunchKernelGGL(k_dt_steady, dim3(nb), dim3(kBlock), 0, c->stream, c->npoin,
                     c->ncomp, U, c->vol, c->cfg.gamma, cfl, dtp, c->red);
  hipLaunchKernelGGL(k_min_final, dim3(1), dim3(kRedBlocks), 0, c->stream, nb,
                     c->red, 1.0, c->red + kRedBlocks);
  XG_HIP(c, hipGetLastError());
  XG_HIP(c, hipMemcpyAsync(dt, c->red + kRedBlocks, sizeof(double),
                           hipMemcpyDeviceToHost, c->stream));
  XG_HIP(c, hipStreamSynchronize(c->stream));
  if (*dt < 2.220446049250313e-16)
    return fail(c, XG_EBLOWUP, "time step below machine epsilon");
  return XG_OK;
}

int xg_riecg_bc(xg_ctx* c, int64_t ndir, const size_t* dirnodes, const int32_t* dirmask,
                const double* dirvals, int64_t nfar, const size_t* farnodes,
                const double* farnorms, const double far[5], int64_t npre,
                const size_t* prenodes, const double* prevals) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (ndir < 0 || nfar < 0 || npre < 0 ||
      (ndir && (!dirnodes || !dirmask || !dirvals)) ||
      (nfar && (!farnodes || !farnorms || !far)) || (npre && (!prenodes || !prevals)))
    return fail(c, XG_EINVAL, "xg_riecg_bc: bad arguments");
  const int nc = c->ncomp;
  std::vector<int> dn(ndir);
  std::vector<uint8_t> dm(ndir * nc);
  for (int64_t i = 0; i < ndir; ++i) {
    if (dirnodes[i] >= (size_t)c->npoin)
      return fail(c, XG_EINVAL, "xg_riecg_bc: Dirichlet node out of range");
    dn[i] = (int)dirnodes[i];
    for (int k = 0; k < nc; ++k) dm[i * nc + k] = (uint8_t)(dirmask[i * nc + k] == 1);
  }
  std::vector<int> fnode, foff, pnode, poff;
  std::vector<double> fnrm, pval;
  int rc;
  if ((rc = group_by_node<3>(c, nfar, farnodes, farnorms, fnode, foff, fnrm, "farfield")) ||
      (rc = group_by_node<2>(c, npre, prenodes, prevals, pnode, poff, pval, "pressure")))
    return rc;
  if (nfar && !(far[0] > 0.0 && far[4] > 0.0))
    return fail(c, XG_EINVAL, "xg_riecg_bc: farfield density and pressure must be positive");
  XG_HIP(c, hipSetDevice(c->device));
  (void)hipStreamSynchronize(c->stream);
  dev_free_all(c->bc_allocs);
  c->ndirnode = c->nfarnode = c->nprenode = 0;
  auto& L = c->bc_allocs;
  if ((rc = upload(c, L, &c->dirnode, dn)) || (rc = upload(c, L, &c->dirmask, dm)) ||
      (rc = upload(c, L, &c->dirval, dirvals, (size_t)ndir * nc)) ||
      (rc = upload(c, L, &c->farnode, fnode)) || (rc = upload(c, L, &c->faroff, foff)) ||
      (rc = upload(c, L, &c->farnorm, fnrm)) || (rc = upload(c, L, &c->prenode, pnode)) ||
      (rc = upload(c, L, &c->preoff, poff)) || (rc = upload(c, L, &c->preval, pval)))
    return rc;
  if (nfar)
    for (int k = 0; k < 5; ++k) c->far[k] = far[k];
  c->ndirnode = (int)ndir;
  c->nfarnode = (int)fnode.size();
  c->nprenode = (int)pnode.size();
  return XG_OK;
}

int xg_riecg_apply_bc_dev(xg_ctx* c, double* U) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (!U) return fail(c, XG_EINVAL, "xg_riecg_apply_bc: null field");
  XG_HIP(c, hipSetDevice(c->device));
  return launch_bc(c, U);
}

int xg_riecg_stage_dev(xg_ctx* c, int stage, double t, double dt, const double* dtp,
                       double* tp, double* U, double* Un, double* G, double* R) {
  (void)t;   // BC values and sources served are independent of time
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (stage < 0 || stage > 2) return fail(c, XG_EINVAL, "stage must be 0, 1 or 2");
  if (!U || !Un || !G || !R) return fail(c, XG_EINVAL, "xg_riecg_stage: null field");
  if ((dtp == nullptr) != (tp == nullptr))
    return fail(c, XG_EINVAL, "xg_riecg_stage: dtp and tp go together");
  XG_HIP(c, hipSetDevice(c->device));
  int rc;
  if ((rc = launch_grad(c, c->ncomp, U, G, true))) return rc;
  if ((rc = launch_rhs(c, c->ncomp, G, U, R, c->vol))) return rc;
  return launch_solve(c, stage, dt, dtp, tp, U, Un, R);
}

int xg_riecg_grad_div_dev(xg_ctx* c, double* G) {
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (!G) return fail(c, XG_EINVAL, "xg_riecg_grad_div: null field");
  XG_HIP(c, hipSetDevice(c->device));
  const int64_t n = (int64_t)c->npoin * 3 * c->ncomp;
  if (c->ncomp == 5)
    hipLaunchKernelGGL(k_div_vol<15>, dim3(nblocks(n)), dim3(kBlock), 0, c->stream,
                       c->npoin, G, c->vol);
  else if (c->ncomp == 6)
    hipLaunchKernelGGL(k_div_vol<18>, dim3(nblocks(n)), dim3(kBlock), 0, c->stream,
                       c->npoin, G, c->vol);
  else
    hipLaunchKernelGGL(k_div_vol<21>, dim3(nblocks(n)), dim3(kBlock), 0, c->stream,
                       c->npoin, G, c->vol);
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

int xg_riecg_solve_dev(xg_ctx* c, int stage, double t, double dt, const double* dtp,
                       double* tp, double* U, double* Un, const double* R) {
  (void)t;
  if (!c) return XG_EINVAL;
  if (!c->have_riecg) return fail(c, XG_ENOMESH, "xg_riecg_setup not called");
  if (stage < 0 || stage > 2) return fail(c, XG_EINVAL, "stage must be 0, 1 or 2");
  if (!U || !Un || !R) return fail(c, XG_EINVAL, "xg_riecg_solve: null field");
  if ((dtp == nullptr) != (tp == nullptr))
    return fail(c, XG_EINVAL, "xg_riecg_solve: dtp and tp go together");
  XG_HIP(c, hipSetDevice(c->device));
  return launch_solve(c, stage, dt, dtp, tp, U, Un, R);
}

int xg_set_problem(xg_ctx* c, const xg_problem* p) {
  if (!c || !p) return XG_EINVAL;
  if (p->kind != XG_PROBLEM_NONE && p->kind != XG_PROBLEM_VORTICAL_FLOW &&
      p->kind != XG_PROBLEM_TAYLOR_GREEN && p->kind != XG_PROBLEM_SLOT_CYL)
    return fail(c, XG_EUNSUPPORTED, "xg_set_problem: no device source for this problem");
  c->problem = *p;
  return XG_OK;
}

int xg_get_problem(const xg_ctx* c, xg_problem* p) {
  if (!c || !p) return XG_EINVAL;
  *p = c->problem;
  return XG_OK;
}

}  // extern "C"
