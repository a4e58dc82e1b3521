// Device side of the smoothed-aggregation AMG preconditioner (no
// counterpart in the reference; setup in xg_amg.cpp).
//
// The hierarchy lives in HBM in FP32 (values), each matrix in row tiles with
// column lists (xg_tiles.hpp): per level the operator B_l, 1/diag(B_l), the
// prolongator P_l and R_l = P_l^T; the coarsest operator's dense inverse.
// One application is a symmetric V(1,1)-cycle on B = S A (S = sign(diag A))
// for the right-hand side S r.  Per level four kernels: the residual of the
// damped-Jacobi sweep from zero, its restriction (which also takes that
// first sweep of the level below), then on the way up the prolongation and
// the second sweep; the finest level's second sweep leaves z as flexible
// CG's SpMV and beta read it.  Every kernel has a fixed summation order, so
// applications are bitwise reproducible.
//
// What bounds it: bytes on the finest level (B twice, P and R: 82 MB at 64^3
// in FP32, 16 us at the copy rate) and the latency of a launch and of
// its chain of loads on the others (4 to 6 us each).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "xg_amg.hpp"
#include "xg_ctx.hpp"
#include "xg_tiles_dev.hpp"

using namespace xgd;

struct AmgDevMat {
  xg::TileMat M;
  float* a = nullptr;
};

struct AmgDevLevel {
  int n = 0;
  float* dinv = nullptr;
  float omega = 0.f;
  AmgDevMat B, P, R;
  // right-hand side, its first sweep and prolonged correction, residual,
  // result
  float *b = nullptr, *x = nullptr, *r = nullptr, *y = nullptr;
};

struct AmgDev {
  int64_t version = -1;
  std::vector<AmgDevLevel> lev;
  float* cinv = nullptr;
  float* sign = nullptr;        // S of the fine level
  std::vector<DevArr> allocs;
  double op_complexity = 0.0, setup_ms = 0.0;
};

namespace {

constexpr int kT = kTileThreads;

struct VecSource {
  using Raw = float;
  const float* v;
  __device__ float load(unsigned c) const { return v[c]; }
  __device__ float value(float x) const { return x; }
};

// r = b - B x
struct ResidualRow {
  using Raw = float;
  const float* b;
  float* r;
  __device__ Raw load(int i) const { return b[i]; }
  __device__ void apply(int i, Raw bi, float s) { r[i] = bi - s; }
};

// b = R r of the level below, and its first sweep x = w D^-1 b
struct RestrictRow {
  using Raw = float;
  const float* dinv;
  float w;
  float *b, *x;
  __device__ Raw load(int i) const { return w * dinv[i]; }
  __device__ void apply(int i, Raw wd, float s) {
    b[i] = s;
    x[i] = wd * s;
  }
};

// x += P y of the level below
struct ProlongRow {
  using Raw = float;
  float* x;
  __device__ Raw load(int i) const { return x[i]; }
  __device__ void apply(int i, Raw xi, float s) { x[i] = xi + s; }
};

// y = x + w D^-1 (b - B x)
struct SweepRow {
  struct Raw {
    float x, b, wd;
  };
  const float *x, *b, *dinv;
  float w;
  float* y;
  __device__ Raw load(int i) const { return Raw{x[i], b[i], w * dinv[i]}; }
  __device__ void apply(int i, const Raw& o, float s) { y[i] = o.x + o.wd * (o.b - s); }
};

// the same on the finest level: z, as the pairs (z, p) and in (z, q)
struct LastSweepRow {
  struct Raw {
    float x, b, wd;
    double p, q;
  };
  const float *x, *b, *dinv;
  float w;
  const double *p, *q;
  double2* zp;
  double zq;
  __device__ Raw load(int i) const {
    return Raw{x[i], b[i], w * dinv[i], p ? p[i] : 0.0, p ? q[i] : 0.0};
  }
  __device__ void apply(int i, const Raw& o, float s) {
    const double z = (double)(o.x + o.wd * (o.b - s));
    zp[i] = make_double2(z, o.p);
    zq += z * o.q;
  }
};

__device__ inline double block_sum(double v, double* sm) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kT / 64; ++k) s += sm[k];
  return s;
}

template <class Row>
__global__ __launch_bounds__(kT) void k_amg_rows(xg::TileMat M, const float* __restrict__ a,
                                                VecSource src, Row row,
                                                const int* __restrict__ done) {
  __shared__ TileLds<float> lds;
  const int stop = *done;
  tiles_spmv<float, true, 3>(M, a, src, row, [&]() { return !stop; }, lds);
}

__global__ __launch_bounds__(kT) void k_amg_last(xg::TileMat M, const float* __restrict__ a,
                                                VecSource src, LastSweepRow row,
                                                double* __restrict__ part,
                                                const int* __restrict__ done) {
  __shared__ TileLds<float> lds;
  const int stop = *done;
  if (!tiles_spmv<float, true, 3>(M, a, src, row, [&]() { return !stop; }, lds)) return;
  const double s = block_sum(row.zq, lds.sm[0]);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// x = C b with C the dense coarsest inverse (one workgroup per row)
__global__ __launch_bounds__(kT) void k_amg_dense(int n, const float* __restrict__ C,
                                                 const float* __restrict__ b,
                                                 float* __restrict__ x,
                                                 const int* __restrict__ done) {
  __shared__ float sm[kT / 64];
  const int stop = *done;
  const int row = blockIdx.x;
  float s = 0.f;
  for (int j = threadIdx.x; j < n; j += kT) s += C[(size_t)row * n + j] * b[j];
  if (stop) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < kT / 64; ++k) t += sm[k];
    x[row] = t;
  }
}

// the pairs (z, p) and partials of (z, q) where the finest level is the
// dense one
__global__ __launch_bounds__(kT) void k_amg_out(int n, const float* __restrict__ x,
                                               const double* __restrict__ p,
                                               const double* __restrict__ q,
                                               double2* __restrict__ zp,
                                               double* __restrict__ part,
                                               const int* __restrict__ done) {
  __shared__ double sm[kT / 64];
  if (*done) return;
  double zq = 0.0;
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) {
    const double z = (double)x[i];
    zp[i] = make_double2(z, p ? p[i] : 0.0);
    if (p) zq += z * q[i];
  }
  const double s = block_sum(zq, sm);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

int nb(int n) { return std::max(1, (n + kT - 1) / kT); }

template <class T>
int up(xg_ctx* c, std::vector<DevArr>& L, T** d, const std::vector<T>& v) {
  return upload(c, L, d, v);
}

std::vector<int> to_i32(const std::vector<int64_t>& v) { return std::vector<int>(v.begin(), v.end()); }
std::vector<float> to_f32(const std::vector<double>& v) { return std::vector<float>(v.begin(), v.end()); }

void free_dev(AmgDev* m) {
  if (!m) return;
  dev_free_all(m->allocs);
  delete m;
}

int up_mat(xg_ctx* c, std::vector<DevArr>& L, const xg::Csr& A, AmgDevMat& D) {
  xg::TileSet t;
  xg::build_tiles(A.nrow, A.ncol, A.ia.data(), A.ja.data(), t);
  xg::Tile* tile;
  int *ia, *ja = nullptr, *ucol;
  uint16_t* lidx;
  int rc;
  if ((rc = up(c, L, &ia, to_i32(A.ia))) || (t.has_long && (rc = up(c, L, &ja, A.ja))) ||
      (rc = up(c, L, &D.a, to_f32(A.a))) || (rc = up(c, L, &tile, t.tile)) ||
      (rc = upload(c, L, &ucol, t.ucol)) || (rc = upload(c, L, &lidx, t.lidx)))
    return rc;
  D.M = xg::TileMat{(int)t.tile.size(), tile, ia, ja, ucol, lidx};
  return XG_OK;
}

int grid_of(const AmgDevMat& D) { return std::max(1, std::min(D.M.ntile, kSpmvGrid)); }

template <class Row>
void rows(xg_ctx* c, const AmgDevMat& D, const float* v, const Row& row, const int* done) {
  hipLaunchKernelGGL(k_amg_rows<Row>, dim3(grid_of(D)), dim3(kT), 0, c->stream, D.M, D.a,
                     VecSource{v}, row, done);
}

// y of level l from its b and x = w D^-1 b; the finest level (l = 0, not the
// coarsest) leaves its second sweep to the caller
void vcycle(xg_ctx* c, AmgDev* m, size_t l, const int* done) {
  AmgDevLevel& L = m->lev[l];
  if (l + 1 == m->lev.size()) {
    hipLaunchKernelGGL(k_amg_dense, dim3(L.n), dim3(kT), 0, c->stream, L.n, m->cinv, L.b, L.y,
                       done);
    return;
  }
  AmgDevLevel& C = m->lev[l + 1];
  rows(c, L.B, L.x, ResidualRow{L.b, L.r}, done);
  rows(c, L.R, L.r, RestrictRow{C.dinv, C.omega, C.b, C.x}, done);
  vcycle(c, m, l + 1, done);
  rows(c, L.P, C.y, ProlongRow{L.x}, done);
  if (l > 0) rows(c, L.B, L.x, SweepRow{L.x, L.b, L.dinv, L.omega, L.y}, done);
}

}  // namespace

void xg_amg_free(xg_ctx* c) {
  free_dev(c->amg);
  c->amg = nullptr;
}

int xg_amg_prepare_internal(xg_ctx* c, int64_t n, const int64_t* ia, const int32_t* ja,
                            const double* a, int64_t version, const xg::TileMat& fine) {
  if (c->amg && c->amg->version == version) return XG_OK;
  if (n >= (1ll << 31) || ia[n] >= (1ll << 31))
    return fail(c, XG_EUNSUPPORTED, "AMG: more than 2^31 rows or nonzeros");
  xg::AmgHierarchy h;
  xg::AmgOptions opt;
  std::string err;
  int rc = xg::amg_setup(n, ia, ja, a, opt, h, err);
  if (rc) return fail(c, rc, err);
  XG_HIP(c, hipStreamSynchronize(c->stream));
  xg_amg_free(c);
  AmgDev* m = new AmgDev;
  auto& L = m->allocs;
  std::vector<float> sg(n);
  for (int64_t i = 0; i < n; ++i) {
    double d = 0.0;
    for (int64_t p = ia[i]; p < ia[i + 1]; ++p)
      if (ja[p] == i) d = a[p];
    sg[i] = d < 0.0 ? -1.f : 1.f;
  }
  if ((rc = up(c, L, &m->sign, sg))) { free_dev(m); return rc; }
  m->lev.resize(h.lev.size());
  for (size_t l = 0; l < h.lev.size(); ++l) {
    const xg::AmgLevel& H = h.lev[l];
    AmgDevLevel& D = m->lev[l];
    D.n = (int)H.B.nrow;
    D.omega = (float)H.omega;
    const size_t nn = (size_t)std::max(1, D.n);
    const bool coarsest = l + 1 == h.lev.size();
    if ((rc = up(c, L, &D.dinv, to_f32(H.dinv))) ||
        (rc = dev_alloc(c, L, (void**)&D.x, nn * 4)) ||
        (rc = dev_alloc(c, L, (void**)&D.b, nn * 4)) ||
        (rc = dev_alloc(c, L, (void**)&D.r, nn * 4)) ||
        (rc = dev_alloc(c, L, (void**)&D.y, nn * 4)) ||
        (!coarsest && ((rc = l ? up_mat(c, L, H.B, D.B) : up(c, L, &D.B.a, to_f32(H.B.a))) || (rc = up_mat(c, L, H.P, D.P)) ||
                       (rc = up_mat(c, L, H.R, D.R))))) {
      free_dev(m);
      return rc;
    }
    if (l == 0) D.B.M = fine;
  }
  if ((rc = up(c, L, &m->cinv, to_f32(h.cinv)))) { free_dev(m); return rc; }
  m->version = version;
  m->op_complexity = h.op_complexity;
  m->setup_ms = h.setup_ms;
  c->amg = m;
  return XG_OK;
}

AmgInput xg_amg_input(xg_ctx* c) {
  AmgDev* m = c->amg;
  AmgDevLevel& F = m->lev[0];
  return AmgInput{F.n, m->sign, F.dinv, F.omega, F.b, F.x};
}

int xg_amg_apply_fcg(xg_ctx* c, const double* p, const double* q, double* zp, double* part,
                     const int* done, int* npart) {
  AmgDev* m = c->amg;
  if (!m) return fail(c, XG_ENOMESH, "AMG hierarchy not built");
  AmgDevLevel& F = m->lev[0];
  double2* pairs = reinterpret_cast<double2*>(zp);
  vcycle(c, m, 0, done);
  if (m->lev.size() == 1) {
    *npart = std::min(nb(F.n), kSpmvGrid);
    hipLaunchKernelGGL(k_amg_out, dim3(*npart), dim3(kT), 0, c->stream, F.n, F.y, p, q, pairs,
                       part, done);
  } else {
    *npart = grid_of(F.B);
    hipLaunchKernelGGL(k_amg_last, dim3(*npart), dim3(kT), 0, c->stream, F.B.M, F.B.a,
                       VecSource{F.x}, LastSweepRow{F.x, F.b, F.dinv, F.omega, p, q, pairs, 0.0},
                       part, done);
  }
  XG_HIP(c, hipGetLastError());
  return XG_OK;
}

extern "C" int xg_amg_info(xg_ctx* c, int* levels, double* op_complexity, double* setup_ms) {
  if (!c) return XG_EINVAL;
  if (!c->amg) return fail(c, XG_ENOMESH, "AMG hierarchy not built");
  if (levels) *levels = (int)c->amg->lev.size();
  if (op_complexity) *op_complexity = c->amg->op_complexity;
  if (setup_ms) *setup_ms = c->amg->setup_ms;
  return XG_OK;
}
