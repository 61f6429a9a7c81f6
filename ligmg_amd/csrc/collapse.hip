// The coarse levels of a V-cycle as one dense matrix.
//
// A V-cycle with fixed smoothers is linear, so the cycle from a level of n
// vertices down is an n x n matrix.  For the first level that collapse_fits
// takes, setup forms it: every operation of the cycle runs once on all n unit
// vectors (row-major blocks of n columns, a thread per column), about ten
// launches per level.  The solve
// then replaces the whole coarse recursion, a chain of small dependent
// launches, by one dense product.
#include <algorithm>

#include "../../include/ligmg_amd.h"
#include "collapse.hpp"
#include "prims.hpp"

namespace lg {

namespace {

// Epilogues: row i's sum s for column c at o = i * ld + c.
struct WStore {
  double *y;
  __device__ __forceinline__ void operator()(int64_t, int64_t o, double s) const { y[o] = s; }
};
struct WResid {
  const double *b;
  double *r;
  __device__ __forceinline__ void operator()(int64_t, int64_t o, double s) const { r[o] = b[o] - s; }
};
struct WCheb {
  const double *dinv, *b, *xc, *xp;  // null xp: zero previous iterate
  double *xn;
  double alpha, beta;
  __device__ __forceinline__ void operator()(int64_t i, int64_t o, double s) const {
    const double c = xc[o], d = alpha * (c - (xp ? xp[o] : 0.0));
    xn[o] = c + d + beta * dinv[i] * (b[o] - s);
  }
};
struct WInterp {
  const double *q, *b;
  double *x;
  __device__ __forceinline__ void operator()(int64_t i, int64_t o, double s) const { x[o] = s + q[i] * b[o]; }
};

// One workgroup per row and 256 columns: the row's columns and values are
// the same for every lane (scalar loads), the lanes read 256 adjacent
// entries of a row of X.  16 reads in flight: a row of a coarse power-law
// operator may hold all n columns.
template <class Epi>
__global__ void __launch_bounds__(256) k_wide(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                              const double *__restrict__ v, const double *__restrict__ X,
                                              int64_t ld, Epi epi) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= ld) return;
  const int a = rp[i], b = rp[i + 1];
  double s = 0;
#pragma unroll 16
  for (int k = a; k < b; k++) s += (v ? v[k] : 1.0) * X[(int64_t)ci[k] * ld + c];
  epi(i, i * ld + c, s);
}

__global__ void __launch_bounds__(256) k_wide_dense(const double *__restrict__ P, int64_t n,
                                                    const double *__restrict__ X, int64_t ld, double *Y) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= ld) return;
  double s = 0;
#pragma unroll 16
  for (int64_t k = 0; k < n; k++) s += P[i * n + k] * X[k * ld + c];
  Y[i * ld + c] = s;
}

__global__ void k_wide_cheb0(const double *dinv, const double *b, double *x, double beta, int64_t ld) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ld) x[i * ld + c] = beta * dinv[i] * b[i * ld + c];
}
__global__ void k_wide_prolong(const int32_t *agg, const double *xc, double *x, int64_t ld) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ld) x[i * ld + c] += xc[(int64_t)agg[i] * ld + c];
}
__global__ void k_wide_unit(double *x, int64_t ld) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ld) x[i * ld + c] = i == c ? 1.0 : 0.0;
}
__global__ void k_wide_scale(double *x, double a, int64_t ld) {
  const int64_t i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ld) x[i * ld + c] *= a;
}

struct Wide {
  const std::vector<DLevel> &H;
  const CycleCoeffs &C;
  int64_t ld;
  hipStream_t s;

  dim3 grid(int64_t n) const { return dim3((unsigned)n, (unsigned)((ld + 255) / 256)); }

  template <class Epi>
  void mul(const DCsr &A, const double *X, const Epi &e) const {
    if (A.n == 0) return;  // a level that eliminates every vertex leaves none
    hipLaunchKernelGGL(k_wide<Epi>, grid(A.n), dim3(256), 0, s, A.rp.p, A.ci.p, A.v.p, X, ld, e);
    LG_LAUNCH_CHECK();
  }
  void step(const DLevel &L, const double *b, const double *xc, const double *xp, double *xn, double al,
            double be) const {
    mul(L.A, xc, WCheb{L.dinv.p, b, xc, xp, xn, al, be});
  }

  // Solver::cycle on the block b, into x
  void cycle(size_t l, const double *b, DevBuf<double> &x) const {
    const DLevel &L = H[l];
    const int64_t n = L.A.n;
    if (n == 0) return;
    if (L.kind == LIGMG_LEVEL_COARSE) {
      x.alloc(n * ld);
      hipLaunchKernelGGL(k_wide_dense, grid(n), dim3(256), 0, s, L.pinv.p, n, b, ld, x.p);
      LG_LAUNCH_CHECK();
      return;
    }
    DevBuf<double> bc(H[l + 1].A.n * ld), xc;
    if (L.kind == LIGMG_LEVEL_ELIM) {
      mul(L.R, b, WStore{bc.p});
      cycle(l + 1, bc.p, xc);
      x.alloc(n * ld);
      mul(L.P, xc.p, WInterp{L.q.p, b, x.p});
      return;
    }
    DevBuf<double> B[3], R(n * ld);
    for (auto &q : B) q.alloc(n * ld);
    int cur = 0;
    const int m = C.pre_smooth;
    if (C.jacobi || m <= 0) {
      fill_f64(B[0].p, 0.0, n * ld, s);
      if (C.jacobi) {
        step(L, b, B[0].p, nullptr, B[1].p, 0.0, 2.0 / 3.0);
        cur = 1;
      }
    } else {
      hipLaunchKernelGGL(k_wide_cheb0, grid(n), dim3(256), 0, s, L.dinv.p, b, B[1].p, C.be_pre[l][0], ld);
      LG_LAUNCH_CHECK();
      for (int k = 1; k < m; k++)
        step(L, b, B[k % 3].p, k == 1 ? nullptr : B[(k - 1) % 3].p, B[(k + 1) % 3].p, C.al_pre[l][k],
             C.be_pre[l][k]);
      cur = m % 3;
    }
    mul(L.A, B[cur].p, WResid{b, R.p});
    mul(L.M, R.p, WStore{bc.p});
    cycle(l + 1, bc.p, xc);
    hipLaunchKernelGGL(k_wide_prolong, grid(n), dim3(256), 0, s, L.agg.p, xc.p, B[cur].p, ld);
    LG_LAUNCH_CHECK();
    if (C.jacobi) {
      step(L, b, B[cur].p, nullptr, B[(cur + 1) % 3].p, 0.0, 2.0 / 3.0);
      cur = (cur + 1) % 3;
    } else {
      for (int k = 0; k < C.post_smooth; k++)
        step(L, b, B[(cur + k) % 3].p, k == 0 ? nullptr : B[(cur + k - 1) % 3].p, B[(cur + k + 1) % 3].p,
             C.al_post[l][k], C.be_post[l][k]);
      if (C.post_smooth > 0) cur = (cur + C.post_smooth) % 3;
    }
    if (C.scale != 1.0) {
      hipLaunchKernelGGL(k_wide_scale, grid(n), dim3(256), 0, s, B[cur].p, C.scale, ld);
      LG_LAUNCH_CHECK();
    }
    x = std::move(B[cur]);
  }
};

}  // namespace

void collapse_cycle(const std::vector<DLevel> &H, const CycleCoeffs &C, size_t l, DevBuf<double> &out,
                    hipStream_t s) {
  const int64_t n = H[l].A.n;
  Wide W{H, C, n, s};
  DevBuf<double> b(n * n);
  hipLaunchKernelGGL(k_wide_unit, W.grid(n), dim3(256), 0, s, b.p, n);
  LG_LAUNCH_CHECK();
  W.cycle(l, b.p, out);
}

}  // namespace lg
