// Block (multi right-hand side) kernels for batched solves.
//
// Block vectors are row-major n x kp (kp = number of right-hand sides
// rounded up to a power of two, at most 64): the kp values of a row are
// contiguous, so one gather of a column index fetches a whole row of X.  A
// group of kp lanes handles one matrix row, lane c handling right-hand
// side c.  Row sums accumulate in FP64.
#include <algorithm>
#include <type_traits>

#include "../../include/ligmg_amd.h"
#include "ops.hpp"
#include "prims.hpp"
#include "solve_dev.hpp"

namespace lg {

namespace {

template <class T>
struct BValOne {
  static constexpr bool one = true;
  __device__ __forceinline__ T operator()(int64_t) const { return (T)1; }
};
template <class T>
struct BValArr {
  static constexpr bool one = false;
  const T *v;
  __device__ __forceinline__ T operator()(int64_t k) const { return v[k]; }
};

// VW adjacent right-hand sides of one row: 16 bytes, or the whole row of a
// narrower block
template <class T, int VW>
struct BVec {
  typedef T type __attribute__((ext_vector_type(VW)));
};
template <class T>
struct BVec<T, 1> {
  typedef T type;
};
template <class T, int VW>
__device__ __forceinline__ double bvec_at(const typename BVec<T, VW>::type &x, int v) {
  if constexpr (VW == 1) return (double)x;
  else return (double)x[v];
}
template <class T, int VW>
__device__ __forceinline__ typename BVec<T, VW>::type bvec_load(const T *p) {
  return *(const typename BVec<T, VW>::type *)p;
}
template <class T, int VW, class F>
__device__ __forceinline__ void bvec_store(T *p, const F &f) {
  typename BVec<T, VW>::type y;
  if constexpr (VW == 1) {
    y = f(0);
  } else {
#pragma unroll
    for (int v = 0; v < VW; v++) y[v] = f(v);
  }
  *(typename BVec<T, VW>::type *)p = y;
}

// ----------------------------------------------------------------- epilogues
// load: a row's other operands, asked for before its sum is formed; store:
// the result of VW adjacent right-hand sides from their sums s.
template <class T>
struct BStore {
  T *y;
  int kp;
  template <int VW>
  struct Pre {};
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t, int) const {
    return {};
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &) const {
    bvec_store<T, VW>(y + i * kp + c, [&](int v) { return (T)s[v]; });
  }
};
// y = s and the next cycle's first Chebyshev step from y
template <class T>
struct BFirst {
  T *y;
  FirstStep<T> f;
  int kp;
  template <int VW>
  struct Pre {
    T dinv;
  };
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t i, int) const {
    return {f.dinv[i]};
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &p) const {
    const int64_t o = i * kp + c;
    bvec_store<T, VW>(y + o, [&](int v) { return (T)s[v]; });
    bvec_store<T, VW>(f.x + o, [&](int v) { return sdev::cheb_first<T>(f.beta, p.dinv, (T)s[v]); });
  }
};
template <class T>
struct BResid {
  const T *b;
  T *r;
  int kp;
  template <int VW>
  struct Pre {
    typename BVec<T, VW>::type b;
  };
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t i, int c) const {
    return {bvec_load<T, VW>(b + i * kp + c)};
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &p) const {
    bvec_store<T, VW>(r + i * kp + c, [&](int v) { return (T)(bvec_at<T, VW>(p.b, v) - s[v]); });
  }
};
template <class T>
struct BCheb {
  const T *dinv, *b, *xc, *xp;
  T *xn;
  double alpha, beta;
  int kp;
  template <int VW>
  struct Pre {
    typename BVec<T, VW>::type b, xc, xp;
    double dinv;
  };
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t i, int c) const {
    const int64_t o = i * kp + c;
    Pre<VW> p;
    p.b = bvec_load<T, VW>(b + o);
    p.xc = bvec_load<T, VW>(xc + o);
    if (xp) p.xp = bvec_load<T, VW>(xp + o);
    else p.xp = p.xc;
    p.dinv = (double)dinv[i];
    return p;
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &p) const {
    bvec_store<T, VW>(xn + i * kp + c, [&](int v) {
      const double cur = bvec_at<T, VW>(p.xc, v);
      // null xp: zero previous iterate
      const double d = alpha * (cur - (xp ? bvec_at<T, VW>(p.xp, v) : 0.0));
      return (T)(cur + d + beta * p.dinv * (bvec_at<T, VW>(p.b, v) - s[v]));
    });
  }
};
template <class T>
struct BInterp {
  const T *q, *b;
  T *x;
  int kp;
  template <int VW>
  struct Pre {
    typename BVec<T, VW>::type b;
    double q;
  };
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t i, int c) const {
    return {bvec_load<T, VW>(b + i * kp + c), (double)q[i]};
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &p) const {
    bvec_store<T, VW>(x + i * kp + c, [&](int v) { return (T)(s[v] + p.q * bvec_at<T, VW>(p.b, v)); });
  }
};
template <class T, class Epi>
struct BDiag {  // FP32 Laplacian form: + d[i] x[i, c]
  const double *d;
  const T *x;
  Epi e;
  int kp;
  template <int VW>
  struct Pre {
    typename BVec<T, VW>::type x;
    double d;
    typename Epi::template Pre<VW> e;
  };
  template <int VW>
  __device__ __forceinline__ Pre<VW> load(int64_t i, int c) const {
    return {bvec_load<T, VW>(x + i * kp + c), d[i], e.template load<VW>(i, c)};
  }
  template <int VW>
  __device__ __forceinline__ void store(int64_t i, int c, const double *s, const Pre<VW> &p) const {
    double t[VW];
#pragma unroll
    for (int v = 0; v < VW; v++) t[v] = s[v] + p.d * bvec_at<T, VW>(p.x, v);
    e.template store<VW>(i, c, t, p.e);
  }
};

// Y = A X by the SpMV's work units; workgroup (u, y) takes part y of the
// rows of unit u.  It stages the part's columns, values and row offsets in
// LDS with coalesced loads, so a row costs one round of gathers of X (U in
// flight, masked past the row's end) with its epilogue operands already
// asked for, instead of a chain of row pointer, column, gather and epilogue
// loads.  A row is summed by S groups of L = kp / VW lanes (S by the unit's
// mean row length: about 16 entries a group), group j adding entries j,
// j + S, ... in order, and the S partials meet in an xor butterfly inside
// one wavefront; S = 1 adds the row in stored order.  S does not depend on U
// or on the parts, so neither changes any bit.  Long-row chunks: every group
// of the workgroup takes a share, butterfly per wavefront, the wavefronts'
// sums added in order into kp partial sums.
// It is bound by gathers in flight.  One FP32 Chebyshev step, against a
// kernel that walked the row from global memory (one group a row, whatever
// its length): 100^3 grid (7 entries a row) x 32: 301 -> 175 us; 12
// Barabasi-Albert graphs (7.7 M entries, hubs) x 16: 252 -> 164 us; their
// 36-unit levels 80 -> 29 us.
template <class T, int VW, int U, class Val, class Epi>
__global__ void __launch_bounds__(256)
    k_spmm_units(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci, Val val,
                 const T *__restrict__ X, int kp, int lg, const int32_t *__restrict__ urow0,
                 const int32_t *__restrict__ unrows, const int32_t *__restrict__ ukoff,
                 double *__restrict__ parts, Epi epi) {
  typedef typename BVec<T, VW>::type V;
  constexpr bool ONE = Val::one;
  __shared__ int32_t scol[UNIT_NNZ];
  __shared__ T sval[ONE ? 1 : UNIT_NNZ];
  __shared__ int32_t soff[UNIT_ROWS + 1];
  __shared__ double red[256 / WAVE][64];
  const int u = blockIdx.x;
  const int row0 = urow0[u], nr = unrows[u], k0 = ukoff[u];
  const int L = 1 << lg, G = 256 >> lg;  // lanes of a group, groups
  const int gid = threadIdx.x >> lg, c0 = (threadIdx.x & (L - 1)) * VW;
  auto stage = [&](int ka, int cnt) {
    for (int t = threadIdx.x; t < cnt; t += 256) {
      scol[t] = ci[ka + t];
      if constexpr (!ONE) sval[t] = val(ka + t);
    }
  };
  // adds entries a, a + step, ... below b to s
  auto add = [&](double *s, int a, int b, int step) {
    for (int j = a; j < b; j += U * step) {
      V xx[U];
      double vv[U];
#pragma unroll
      for (int t = 0; t < U; t++) {
        const int e = j + t * step < b ? j + t * step : j;
        xx[t] = *(const V *)(X + (int64_t)scol[e] * kp + c0);
        if constexpr (ONE) vv[t] = 1.0;
        else vv[t] = (double)sval[e];
      }
#pragma unroll
      for (int t = 0; t < U; t++)
#pragma unroll
        for (int v = 0; v < VW; v++) s[v] += j + t * step < b ? vv[t] * bvec_at<T, VW>(xx[t], v) : 0.0;
    }
  };
  double s[VW];
  if (nr > 0) {
    const int per = (nr + gridDim.y - 1) / gridDim.y, ra = blockIdx.y * per, nl = min(per, nr - ra);
    if (nl <= 0) return;
    const int ka = rp[row0 + ra], cnt = rp[row0 + ra + nl] - ka;
    for (int t = threadIdx.x; t <= nl; t += 256) soff[t] = rp[row0 + ra + t] - ka;
    stage(ka, cnt);
    const int avg = (rp[row0 + nr] - k0 + nr - 1) / nr;
    int S = 1;
    while (S * L < WAVE && 16 * S < avg) S <<= 1;
    const int sub = gid & (S - 1), RG = G / S, rg = gid / S;
    __syncthreads();
    for (int r0 = 0; r0 < nl; r0 += RG) {  // same trip count for the whole workgroup
      const int r = r0 + rg;
      const bool ok = r < nl, mine = ok && sub == 0;
      const int64_t row = row0 + ra + r;
      typename Epi::template Pre<VW> pre;
      if (mine) pre = epi.template load<VW>(row, c0);
#pragma unroll
      for (int v = 0; v < VW; v++) s[v] = 0;
      if (ok) add(s, soff[r] + sub, soff[r + 1], S);
      for (int off = L * S >> 1; off >= L; off >>= 1)
#pragma unroll
        for (int v = 0; v < VW; v++) s[v] += __shfl_xor(s[v], off, WAVE);
      if (mine) epi.template store<VW>(row, c0, s, pre);
    }
  } else {
    if (blockIdx.y > 0) return;
    const int cnt = min(k0 + UNIT_NNZ, rp[row0 + 1]) - k0;
    stage(k0, cnt);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < VW; v++) s[v] = 0;
    add(s, gid, cnt, G);
    for (int off = WAVE >> 1; off >= L; off >>= 1)
#pragma unroll
      for (int v = 0; v < VW; v++) s[v] += __shfl_xor(s[v], off, WAVE);
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    if (lane < L)
#pragma unroll
      for (int v = 0; v < VW; v++) red[w][c0 + v] = s[v];
    __syncthreads();
    if ((int)threadIdx.x < kp) {
      double t = 0;
      for (int q = 0; q < 256 / WAVE; q++) t += red[q][threadIdx.x];
      parts[(int64_t)(-nr) * kp + threadIdx.x] = t;
    }
  }
}

template <class Epi>
__global__ void k_spmm_long(const int32_t *lrow, const int32_t *lpart, int64_t nlong, int kp,
                            const double *parts, Epi epi) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nlong * kp;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = t / kp;
    const int c = (int)(t % kp);
    double s = 0;
    for (int p = lpart[j]; p < lpart[j + 1]; p++) s += parts[(int64_t)p * kp + c];
    epi.template store<1>(lrow[j], c, &s, epi.template load<1>(lrow[j], c));
  }
}

int log2i(int k) {
  int l = 0;
  while ((1 << l) < k) l++;
  return l;
}

template <class T>
const T *bvals(const DCsr &A);
template <>
const double *bvals<double>(const DCsr &A) {
  return A.v.p;
}
template <>
const float *bvals<float>(const DCsr &A) {
  return A.v32.p;
}

// SpMM tiles: gathers in flight U by id.  A lane holds 16 bytes of a row of
// X (4 FP32 or 2 FP64 right-hand sides), or the whole row of a narrower block.
constexpr int SPMM_NCFG = 2;
constexpr int SPMM_U[SPMM_NCFG] = {4, 8};

template <class T>
constexpr int prec_slot() {
  return std::is_same<T, float>::value ? 1 : 0;
}
template <class T>
constexpr int spmm_vw(int kp) {
  return std::min<int>(16 / (int)sizeof(T), kp);
}
// the tile without timing: rows that one round of 4 gathers covers take 4
inline int spmm_rule(const DCsr &A) { return A.nnz <= 4 * A.n ? 0 : 1; }
// parts of a unit's rows: operators of few units spread over the CUs
inline unsigned spmm_parts(int64_t nunits) {
  unsigned y = 1;
  while (nunits * y < 1024 && y < 16) y <<= 1;
  return y;
}

template <class T, int VW, class Val, class Epi>
void launch_spmm_vw(int cfg, const DCsr &A, Val val, const T *X, int kp, Epi epi, double *parts, hipStream_t s) {
  const dim3 grid((unsigned)A.U.nunits, spmm_parts(A.U.nunits));
  const int lg = log2i(kp / VW);
  if (cfg == 0)
    hipLaunchKernelGGL((k_spmm_units<T, VW, 4, Val, Epi>), grid, dim3(256), 0, s, A.rp.p, A.ci.p, val, X, kp, lg,
                       A.U.row0.p, A.U.nrows.p, A.U.koff.p, parts, epi);
  else
    hipLaunchKernelGGL((k_spmm_units<T, VW, 8, Val, Epi>), grid, dim3(256), 0, s, A.rp.p, A.ci.p, val, X, kp, lg,
                       A.U.row0.p, A.U.nrows.p, A.U.koff.p, parts, epi);
  LG_LAUNCH_CHECK();
}

template <class T, class Val, class Epi>
void launch_spmm(const DCsr &A, Val val, const T *X, int kp, Epi epi, DevBuf<double> &parts,
                 hipStream_t s) {
  if (A.U.nunits == 0) return;
  LG_CHECK(parts.n >= (size_t)std::max<int64_t>(A.U.nparts, 1) * kp, LIGMG_ERR_INVALID,
           "spmm partial-sum buffer too small");
  int cfg = A.U.spmm_cfg[prec_slot<T>()][log2i(kp)];
  if (cfg < 0) cfg = spmm_rule(A);
  switch (spmm_vw<T>(kp)) {
    case 1: launch_spmm_vw<T, 1>(cfg, A, val, X, kp, epi, parts.p, s); break;
    case 2: launch_spmm_vw<T, 2>(cfg, A, val, X, kp, epi, parts.p, s); break;
    default:
      if constexpr (sizeof(T) == 4) launch_spmm_vw<T, 4>(cfg, A, val, X, kp, epi, parts.p, s);
  }
  if (A.U.nlong) {
    hipLaunchKernelGGL((k_spmm_long<Epi>), dim3(grid_for(A.U.nlong * kp, 256)), dim3(256), 0, s,
                       A.U.lrow.p, A.U.lpart.p, A.U.nlong, kp, (const double *)parts.p, epi);
    LG_LAUNCH_CHECK();
  }
}

template <class T, class Epi>
void dispatch_spmm(const DCsr &A, const T *X, int kp, Epi epi, DevBuf<double> &parts, hipStream_t s) {
  const T *v = bvals<T>(A);
  if (std::is_same<T, float>::value && A.d32.p)
    launch_spmm<T>(A, BValArr<T>{v}, X, kp, BDiag<T, Epi>{A.d32.p, X, epi, kp}, parts, s);
  else if (v) launch_spmm<T>(A, BValArr<T>{v}, X, kp, epi, parts, s);
  else launch_spmm<T>(A, BValOne<T>{}, X, kp, epi, parts, s);
}

// ------------------------------------------------------------- elementwise
template <class T>
__global__ void k_bcheb_zero(const T *dinv, const T *b, T *xn, double beta, int64_t n, int lk) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (n << lk);
       t += (int64_t)gridDim.x * blockDim.x)
    xn[t] = (T)(beta * (double)dinv[t >> lk] * (double)b[t]);
}

// x += xc[agg], 16 bytes a thread (or the whole row of a narrower block); lv =
// log2 of the threads per row
template <class T, int VW>
__global__ void __launch_bounds__(256) k_bprolong(const int32_t *__restrict__ agg, int64_t n, int lv, const T *__restrict__ xc,
                                                  T *__restrict__ x) {
  typedef typename BVec<T, VW>::type V;
  const V *c = (const V *)xc;
  V *y = (V *)x;
  for (int64_t t = blockIdx.x * (int64_t)256 + threadIdx.x; t < (n << lv); t += (int64_t)gridDim.x * 256)
    y[t] += c[((int64_t)agg[t >> lv] << lv) + (t & ((1 << lv) - 1))];
}

// Column-major caller block (ld n, vertex order given by perm, identity when
// null) <-> row-major internal block (padding columns zero).  A workgroup
// turns 64 rows in LDS, so both sides are read and written along their rows
// (one entry a thread left every access on a line of its own: 649 us for
// 10^6 x 32, 262 us now).
constexpr int TURN_ROWS = 64;
__global__ void __launch_bounds__(256) k_to_block(const double *__restrict__ B, int64_t n, int k, int kp, int lk,
                                                  const int32_t *__restrict__ perm, double *__restrict__ X) {
  __shared__ double tile[TURN_ROWS * 65];
  const int64_t i0 = (int64_t)blockIdx.x * TURN_ROWS;
  const int rows = (int)min((int64_t)TURN_ROWS, n - i0);
  const int r = threadIdx.x % TURN_ROWS;
  if (r < rows) {
    const int64_t src = perm ? perm[i0 + r] : i0 + r;
    for (int c = threadIdx.x / TURN_ROWS; c < kp; c += 256 / TURN_ROWS)
      tile[r * (kp + 1) + c] = c < k ? B[(int64_t)c * n + src] : 0.0;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < rows << lk; t += 256) X[(i0 << lk) + t] = tile[(t >> lk) * (kp + 1) + (t & (kp - 1))];
}
__global__ void __launch_bounds__(256) k_from_block(const double *__restrict__ X, int64_t n, int k, int kp, int lk,
                                                    const int32_t *__restrict__ perm, double *__restrict__ B) {
  __shared__ double tile[TURN_ROWS * 65];
  const int64_t i0 = (int64_t)blockIdx.x * TURN_ROWS;
  const int rows = (int)min((int64_t)TURN_ROWS, n - i0);
  for (int t = threadIdx.x; t < rows << lk; t += 256) tile[(t >> lk) * (kp + 1) + (t & (kp - 1))] = X[(i0 << lk) + t];
  __syncthreads();
  const int r = threadIdx.x % TURN_ROWS;
  if (r >= rows) return;
  const int64_t dst = perm ? perm[i0 + r] : i0 + r;
  for (int c = threadIdx.x / TURN_ROWS; c < k; c += 256 / TURN_ROWS) B[(int64_t)c * n + dst] = tile[r * (kp + 1) + c];
}

// ------------------------------------------------------- coarse dense apply
// Y (n x kp) = Pm (n x n, FP64, row-major) * X (n x kp) with FP64 MFMA
// 16x16x4 tiles.  Operand layout of v_mfma_f64_16x16x4f64 (measured on
// gfx950): lane l = 16 lk + li supplies A[li][lk] and B[lk][li] of the
// 16x4 / 4x16 slices and holds D[lk + 4v][li], v = 0..3.
//
// One workgroup per 16 rows of Y and all kp = 16 NT columns, so Pm is read
// once.  Its four wavefronts split the K range: lane (li, lk) of wavefront w
// takes K = (4 w + lk) Q + q, q = 0 .. Q-1 (Q = ceil(n / 16)), one contiguous
// run of its row of Pm; two accumulator sets alternate on q so consecutive
// products into one tile do not wait on each other.  The four partial tiles
// are added in LDS in wavefront order.
template <class T, int NT>
__global__ void __launch_bounds__(256) k_dense_mfma(const double *__restrict__ Pm, int n,
                                                    const T *__restrict__ X, int kp, int Q,
                                                    T *__restrict__ Y) {
  typedef double v4d __attribute__((ext_vector_type(4)));
  __shared__ double part[4][16 * 16 * NT];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int li = lane & 15, lk = lane >> 4;
  const int i0 = blockIdx.x * 16, row = i0 + li;
  const double *prow = Pm + (int64_t)(row < n ? row : n - 1) * n;
  const int kb = (4 * w + lk) * Q;
  v4d acc[2][NT];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int tj = 0; tj < NT; tj++) acc[h][tj] = v4d{0, 0, 0, 0};
  // K slots go in blocks of QB (16 products), each block's operands loaded
  // one block ahead
  constexpr int QB = 16 / NT;
  auto load_blk = [&](int q0, double *aa, double (*bb)[NT]) {
#pragma unroll
    for (int u = 0; u < QB; u++) {
      const int kk = kb + q0 + u;
      const bool ok = q0 + u < Q && kk < n;
      aa[u] = (ok && row < n) ? prow[kk] : 0.0;
#pragma unroll
      for (int tj = 0; tj < NT; tj++) bb[u][tj] = ok ? (double)X[(int64_t)kk * kp + 16 * tj + li] : 0.0;
    }
  };
  double a[QB], b[QB][NT];
  load_blk(0, a, b);
  for (int q0 = 0; q0 < Q; q0 += QB) {
    double an[QB], bn[QB][NT];
    if (q0 + QB < Q) load_blk(q0 + QB, an, bn);
#pragma unroll
    for (int u = 0; u < QB; u++)
#pragma unroll
      for (int tj = 0; tj < NT; tj++)
        acc[u & 1][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u][tj], acc[u & 1][tj], 0, 0, 0);
#pragma unroll
    for (int u = 0; u < QB; u++) {
      a[u] = an[u];
#pragma unroll
      for (int tj = 0; tj < NT; tj++) b[u][tj] = bn[u][tj];
    }
  }
#pragma unroll
  for (int tj = 0; tj < NT; tj++)
#pragma unroll
    for (int v = 0; v < 4; v++) part[w][(lk + 4 * v) * 16 * NT + 16 * tj + li] = acc[0][tj][v] + acc[1][tj][v];
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * 16 * NT; e += blockDim.x) {
    const int r = e / (16 * NT), c = e % (16 * NT);
    if (i0 + r < n) Y[(int64_t)(i0 + r) * kp + c] = (T)(((part[0][e] + part[1][e]) + part[2][e]) + part[3][e]);
  }
}

// kp < 16: one wavefront per row of the matrix, KP sums per lane.  (One
// thread per output walked the row alone: 24 us for 157 x 157 x 4, 3.8 us now.)
template <class T, int KP>
__global__ void __launch_bounds__(256) k_dense_small(const double *__restrict__ Pm, int64_t n,
                                                     const T *__restrict__ X, T *__restrict__ Y) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / WAVE;
  if (i >= n) return;  // the whole wavefront
  double s[KP] = {};
#pragma unroll 4
  for (int64_t j = lane; j < n; j += WAVE) {
    const double a = Pm[i * n + j];
#pragma unroll
    for (int c = 0; c < KP; c++) s[c] += a * (double)X[j * KP + c];
  }
#pragma unroll
  for (int c = 0; c < KP; c++) {
    s[c] = sdev::wave_sum(s[c]);
    if (lane == 0) Y[i * KP + c] = (T)s[c];
  }
}

// -------------------------------------------------- per-(block, column) dots
// The vector passes below take a segment of rows per workgroup
// (RedPlan::build with block_seg_rows(kp) rows) and VW = 2 adjacent columns
// per thread (1 when kp = 1), four rows in flight.  With 4096-row segments and
// 8-byte accesses a 10^6 x 32 block had 245 workgroups, less than one per CU:
// the update took 852 us for 1.73 GB (2.0 TB/s), now 305 us (5.7 TB/s, part
// of it from the Infinity Cache).

// this workgroup's rows [lo, hi); the thread takes rows lo + g, lo + g + G,
// ... and columns c .. c + VW - 1
template <int VW>
struct BSeg {
  int64_t lo, hi;
  int G, g, c;
  __device__ __forceinline__ BSeg(int64_t l, int64_t h, int kp) : lo(l), hi(h) {
    const int L = kp / VW;  // a power of two
    G = 256 / L;
    g = threadIdx.x / L;
    c = (threadIdx.x & (L - 1)) * VW;
  }
};

// sums of the workgroup's per-thread partials: part[c + v], columns combined
// over the row groups in order
template <int VW>
__device__ __forceinline__ void bseg_sum(const BSeg<VW> &B, int kp, const double *acc, double (*red)[256],
                                         double *part) {
#pragma unroll
  for (int v = 0; v < VW; v++) red[v][threadIdx.x] = acc[v];
  __syncthreads();
  if (B.g == 0) {
    const int L = kp / VW;
#pragma unroll
    for (int v = 0; v < VW; v++) {
      double t = 0;
      for (int gg = 0; gg < B.G; gg++) t += red[v][gg * L + threadIdx.x];
      part[B.c + v] = t;
    }
  }
  __syncthreads();
}

// part[(s * np + j) * kp + c] for segment s; out[(blk * np + j) * kp + c]
template <class T, int VW>
__global__ void __launch_bounds__(256) k_bred1(int np, int kp, const T *a0, const T *b0, const T *a1, const T *b1,
                                               const int64_t *lo, const int64_t *hi, double *part) {
  const int s = blockIdx.x;
  const BSeg<VW> B(lo[s], hi[s], kp);
  double acc0[VW] = {}, acc1[VW] = {};
  for (int64_t i = B.lo + B.g; i < B.hi; i += 4 * B.G) {
    typename BVec<T, VW>::type x0[4], y0[4], x1[4], y1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int64_t o = min(i + t * B.G, B.hi - 1) * kp + B.c;
      x0[t] = bvec_load<T, VW>(a0 + o);
      if (b0) y0[t] = bvec_load<T, VW>(b0 + o);
      if (np > 1) {
        x1[t] = a1 == a0 ? x0[t] : bvec_load<T, VW>(a1 + o);
        if (b1) y1[t] = bvec_load<T, VW>(b1 + o);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
      if (i + t * B.G < B.hi)
#pragma unroll
        for (int v = 0; v < VW; v++) {
          acc0[v] += bvec_at<T, VW>(x0[t], v) * (b0 ? bvec_at<T, VW>(y0[t], v) : 1.0);
          if (np > 1) acc1[v] += bvec_at<T, VW>(x1[t], v) * (b1 ? bvec_at<T, VW>(y1[t], v) : 1.0);
        }
  }
  __shared__ double red[VW][256];
  bseg_sum<VW>(B, kp, acc0, red, part + (int64_t)s * np * kp);
  if (np > 1) bseg_sum<VW>(B, kp, acc1, red, part + ((int64_t)s * np + 1) * kp);
}

// what follows the sums of set (blk, c)
__device__ __forceinline__ void block_post(const BlockPost &P, int blk, int c, int np, int kp, const double *sum) {
  if (P.kind == BlockPost::OUT) {
    for (int j = 0; j < np; j++) P.out[((int64_t)blk * np + j) * kp + c] = sum[j];
    return;
  }
  using namespace sdev;
  const int64_t set = (int64_t)blk * kp + c;
  double *S = P.sc + set * SC_N;
  switch (P.kind) {
    case BlockPost::ALPHA:
      S[SC_DELTA] = sum[0];
      if (P.fcg) S[SC_T1] = sum[1];
      kr_alpha(S, P.fcg);
      break;
    case BlockPost::BETA:
      S[P.fcg ? SC_T1 : SC_GN] = sum[0];
      kr_beta(S, P.fcg);
      break;
    default: {  // INIT, NORM
      const bool init = P.kind == BlockPost::INIT;
      if (init) {
        kr_init(S);
        S[SC_BN2] = sum[0];
      } else if (S[SC_ACTIVE] != 0) {
        S[SC_ITS] += 1;
      }
      S[SC_RN2] = sum[0];
      kr_check(S, P.rtol);
      if (P.to.host) kr_publish(P.to, set, init, sum[0], S[SC_ACTIVE]);
    }
  }
}

// The segment partials of block blk, summed per column, and what follows
// (BlockPost): one workgroup per block and cw = min(kp, 8) columns.  Thread (g,
// c) adds segments g, g + G, ... (G = 1024 / cw) in order, and the G partials of
// a column are added 16 at a time.  (All 32 columns of 2045 segments in one
// workgroup took 21 us, bound by that CU's reads.)  The scalar steps of the
// (blk, column) sets run here, so a dot costs no launch beyond its two stages.
constexpr int BRED_COLS = 8;
__global__ void __launch_bounds__(1024) k_bred2(int np, int kp, int lw, const int32_t *bseg, const double *part,
                                                BlockPost P) {
  const int blk = blockIdx.x;
  const int cw = 1 << lw, G = 1024 >> lw;
  const int g = threadIdx.x >> lw, cl = threadIdx.x & (cw - 1), c = blockIdx.y * cw + cl;
  const int end = bseg[blk + 1];
  __shared__ double red[1024];
  double sum[2] = {0, 0};
  for (int j = 0; j < np; j++) {
    double acc = 0;
#pragma unroll 8
    for (int sg = bseg[blk] + g; sg < end; sg += G) acc += part[((int64_t)sg * np + j) * kp + c];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int n = G; n > 1; n = (n + 15) / 16) {
      const int m = (n + 15) / 16;
      double t = 0;
      if (g < m)
        for (int q = 16 * g; q < min(16 * g + 16, n); q++) t += red[q * cw + cl];
      __syncthreads();
      if (g < m) red[threadIdx.x] = t;
      __syncthreads();
    }
    sum[j] = red[cl];
    __syncthreads();
  }
  if (g == 0) block_post(P, blk, c, np, kp, sum);
}

// The same for plans of at most BRED_FEW segments a block, a thread per set:
// its partials in order, the sums k_bred2 forms there.  A workgroup per small
// block was mostly idle threads and barriers (3000 blocks of one segment x 64
// columns: 117 to 225 us a call, now 4 to 9; one block of 12 segments x 32 columns
// 5.1 us, now 4.6).
constexpr int BRED_FEW = 16;
template <int NP>
__global__ void __launch_bounds__(256) k_bred2_few(int kp, int lk, int64_t sets, const int32_t *bseg,
                                                   const double *part, BlockPost P) {
  const int64_t set = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (set >= sets) return;
  const int blk = (int)(set >> lk), c = (int)(set & (kp - 1));
  const int a = bseg[blk], b = bseg[blk + 1];
  double sum[NP] = {};
  for (int sg = a; sg < b; sg += 8) {
    double v[8][NP];
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
      for (int j = 0; j < NP; j++) v[t][j] = part[((int64_t)min(sg + t, b - 1) * NP + j) * kp + c];
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
      for (int j = 0; j < NP; j++) sum[j] += sg + t < b ? v[t][j] : 0.0;
  }
  block_post(P, blk, c, NP, kp, sum);
}

template <class T, int VW>
__global__ void __launch_bounds__(256) k_bsub_mean(T *a, int kp, const int64_t *lo, const int64_t *hi,
                                                   const int32_t *segblk, const int64_t *bptr, const double *sums) {
  const int s = blockIdx.x;
  const int blk = segblk[s];
  const BSeg<VW> B(lo[s], hi[s], kp);
  T m[VW];
#pragma unroll
  for (int v = 0; v < VW; v++) m[v] = (T)(sums[(int64_t)blk * kp + B.c + v] / (double)(bptr[blk + 1] - bptr[blk]));
#pragma unroll 4
  for (int64_t i = B.lo + B.g; i < B.hi; i += B.G) {
    const typename BVec<T, VW>::type x = bvec_load<T, VW>(a + i * kp + B.c);
    bvec_store<T, VW>(a + i * kp + B.c, [&](int v) {
      if constexpr (VW == 1) return x - m[0];
      else return x[v] - m[v];
    });
  }
}

// z = c - (block mean) and the segment partials of z.w as the block dots
// form them (part[s * kp + c])
template <class T, class C, int VW>
__global__ void __launch_bounds__(256) k_bcenter(T *z, const C *cv, const T *w, int kp, const int64_t *lo,
                                                 const int64_t *hi, const int32_t *segblk, const int64_t *bptr,
                                                 const double *sums, double *part) {
  const int s = blockIdx.x;
  const int blk = segblk[s];
  const BSeg<VW> B(lo[s], hi[s], kp);
  T m[VW];
  double acc[VW] = {};
#pragma unroll
  for (int v = 0; v < VW; v++) m[v] = (T)(sums[(int64_t)blk * kp + B.c + v] / (double)(bptr[blk + 1] - bptr[blk]));
  for (int64_t i = B.lo + B.g; i < B.hi; i += 4 * B.G) {
    typename BVec<C, VW>::type x[4];
    typename BVec<T, VW>::type y[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int64_t o = min(i + t * B.G, B.hi - 1) * kp + B.c;
      x[t] = bvec_load<C, VW>(cv + o);
      y[t] = bvec_load<T, VW>(w + o);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (i + t * B.G >= B.hi) continue;
      T zv[VW];
#pragma unroll
      for (int v = 0; v < VW; v++) {
        zv[v] = (T)bvec_at<C, VW>(x[t], v) - m[v];
        acc[v] += (double)zv[v] * bvec_at<T, VW>(y[t], v);
      }
      bvec_store<T, VW>(z + (i + t * B.G) * kp + B.c, [&](int v) { return zv[v]; });
    }
  }
  __shared__ double red[VW][256];
  bseg_sum<VW>(B, kp, acc, red, part + (int64_t)s * kp);
}

// x = 0, r = b and the segment partials of b.b; rf and f as in k_kr_bupdate
template <class T, class F, int VW>
__global__ void __launch_bounds__(256) k_kr_bbegin(const T *b, T *x, T *r, F *rf, FirstStep<F> f, int kp,
                                                   const int64_t *lo, const int64_t *hi, double *part) {
  const int s = blockIdx.x;
  const BSeg<VW> B(lo[s], hi[s], kp);
  double acc[VW] = {};
#pragma unroll 4
  for (int64_t i = B.lo + B.g; i < B.hi; i += B.G) {
    const int64_t o = i * kp + B.c;
    const typename BVec<T, VW>::type v = bvec_load<T, VW>(b + o);
    bvec_store<T, VW>(x + o, [&](int) { return (T)0; });
    *(typename BVec<T, VW>::type *)(r + o) = v;
    if (rf) bvec_store<F, VW>(rf + o, [&](int u) { return (F)bvec_at<T, VW>(v, u); });
    if (f.x) {
      const F dv = f.dinv[i];
      bvec_store<F, VW>(f.x + o, [&](int u) { return sdev::cheb_first<F>(f.beta, dv, (F)bvec_at<T, VW>(v, u)); });
    }
#pragma unroll
    for (int u = 0; u < VW; u++) acc[u] += bvec_at<T, VW>(v, u) * bvec_at<T, VW>(v, u);
  }
  __shared__ double red[VW][256];
  bseg_sum<VW>(B, kp, acc, red, part + (int64_t)s * kp);
}

// x += alpha p, r -= alpha q per (block, column); alpha = 0 marks a finished
// column, whose x and r stay.  Also writes the segment partials of r.r as
// the block dots form them (part[s * kp + c]); with rf set r in the cycle's
// type, with f.x set the cycle's first step from r.
template <class T, class F, int VW>
__global__ void __launch_bounds__(256) k_kr_bupdate(T *x, T *r, const T *p, const T *q, F *rf, FirstStep<F> f,
                                                    int kp, const int64_t *lo, const int64_t *hi,
                                                    const int32_t *segblk, const double *sc, double *part) {
  const int s = blockIdx.x;
  const BSeg<VW> B(lo[s], hi[s], kp);
  T at[VW];
  bool any = false;
  double acc[VW] = {};
#pragma unroll
  for (int v = 0; v < VW; v++) {
    const double a = sc[((int64_t)segblk[s] * kp + B.c + v) * sdev::SC_N + sdev::SC_ALPHA];
    at[v] = (T)a;
    any |= a != 0.0;
  }
  typedef typename BVec<T, VW>::type V;
  for (int64_t i = B.lo + B.g; i < B.hi; i += 4 * B.G) {
    V xv[4], rv[4], pv[4], qv[4];
    F dv[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int64_t row = min(i + t * B.G, B.hi - 1), o = row * kp + B.c;
      rv[t] = bvec_load<T, VW>(r + o);
      if (f.x) dv[t] = f.dinv[row];
      if (any) {
        xv[t] = bvec_load<T, VW>(x + o);
        pv[t] = bvec_load<T, VW>(p + o);
        qv[t] = bvec_load<T, VW>(q + o);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (i + t * B.G >= B.hi) continue;
      const int64_t o = (i + t * B.G) * kp + B.c;
      T xn[VW], rn[VW];
#pragma unroll
      for (int v = 0; v < VW; v++) {
        if constexpr (VW == 1) {
          rn[v] = any ? rv[t] - at[v] * qv[t] : rv[t];
          if (any) xn[v] = xv[t] + at[v] * pv[t];
        } else {
          // a finished column of a pair keeps its bits (alpha p may not be 0)
          const bool on = any && at[v] != (T)0;
          rn[v] = on ? rv[t][v] - at[v] * qv[t][v] : rv[t][v];
          if (any) xn[v] = on ? xv[t][v] + at[v] * pv[t][v] : xv[t][v];
        }
        acc[v] += (double)rn[v] * (double)rn[v];
      }
      if (any) {
        bvec_store<T, VW>(x + o, [&](int v) { return xn[v]; });
        bvec_store<T, VW>(r + o, [&](int v) { return rn[v]; });
      }
      if (rf) bvec_store<F, VW>(rf + o, [&](int v) { return (F)rn[v]; });
      if (f.x) bvec_store<F, VW>(f.x + o, [&](int v) { return sdev::cheb_first<F>(f.beta, dv[t], (F)rn[v]); });
    }
  }
  __shared__ double red[VW][256];
  bseg_sum<VW>(B, kp, acc, red, part + (int64_t)s * kp);
}

// p = z + beta p; where beta is 0 (the first step) p is not used
template <class T, int VW>
__global__ void __launch_bounds__(256) k_kr_bpupdate(T *p, const T *z, int kp, const int64_t *lo, const int64_t *hi,
                                                     const int32_t *segblk, const double *sc) {
  const int s = blockIdx.x;
  const BSeg<VW> B(lo[s], hi[s], kp);
  T bt[VW];
#pragma unroll
  for (int v = 0; v < VW; v++)
    bt[v] = (T)sc[((int64_t)segblk[s] * kp + B.c + v) * sdev::SC_N + sdev::SC_BETA];
  typedef typename BVec<T, VW>::type V;
  for (int64_t i = B.lo + B.g; i < B.hi; i += 4 * B.G) {
    V pv[4], zv[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int64_t o = min(i + t * B.G, B.hi - 1) * kp + B.c;
      pv[t] = bvec_load<T, VW>(p + o);
      zv[t] = bvec_load<T, VW>(z + o);
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
      if (i + t * B.G < B.hi)
        bvec_store<T, VW>(p + (i + t * B.G) * kp + B.c, [&](int v) {
          if constexpr (VW == 1) return bt[0] != (T)0 ? zv[t] + bt[0] * pv[t] : zv[t];
          else return bt[v] != (T)0 ? zv[t][v] + bt[v] * pv[t][v] : zv[t][v];
        });
  }
}

}  // namespace

// ---------------------------------------------------------------- host side
// Operators of less work than this take the rule's tile: timing it costs
// more than a wrong pick over a solve.
constexpr int64_t SPMM_TUNE_MIN = (int64_t)32 << 20;

// Times every tile on A (the operator's own values and
// Laplacian-form diagonal, X of zeros, a plain store) and records the
// fastest for this precision and width; a tile already picked is kept.
template <class T>
int tune_spmm(DCsr &A, int kp, DevBuf<double> &parts, hipStream_t s) {
  int8_t &pick = A.U.spmm_cfg[prec_slot<T>()][log2i(kp)];
  if (pick < 0 && A.nnz * kp < SPMM_TUNE_MIN) pick = (int8_t)spmm_rule(A);
  if (pick >= 0 || A.U.nunits == 0) return pick < 0 ? 0 : pick;
  DevBuf<T> X((size_t)std::max<int64_t>(A.ncols, 1) * kp), Y((size_t)std::max<int64_t>(A.n, 1) * kp);
  fill_u8((uint8_t *)X.p, 0, (int64_t)X.bytes(), s);
  hipEvent_t e0, e1;
  LG_HIP(hipEventCreate(&e0));
  LG_HIP(hipEventCreate(&e1));
  float best = 0;
  int besti = 0;
  for (int c = 0; c < SPMM_NCFG; c++) {
    A.U.spmm_cfg[prec_slot<T>()][log2i(kp)] = (int8_t)c;
    op_bspmv<T>(A, X.p, Y.p, kp, parts, s);  // warm
    LG_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < 3; r++) op_bspmv<T>(A, X.p, Y.p, kp, parts, s);
    LG_HIP(hipEventRecord(e1, s));
    LG_HIP(hipEventSynchronize(e1));
    float ms = 0;
    LG_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (c == 0 || ms < best) {
      best = ms;
      besti = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  pick = (int8_t)besti;
  return besti;
}

void spmm_tile(int cfg, int *u) { *u = SPMM_U[cfg]; }

template <class T>
void op_bspmv(const DCsr &A, const T *X, T *Y, int kp, DevBuf<double> &parts, hipStream_t s) {
  dispatch_spmm<T>(A, X, kp, BStore<T>{Y, kp}, parts, s);
}
template <class T>
void op_bspmv_first(const DCsr &A, const T *X, T *Y, const FirstStep<T> &f, int kp, DevBuf<double> &parts,
                    hipStream_t s) {
  if (f.x) dispatch_spmm<T>(A, X, kp, BFirst<T>{Y, f, kp}, parts, s);
  else op_bspmv<T>(A, X, Y, kp, parts, s);
}
template <class T>
void op_bresidual(const DCsr &A, const T *X, const T *B, T *R, int kp, DevBuf<double> &parts,
                  hipStream_t s) {
  dispatch_spmm<T>(A, X, kp, BResid<T>{B, R, kp}, parts, s);
}
template <class T>
void op_bcheb_step(const DCsr &A, const T *dinv, const T *B, const T *Xc, const T *Xp, T *Xn,
                   double alpha, double beta, int kp, DevBuf<double> &parts, hipStream_t s) {
  if (!Xc) {
    hipLaunchKernelGGL(k_bcheb_zero<T>, dim3(grid_for(A.n * kp, 256, 16384)), dim3(256), 0, s, dinv, B,
                       Xn, beta, A.n, log2i(kp));
    LG_LAUNCH_CHECK();
    return;
  }
  dispatch_spmm<T>(A, Xc, kp, BCheb<T>{dinv, B, Xc, Xp, Xn, alpha, beta, kp}, parts, s);
}
template <class T>
void op_binterp(const DCsr &P, const T *q, const T *Xc, const T *B, T *X, int kp,
                DevBuf<double> &parts, hipStream_t s) {
  dispatch_spmm<T>(P, Xc, kp, BInterp<T>{q, B, X, kp}, parts, s);
}
template <class T>
void op_bprolong_add(const int32_t *agg, int64_t n, const T *Xc, T *X, int kp, hipStream_t s) {
  const int vw = spmm_vw<T>(kp), lv = log2i(kp / vw);
  const dim3 g(grid_for(n << lv, 256, 16384));
  switch (vw) {
    case 1: hipLaunchKernelGGL((k_bprolong<T, 1>), g, dim3(256), 0, s, agg, n, lv, Xc, X); break;
    case 2: hipLaunchKernelGGL((k_bprolong<T, 2>), g, dim3(256), 0, s, agg, n, lv, Xc, X); break;
    default: hipLaunchKernelGGL((k_bprolong<T, 4>), g, dim3(256), 0, s, agg, n, lv, Xc, X);
  }
  LG_LAUNCH_CHECK();
}
template <class T>
void op_bdense_apply(const double *Pm, int64_t n, const T *X, T *Y, int kp, hipStream_t s) {
  if (n == 0) return;  // an elimination took every vertex: a grid of 0 is a launch error
  if (kp >= 16) {
    LG_CHECK(kp == 16 || kp == 32 || kp == 64, LIGMG_ERR_INVALID, "dense apply: kp must be 16, 32 or 64");
    const unsigned g = (unsigned)((n + 15) / 16);
    const int Q = (int)((n + 15) / 16);
    if (kp == 16) hipLaunchKernelGGL((k_dense_mfma<T, 1>), dim3(g), dim3(256), 0, s, Pm, (int)n, X, kp, Q, Y);
    else if (kp == 32) hipLaunchKernelGGL((k_dense_mfma<T, 2>), dim3(g), dim3(256), 0, s, Pm, (int)n, X, kp, Q, Y);
    else hipLaunchKernelGGL((k_dense_mfma<T, 4>), dim3(g), dim3(256), 0, s, Pm, (int)n, X, kp, Q, Y);
  } else {
    const dim3 g((unsigned)((n + 3) / 4));
    switch (kp) {
      case 1: hipLaunchKernelGGL((k_dense_small<T, 1>), g, dim3(256), 0, s, Pm, n, X, Y); break;
      case 2: hipLaunchKernelGGL((k_dense_small<T, 2>), g, dim3(256), 0, s, Pm, n, X, Y); break;
      case 4: hipLaunchKernelGGL((k_dense_small<T, 4>), g, dim3(256), 0, s, Pm, n, X, Y); break;
      default:
        LG_CHECK(kp == 8, LIGMG_ERR_INVALID, "dense apply: kp must be a power of two");
        hipLaunchKernelGGL((k_dense_small<T, 8>), g, dim3(256), 0, s, Pm, n, X, Y);
    }
  }
  LG_LAUNCH_CHECK();
}

void op_to_block(const double *B, int64_t n, int k, int kp, double *X, const int32_t *perm, hipStream_t s) {
  hipLaunchKernelGGL(k_to_block, dim3((unsigned)((n + TURN_ROWS - 1) / TURN_ROWS)), dim3(256), 0, s, B, n, k, kp,
                     log2i(kp), perm, X);
  LG_LAUNCH_CHECK();
}
void op_from_block(const double *X, int64_t n, int k, int kp, double *B, const int32_t *perm,
                   hipStream_t s) {
  hipLaunchKernelGGL(k_from_block, dim3((unsigned)((n + TURN_ROWS - 1) / TURN_ROWS)), dim3(256), 0, s, X, n, k, kp,
                     log2i(kp), perm, B);
  LG_LAUNCH_CHECK();
}

template <class T>
void RedPlan::bpartials(int np, int kp, const T *a0, const T *b0, const T *a1, const T *b1, DevBuf<double> &bpart,
                        hipStream_t s) const {
  if (nseg == 0) return;
  LG_CHECK(bpart.n >= (size_t)nseg * np * kp, LIGMG_ERR_INVALID, "block reduction buffer too small");
  if (kp == 1)
    hipLaunchKernelGGL((k_bred1<T, 1>), dim3(nseg), dim3(256), 0, s, np, kp, a0, b0, a1, b1, seg_lo.p, seg_hi.p,
                       bpart.p);
  else
    hipLaunchKernelGGL((k_bred1<T, 2>), dim3(nseg), dim3(256), 0, s, np, kp, a0, b0, a1, b1, seg_lo.p, seg_hi.p,
                       bpart.p);
  LG_LAUNCH_CHECK();
}

template <class T>
void RedPlan::bdots(int np, int kp, const T *a0, const T *b0, const T *a1, const T *b1, double *out,
                    DevBuf<double> &bpart, hipStream_t s) const {
  if (nseg == 0) return;
  bpartials<T>(np, kp, a0, b0, a1, b1, bpart, s);
  BlockPost P;
  P.out = out;
  bfinish(np, kp, P, bpart, s);
}

void RedPlan::bfinish(int np, int kp, const BlockPost &P, const DevBuf<double> &bpart, hipStream_t s) const {
  if (nb == 0) return;
  LG_CHECK(bpart.n >= (size_t)nseg * np * kp, LIGMG_ERR_INVALID, "block reduction buffer too small");
  const int64_t sets = (int64_t)nb * kp;
  BlockPost Q = P;
  Q.to = P.to.each(sets);
  if (most <= BRED_FEW) {
    const dim3 g((unsigned)((sets + 255) / 256));
    const double *bp = bpart.p;
    if (np == 1) hipLaunchKernelGGL(k_bred2_few<1>, g, dim3(256), 0, s, kp, log2i(kp), sets, bseg.p, bp, Q);
    else hipLaunchKernelGGL(k_bred2_few<2>, g, dim3(256), 0, s, kp, log2i(kp), sets, bseg.p, bp, Q);
  } else {
    const int cw = std::min(kp, BRED_COLS);
    hipLaunchKernelGGL(k_bred2, dim3((unsigned)nb, (unsigned)(kp / cw)), dim3(1024), 0, s, np, kp, log2i(cw), bseg.p,
                       (const double *)bpart.p, Q);
  }
  LG_LAUNCH_CHECK();
  if (P.to.host && !Q.to.host) kr_total(P.sc, sets, P.kind == BlockPost::INIT, P.to, s);
}

#define LG_SEGS dim3((unsigned)R.nseg), dim3(256), 0, s
template <class T, class C>
void op_bcenter(const RedPlan &R, T *z, const C *c, const T *w, int kp, const double *sums, DevBuf<double> &bpart,
                hipStream_t s) {
  if (R.nseg == 0) return;
  LG_CHECK(bpart.n >= (size_t)R.nseg * kp, LIGMG_ERR_INVALID, "block reduction buffer too small");
  if (kp == 1)
    hipLaunchKernelGGL((k_bcenter<T, C, 1>), LG_SEGS, z, c, w, kp, R.seg_lo.p, R.seg_hi.p, R.bseg.p + R.nb + 1,
                       R.bptr.p, sums, bpart.p);
  else
    hipLaunchKernelGGL((k_bcenter<T, C, 2>), LG_SEGS, z, c, w, kp, R.seg_lo.p, R.seg_hi.p, R.bseg.p + R.nb + 1,
                       R.bptr.p, sums, bpart.p);
  LG_LAUNCH_CHECK();
}
template <class T, class F>
void op_kr_bbegin(const RedPlan &R, const T *b, T *x, T *r, F *rf, const FirstStep<F> &f, int kp,
                  DevBuf<double> &bpart, hipStream_t s) {
  if (R.nseg == 0) return;
  LG_CHECK(bpart.n >= (size_t)R.nseg * kp, LIGMG_ERR_INVALID, "block reduction buffer too small");
  if (kp == 1)
    hipLaunchKernelGGL((k_kr_bbegin<T, F, 1>), LG_SEGS, b, x, r, rf, f, kp, R.seg_lo.p, R.seg_hi.p, bpart.p);
  else
    hipLaunchKernelGGL((k_kr_bbegin<T, F, 2>), LG_SEGS, b, x, r, rf, f, kp, R.seg_lo.p, R.seg_hi.p, bpart.p);
  LG_LAUNCH_CHECK();
}
#undef LG_SEGS

template <class T>
void op_bsub_block_mean(T *a, int kp, const RedPlan &P, const double *sums, hipStream_t s) {
  if (P.nseg == 0) return;
  if (kp == 1)
    hipLaunchKernelGGL((k_bsub_mean<T, 1>), dim3(P.nseg), dim3(256), 0, s, a, kp, P.seg_lo.p, P.seg_hi.p,
                       P.bseg.p + P.nb + 1, P.bptr.p, sums);
  else
    hipLaunchKernelGGL((k_bsub_mean<T, 2>), dim3(P.nseg), dim3(256), 0, s, a, kp, P.seg_lo.p, P.seg_hi.p,
                       P.bseg.p + P.nb + 1, P.bptr.p, sums);
  LG_LAUNCH_CHECK();
}

template <class T, class F>
void op_kr_bupdate(const RedPlan &R, T *x, T *r, const T *p, const T *q, F *rf, const FirstStep<F> &f, int kp,
                   const double *sc, DevBuf<double> &bpart, hipStream_t s) {
  if (R.nseg == 0) return;
  LG_CHECK(bpart.n >= (size_t)R.nseg * kp, LIGMG_ERR_INVALID, "block reduction buffer too small");
  if (kp == 1)
    hipLaunchKernelGGL((k_kr_bupdate<T, F, 1>), dim3(R.nseg), dim3(256), 0, s, x, r, p, q, rf, f, kp, R.seg_lo.p,
                       R.seg_hi.p, R.bseg.p + R.nb + 1, sc, bpart.p);
  else
    hipLaunchKernelGGL((k_kr_bupdate<T, F, 2>), dim3(R.nseg), dim3(256), 0, s, x, r, p, q, rf, f, kp, R.seg_lo.p,
                       R.seg_hi.p, R.bseg.p + R.nb + 1, sc, bpart.p);
  LG_LAUNCH_CHECK();
}

template <class T>
void op_kr_bpupdate(T *p, const T *z, int kp, const RedPlan &P, const double *sc, hipStream_t s) {
  if (P.nseg == 0) return;
  if (kp == 1)
    hipLaunchKernelGGL((k_kr_bpupdate<T, 1>), dim3(P.nseg), dim3(256), 0, s, p, z, kp, P.seg_lo.p, P.seg_hi.p,
                       P.bseg.p + P.nb + 1, sc);
  else
    hipLaunchKernelGGL((k_kr_bpupdate<T, 2>), dim3(P.nseg), dim3(256), 0, s, p, z, kp, P.seg_lo.p, P.seg_hi.p,
                       P.bseg.p + P.nb + 1, sc);
  LG_LAUNCH_CHECK();
}

#define LG_BINST(T)                                                                                  \
  template void op_bspmv<T>(const DCsr &, const T *, T *, int, DevBuf<double> &, hipStream_t);       \
  template int tune_spmm<T>(DCsr &, int, DevBuf<double> &, hipStream_t);                             \
  template void op_bresidual<T>(const DCsr &, const T *, const T *, T *, int, DevBuf<double> &,     \
                                hipStream_t);                                                        \
  template void op_bcheb_step<T>(const DCsr &, const T *, const T *, const T *, const T *, T *,     \
                                 double, double, int, DevBuf<double> &, hipStream_t);                \
  template void op_binterp<T>(const DCsr &, const T *, const T *, const T *, T *, int,              \
                              DevBuf<double> &, hipStream_t);                                        \
  template void op_bprolong_add<T>(const int32_t *, int64_t, const T *, T *, int, hipStream_t);      \
  template void op_bdense_apply<T>(const double *, int64_t, const T *, T *, int, hipStream_t);       \
  template void RedPlan::bpartials<T>(int, int, const T *, const T *, const T *, const T *,          \
                                      DevBuf<double> &, hipStream_t) const;                          \
  template void RedPlan::bdots<T>(int, int, const T *, const T *, const T *, const T *, double *,    \
                                  DevBuf<double> &, hipStream_t) const;                              \
  template void op_bspmv_first<T>(const DCsr &, const T *, T *, const FirstStep<T> &, int,             \
                                  DevBuf<double> &, hipStream_t);                                    \
  template void op_kr_bpupdate<T>(T *, const T *, int, const RedPlan &, const double *, hipStream_t);
LG_BINST(double)
LG_BINST(float)
#undef LG_BINST
template void op_bsub_block_mean<double>(double *, int, const RedPlan &, const double *, hipStream_t);
#define LG_BKR(T, F)                                                                                            \
  template void op_kr_bbegin<T, F>(const RedPlan &, const T *, T *, T *, F *, const FirstStep<F> &, int,        \
                                   DevBuf<double> &, hipStream_t);                                             \
  template void op_kr_bupdate<T, F>(const RedPlan &, T *, T *, const T *, const T *, F *, const FirstStep<F> &, \
                                    int, const double *, DevBuf<double> &, hipStream_t);                       \
  template void op_bcenter<T, F>(const RedPlan &, T *, const F *, const T *, int, const double *,              \
                                 DevBuf<double> &, hipStream_t);
LG_BKR(double, double)
LG_BKR(double, float)
LG_BKR(float, float)
#undef LG_BKR

}  // namespace lg
