// Device code shared by the per-operator solve kernels (solve.hip,
// solver.hip) and the fused coarse-tail kernel (tail.hip): value access,
// SpMV epilogues, the wavefront sum and the per-block CG / FCG scalar
// logic.  Both paths evaluate the same expressions in the same order, so a
// level solved inside the fused tail produces the bits the separate
// launches produce.
#pragma once
#include "ops.hpp"

namespace lg {
namespace sdev {

// ------------------------------------------------------------ value access
// Matrix data is streamed once per product: non-temporal loads keep it from
// displacing the gathered vector in L2.
template <class T>
struct ValOne {
  __device__ __forceinline__ T operator()(int64_t) const { return (T)1; }
};
template <class T>
struct ValArr {
  const T *v;
  __device__ __forceinline__ T operator()(int64_t k) const { return __builtin_nontemporal_load(v + k); }
};

// --------------------------------------------------------------- epilogues
// Row sums are always accumulated in FP64 (a product of two FP32 numbers
// is exact in FP64), so the FP32 path only rounds storage, not the
// heavily cancelling Laplacian row sums of hub vertices.
// load(i) reads row i's other operands (asked for before the sum is known
// where a kernel can), put(i, s, load(i)) writes the result.
template <class T>
struct EpiStore {
  T *y;
  struct Pre {};
  __device__ __forceinline__ Pre load(int64_t) const { return {}; }
  __device__ __forceinline__ void put(int64_t r, double s, const Pre &) const { y[r] = (T)s; }
  __device__ __forceinline__ void operator()(int64_t r, double s) const { put(r, s, load(r)); }
};
// first Chebyshev step from a zero iterate: xn = beta dinv b
template <class T>
__device__ __forceinline__ T cheb_first(double beta, T dinv, T b) {
  return (T)(beta * (double)dinv * (double)b);
}

// y = s and the next cycle's first Chebyshev step from y
template <class T>
struct EpiFirst {
  T *y;
  const T *dinv;
  T *x;
  double beta;
  struct Pre {
    T dinv;
  };
  __device__ __forceinline__ Pre load(int64_t i) const { return {dinv[i]}; }
  __device__ __forceinline__ void put(int64_t i, double s, const Pre &p) const {
    const T v = (T)s;
    y[i] = v;
    x[i] = cheb_first<T>(beta, p.dinv, v);
  }
  __device__ __forceinline__ void operator()(int64_t i, double s) const { put(i, s, load(i)); }
};
template <class T>
struct EpiResid {
  const T *b;
  T *r;
  struct Pre {
    T b;
  };
  __device__ __forceinline__ Pre load(int64_t i) const { return {b[i]}; }
  __device__ __forceinline__ void put(int64_t i, double s, const Pre &p) const { r[i] = (T)((double)p.b - s); }
  __device__ __forceinline__ void operator()(int64_t i, double s) const { put(i, s, load(i)); }
};
template <class T>
struct EpiCheb {
  const T *dinv, *b, *xc, *xp;
  T *xn;
  double alpha, beta;
  struct Pre {
    T c, p, dinv, b;
  };
  // a null xp is a zero previous iterate (second step from a zero guess);
  // every other caller passes alpha = 0 with it
  __device__ __forceinline__ Pre load(int64_t i) const { return {xc[i], xp ? xp[i] : (T)0, dinv[i], b[i]}; }
  __device__ __forceinline__ void put(int64_t i, double s, const Pre &p) const {
    double c = (double)p.c;
    double d = alpha * (c - (double)p.p);
    xn[i] = (T)(c + d + beta * (double)p.dinv * ((double)p.b - s));
  }
  __device__ __forceinline__ void operator()(int64_t i, double s) const { put(i, s, load(i)); }
};
template <class T>
struct EpiInterp {
  const T *q, *b;
  T *x;
  struct Pre {
    T q, b;
  };
  __device__ __forceinline__ Pre load(int64_t i) const { return {q[i], b[i]}; }
  __device__ __forceinline__ void put(int64_t i, double s, const Pre &p) const {
    x[i] = (T)(s + (double)p.q * (double)p.b);
  }
  __device__ __forceinline__ void operator()(int64_t i, double s) const { put(i, s, load(i)); }
};
// adds d[i] x[i] (FP64) before the wrapped epilogue: the diagonal term of an
// FP32 operator stored in Laplacian form
template <class T, class Epi>
struct EpiDiag {
  const double *d;
  const T *x;
  Epi e;
  struct Pre {
    double d;
    T x;
    typename Epi::Pre e;
  };
  __device__ __forceinline__ Pre load(int64_t i) const { return {d[i], x[i], e.load(i)}; }
  __device__ __forceinline__ void put(int64_t i, double s, const Pre &p) const {
    e.put(i, s + p.d * (double)p.x, p.e);
  }
  __device__ __forceinline__ void operator()(int64_t i, double s) const { put(i, s, load(i)); }
};

// xor butterfly: every lane ends with the same bits
template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}

// xor butterfly over aligned groups of K lanes (K a power of two <= 64)
__device__ __forceinline__ double group_sum(double v, int K) {
  for (int off = K >> 1; off >= 1; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}

// ------------------------------------------------- CG / FCG scalar logic
// One set of scalars per (block, column): the Krylov coefficients of each
// independent graph are kept apart.  SC_ITS counts a batched set's iterations.
enum { SC_BN2 = 0, SC_RN2, SC_GAMMA, SC_DELTA, SC_T1, SC_ALPHA, SC_BETA, SC_ACTIVE, SC_GN, SC_ITS, SC_N };

__device__ __forceinline__ void kr_init(double *S) {
  for (int j = 0; j < SC_N; j++) S[j] = 0;
  S[SC_ACTIVE] = 1;
}
__device__ __forceinline__ void kr_alpha(double *S, int fcg) {
  double num = fcg ? S[SC_T1] : S[SC_GAMMA];
  S[SC_ALPHA] = (S[SC_ACTIVE] != 0 && S[SC_DELTA] != 0) ? num / S[SC_DELTA] : 0.0;
}
__device__ __forceinline__ void kr_check(double *S, double rtol) {
  if (S[SC_ACTIVE] != 0 && !(sqrt(S[SC_RN2]) > rtol * sqrt(S[SC_BN2]))) S[SC_ACTIVE] = 0;
}
// a set's norm for the host: the counter last, once the rest is visible
__device__ __forceinline__ void kr_publish(const KrSink &to, int64_t entry, bool init, double rn2, double active) {
  const unsigned long long k = init ? 1 : to.seq[entry] + 1;
  to.seq[entry] = k;
  volatile KrHost *h = to.host + entry;
  h->rn2 = rn2;
  h->active = active;
  __threadfence_system();
  h->seq = k;
}
__device__ __forceinline__ void kr_beta(double *S, int fcg) {
  if (fcg) {
    S[SC_BETA] = (S[SC_ACTIVE] != 0 && S[SC_DELTA] != 0) ? -S[SC_T1] / S[SC_DELTA] : 0.0;
  } else {
    S[SC_BETA] = (S[SC_ACTIVE] != 0 && S[SC_GAMMA] != 0) ? S[SC_GN] / S[SC_GAMMA] : 0.0;
    S[SC_GAMMA] = S[SC_GN];
  }
}

}  // namespace sdev
}  // namespace lg
