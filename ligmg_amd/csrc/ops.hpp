// Solve-phase device operators (row-block SpMV family, vector ops,
// deterministic reductions).  T is the vector element type (double or
// float); matrix values are read in the same precision (A.v or A.v32), or
// as 1 for pattern-only operators.
#pragma once
#include <algorithm>

#include "hierarchy.hpp"

namespace lg {

// Build the SpMV work units of A from its row pointers: the greedy packing
// of complete rows and UNIT_NNZ-chunks, on the device for operators of at
// least UNITS_DEVICE_MIN_ROWS rows.  build_units_host makes the same tables
// with a loop on the host.
constexpr int64_t UNITS_DEVICE_MIN_ROWS = 65536;
void build_units(DCsr &A, hipStream_t s);
void build_units_host(DCsr &A, hipStream_t s);
int32_t longest_row(const DCsr &A, hipStream_t s);
// Column-sliced copy of A for precision prec (0: FP64, 1: FP32) with
// slices of `width` columns (width >= ncols: no slicing).
void build_slices(DCsr &A, int prec, int64_t width, hipStream_t s);
// Milliseconds per y = A x launch (HIP events, `iters` launches), for tuning.
double time_spmv(const DCsr &A, int prec, int iters, hipStream_t s);

// FP32 copy of the values.  laplacian: store the operator in Laplacian form
// (rounded off-diagonals + FP64 diagonal = -their sum).
void make_v32(DCsr &A, hipStream_t s, bool laplacian = false);

// y = A x
template <class T> void op_spmv(const DCsr &A, const T *x, T *y, hipStream_t s);
// The first Chebyshev step of the cycle that takes y as its right-hand side,
// x = beta dinv y, written by y's producer (null x: none).
template <class T>
struct FirstStep {
  const T *dinv = nullptr;
  T *x = nullptr;
  double beta = 0;
};
template <class T>
void op_spmv_first(const DCsr &A, const T *x, T *y, const FirstStep<T> &f, hipStream_t s);
// r = b - A x
template <class T> void op_residual(const DCsr &A, const T *x, const T *b, T *r, hipStream_t s);
// One Chebyshev step: xn = xc + alpha (xc - xp) + beta dinv (b - A xc).
// With xc == nullptr the current iterate is zero: xn = beta dinv b.
template <class T>
void op_cheb_step(const DCsr &A, const T *dinv, const T *b, const T *xc, const T *xp, T *xn,
                  double alpha, double beta, hipStream_t s);
// x = P xc + q b (elimination interpolation, P has values)
template <class T>
void op_interp(const DCsr &P, const T *q, const T *xc, const T *b, T *x, hipStream_t s);
// x[i] += xc[agg[i]]
template <class T>
void op_prolong_add(const int32_t *agg, int64_t n, const T *xc, T *x, hipStream_t s);
// x[i] += (P xc + q b)[agg[i]], for P of short rows (row_k 1)
template <class T>
void op_prolong_interp(const int32_t *agg, int64_t n, const DCsr &P, const T *q, const T *xc, const T *b, T *x,
                       hipStream_t s);
// y = pinv x (dense n x n, FP64 matrix; T vectors)
template <class T>
void op_dense_apply(const double *Pinv, int64_t n, const T *x, T *y, hipStream_t s);

void op_d2f(const double *a, float *b, int64_t n, hipStream_t s);
void op_f2d(const float *a, double *b, int64_t n, hipStream_t s);

// What the host sees of a solve's convergence, in pinned memory, by Krylov set
// (a block, or a block's column); seq counts the norms of a solve from 1.
struct KrHost {
  double rn2, active;
  unsigned long long seq, pad;
};
// Up to this many sets are written to the host one by one; more are added up
// on the device first (kr_total), into the host's first entry.  A set's three
// words cross the bus on their own, about 0.1 us a set (12 000 sets 1.24 ms,
// 192 000 sets 25 ms of an iteration); adding them up takes a launch or two,
// 2 us more at 100 sets.
constexpr int KR_HOST_SETS = 128;
inline int kr_host_entries(int64_t sets) { return sets <= KR_HOST_SETS ? (int)sets : 1; }
// Where norms go besides the sets' own scalars: nowhere (host null), or to
// KR_HOST_SETS host entries, with as many counters on the device and
// KR_TOTAL_PARTS partials of kr_total.
constexpr int KR_TOTAL_PARTS = 2 * 256;
struct KrSink {
  KrHost *host = nullptr;
  unsigned long long *seq = nullptr;
  double *part = nullptr;
  // the sink a norm kernel writes set by set, none where kr_total follows
  KrSink each(int64_t sets) const { return sets <= KR_HOST_SETS ? *this : KrSink(); }
};
// r.r and the active flags of all sets, into the first host entry
void kr_total(const double *sc, int64_t sets, bool init, const KrSink &to, hipStream_t s);
// What follows a block reduction: its sums to out[(blk * np + j) * kp + c],
// or a scalar step of the Krylov sets (blk, c) on them (INIT, NORM: also for
// the host, when to has one).
struct BlockPost {
  enum Kind { OUT, INIT, NORM, ALPHA, BETA };
  Kind kind = OUT;
  double *out = nullptr, *sc = nullptr;
  int fcg = 0;
  double rtol = 0;
  KrSink to;
};

// Plan of a deterministic blocked reduction over vectors of length n split
// into contiguous blocks (independent graphs).  Stage 1 sums fixed chunks
// clipped to block boundaries (one workgroup each, fixed tree); stage 2
// adds the chunks of each block in order, so results are run-to-run
// reproducible.
struct RedPlan {
  int64_t n = 0;
  int nb = 1, nseg = 0, most = 0;  // most: segments of the block that has most
  DevBuf<int64_t> seg_lo, seg_hi;  // nseg
  DevBuf<int32_t> bseg;            // nb + 1
  DevBuf<int64_t> bptr;            // nb + 1 block offsets
  mutable DevBuf<double> part;     // nseg * 4
  std::vector<int64_t> hbptr;
  // segments of at most seg_rows rows (0: the vector dots' length)
  void build(int64_t n, const std::vector<int64_t> &blocks, hipStream_t s, int64_t seg_rows = 0);
  // out[c*np + j] = sum over block c of a_j[i] * b_j[i] (b_j == nullptr:
  // 1), j < np (np <= 4), accumulated in FP64.
  template <class T>
  void dots(int np, const T *const *a, const T *const *b, double *out, hipStream_t s) const;
  // out[c] = sum over block c of a[i]
  template <class T> void sums(const T *a, double *out, hipStream_t s) const;
  // block vectors (n x kp row-major): out[(blk * np + j) * kp + c] = sum over
  // block blk of a_j[i, c] * b_j[i, c]  (np <= 2, b_j == nullptr: 1)
  template <class T>
  void bdots(int np, int kp, const T *a0, const T *b0, const T *a1, const T *b1, double *out,
             DevBuf<double> &bpart, hipStream_t s) const;
  // segment partials only (part[(s * np + j) * kp + c]), for bfinish
  template <class T>
  void bpartials(int np, int kp, const T *a0, const T *b0, const T *a1, const T *b1, DevBuf<double> &bpart,
                 hipStream_t s) const;
  // the second stage and what follows it, from such partials
  void bfinish(int np, int kp, const BlockPost &P, const DevBuf<double> &bpart, hipStream_t s) const;
};

// One Krylov iteration on a level (sc: SC_N scalars per block): the start
// from x = 0, the norm of r with the convergence flag, then z = c - mean
// (with z.w: q for FCG, r for CG), p = z + beta p, the dots of q = A p (r only
// for FCG), and x += alpha p, r -= alpha q.  rf: also r in the cycle's type F;
// f: the cycle's first step from r.
template <class T, class F>
void kr_begin(const RedPlan &R, const T *b, T *x, T *r, F *rf, const FirstStep<F> &f, hipStream_t s);
void kr_norm(const RedPlan &R, double *sc, bool init, double rtol, const KrSink &to, hipStream_t s);
template <class T, class C>
void kr_center(const RedPlan &R, T *z, const C *c, const T *w, hipStream_t s);
template <class T>
void kr_pupdate(const RedPlan &R, T *p, const T *z, double *sc, bool fcg, hipStream_t s);
template <class T>
void kr_dots(const RedPlan &R, const T *p, const T *q, const T *r, hipStream_t s);
template <class T, class F>
void kr_update(const RedPlan &R, T *x, T *r, const T *p, const T *q, double *sc, bool fcg, F *rf,
               const FirstStep<F> &f, hipStream_t s);

// Device scalars of the eigenvalue estimate's CG by step (eig_begin, eig_step
// on a one-block plan): gamma (steps + 1), running flag (steps + 1), delta,
// alpha, beta (steps each).
struct EigState {
  double *G, *A, *D, *AL, *BE;
};
void eig_begin(const RedPlan &R, double *r, const double *dinv, double *z, double *p, const EigState &E, hipStream_t s);
// after q = A p
void eig_step(const RedPlan &R, double *r, const double *dinv, double *z, double *p, const double *q,
              const EigState &E, int it, hipStream_t s);

// a -= mean of a over each block, means taken from sums[c] (device)
template <class T> void op_sub_block_mean(T *a, const RedPlan &P, const double *sums, hipStream_t s);

// ---- block (k right-hand sides) operators, batch.hip.  Block vectors are
// row-major n x kp, kp a power of two <= 64.
template <class T>
void op_bspmv(const DCsr &A, const T *X, T *Y, int kp, DevBuf<double> &parts, hipStream_t s);
template <class T>
void op_bspmv_first(const DCsr &A, const T *X, T *Y, const FirstStep<T> &f, int kp, DevBuf<double> &parts,
                    hipStream_t s);
// picks A's batched SpMM tile for this precision and block width by timing
// the candidates once (kept in A.U); returns the tile id
template <class T>
int tune_spmm(DCsr &A, int kp, DevBuf<double> &parts, hipStream_t s);
// gathers in flight of tile id cfg
void spmm_tile(int cfg, int *u);
template <class T>
void op_bresidual(const DCsr &A, const T *X, const T *B, T *R, int kp, DevBuf<double> &parts,
                  hipStream_t s);
template <class T>
void op_bcheb_step(const DCsr &A, const T *dinv, const T *B, const T *Xc, const T *Xp, T *Xn,
                   double alpha, double beta, int kp, DevBuf<double> &parts, hipStream_t s);
template <class T>
void op_binterp(const DCsr &P, const T *q, const T *Xc, const T *B, T *X, int kp,
                DevBuf<double> &parts, hipStream_t s);
template <class T>
void op_bprolong_add(const int32_t *agg, int64_t n, const T *Xc, T *X, int kp, hipStream_t s);
// Y = Pm X with FP64 MFMA tiles (kp >= 16)
template <class T>
void op_bdense_apply(const double *Pm, int64_t n, const T *X, T *Y, int kp, hipStream_t s);
template <class T>
void op_bsub_block_mean(T *a, int kp, const RedPlan &P, const double *sums, hipStream_t s);
// Rows of a block vector's segment: 8192 entries, 16 pairs for each of a
// workgroup's 256 threads, at most the vector dots' 4096 rows; longer where
// there would be more than 2048 segments, whose partials one workgroup adds.
inline int64_t block_seg_rows(int64_t n, int kp) {
  const int64_t rows = kp >= 2 ? 8192 / kp : 4096;
  return std::max(rows, (n + 2047) / 2048);
}
// One block Krylov iteration, as the vector steps above: the start from x =
// 0, z = c - mean with the partials of z.w, p = z + beta p, and x += alpha p,
// r -= alpha q with the partials of r.r; rf, f as in kr_update.
template <class T, class F>
void op_kr_bbegin(const RedPlan &R, const T *b, T *x, T *r, F *rf, const FirstStep<F> &f, int kp,
                  DevBuf<double> &bpart, hipStream_t s);
template <class T, class C>
void op_bcenter(const RedPlan &R, T *z, const C *c, const T *w, int kp, const double *sums, DevBuf<double> &bpart,
                hipStream_t s);
template <class T, class F>
void op_kr_bupdate(const RedPlan &R, T *x, T *r, const T *p, const T *q, F *rf, const FirstStep<F> &f, int kp,
                   const double *sc, DevBuf<double> &bpart, hipStream_t s);
template <class T>
void op_kr_bpupdate(T *p, const T *z, int kp, const RedPlan &P, const double *sc, hipStream_t s);
// column-major n x k caller block <-> row-major n x kp internal block; the
// caller's vertex of internal row i is perm[i] (identity when perm is null)
void op_to_block(const double *B, int64_t n, int k, int kp, double *X, const int32_t *perm, hipStream_t s);
void op_from_block(const double *X, int64_t n, int k, int kp, double *B, const int32_t *perm,
                   hipStream_t s);

}  // namespace lg
