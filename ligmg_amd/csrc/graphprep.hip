// Graph preprocessing on the device: input validation, connected
// components, largest-component extraction and adjacency -> Laplacian.
//
// The reference does these steps in its driver on CombBLAS matrices:
// connected_components (cc.hpp:22-51) iterates a max-label SpMV to a fixed
// point, largest_cc (cc.hpp:55-105) keeps the biggest component renumbered
// in ascending order, and main.cpp:79-110 forms L = D - A.  Here components
// come from hook-and-shortcut passes (every root is hooked below its
// smallest neighbouring root, then every vertex jumps to its root), which
// need O(log n) full passes instead of O(diameter); the reference's labels
// (largest index of the component) are then read off the final forest, so
// the result is the same.  Every kernel is a bounded data-parallel pass: the
// host repeats them until nothing changes.
#include <algorithm>
#include <mutex>
#include <string>

#include "../../include/ligmg_amd.h"
#include "prims.hpp"
#include "setup.hpp"

namespace lg {

namespace {

// pass 1 reads only the row pointers: rp[0] = 0, non-decreasing, rp[n] = m
__global__ void k_rowptr_check(int64_t n, int64_t m, const int32_t *rp, int *bad) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t a = rp[i];
    if ((i == 0 && a != 0) || (i == n && a != m) || (i < n && rp[i + 1] < a)) atomicOr(bad, 1);
  }
}

// pass 2, once the row pointers are known good: columns in [0, ncols)
__global__ void k_colind_check(int64_t m, int64_t ncols, const int32_t *ci, int *bad) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < m;
       k += (int64_t)gridDim.x * blockDim.x)
    if (ci[k] < 0 || ci[k] >= ncols) atomicOr(bad, 2);
}

__global__ void k_cc_init(int64_t n, int32_t *parent) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    parent[i] = (int32_t)i;
}

// The passes over stored entries below deal edge_chunk consecutive entries to
// each wavefront, whatever rows they belong to, so a hub row is spread over
// many wavefronts and short rows share one.  With a wavefront per row an
// R-MAT 20 adjacency (33.5 M entries, 1.25 M rows, hubs of 10^5 entries) spent
// most of its time on lanes without an entry and on the hubs: hook 8.3 ms a
// pass, count 2.1 ms, fill 5.6 ms; a thread per row took 34.6 ms for the
// Laplacian's fill.  Each lane finds its entry's row by a binary search among
// the few rows of its wavefront's chunk (the row pointers it reads stay in L1).
// A chunk is a chain of 64-entry steps, so below 4 M entries chunks shrink, to
// 64 entries, while that keeps at most EDGE_WAVES wavefronts (2000 entries: a
// pass 16 to 25 -> 4 to 6 us, largest component 0.530 -> 0.437 ms; 330 000
// entries 0.605 -> 0.496 ms; 3.3 M 0.753 -> 0.751).
constexpr int EDGE_CHUNK = 1024;
constexpr int64_t EDGE_WAVES = 4096;
__host__ __device__ inline int64_t edge_chunk(int64_t m) {
  int64_t c = WAVE;
  while (c < EDGE_CHUNK && c * EDGE_WAVES < m) c <<= 1;
  return c;
}
inline unsigned edge_grid(int64_t m) {
  const int64_t c = edge_chunk(m), waves = (m + c - 1) / c;
  return (unsigned)std::max<int64_t>(1, (waves + 3) / 4);
}

// the row of stored entry k: the last r in [lo, hi] with rp[r] <= k, given
// rp[lo] <= k < rp[hi + 1]
__device__ __forceinline__ int64_t entry_row(const int32_t *__restrict__ rp, int64_t lo, int64_t hi, int64_t k) {
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (rp[mid] <= k) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// f(k, row, ok) for the entries of this wavefront's chunk, 64 at a time in
// stored order; the whole wavefront calls f together, ok marks lanes that
// hold an entry (the others get the row of the chunk's last entry)
template <class F>
__device__ __forceinline__ void for_entries(int64_t n, int64_t m, const int32_t *__restrict__ rp, const F &f) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t c = edge_chunk(m), k0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / WAVE * c;
  if (k0 >= m) return;
  const int64_t k1 = min(k0 + c, m);
  const int64_t r0 = entry_row(rp, 0, n - 1, k0), r1 = entry_row(rp, r0, n - 1, k1 - 1);
  for (int64_t base = k0; base < k1; base += WAVE) {
    const int64_t k = base + lane;
    const bool ok = k < k1;
    f(k, entry_row(rp, r0, r1, ok ? k : k1 - 1), ok);
  }
}

// First pass: the smallest neighbour below each vertex becomes its parent.
// The lanes of one row take their minimum by a segmented scan, so a row
// costs one atomic per 64 entries and hubs are not contended.
__global__ void __launch_bounds__(256) k_cc_first(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                  const int32_t *__restrict__ ci, int32_t *parent) {
  const int lane = threadIdx.x & (WAVE - 1);
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    int32_t v = ok ? ci[k] : INT32_MAX;
    const int32_t r = (int32_t)row;
    for (int off = 1; off < WAVE; off <<= 1) {
      const int32_t ov = __shfl_up(v, off, WAVE), orow = __shfl_up(r, off, WAVE);
      if (lane >= off && orow == r) v = min(v, ov);
    }
    const int32_t nrow = __shfl_down(r, 1, WAVE);
    if ((lane == WAVE - 1 || nrow != r) && v < r) atomicMin(&parent[r], v);
  });
}

// every parent is a vertex of the same component with a smaller or equal
// index, so hooking a root below a smaller root (atomicMin) never closes a
// cycle, whatever order the edges are seen in.  After the first pass almost
// every entry joins two vertices of one star; where it does not, the plain
// read before the atomic skips the roots that are already hooked lower (a
// stale value only costs the atomic it would have skipped).
__global__ void __launch_bounds__(256) k_cc_hook(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                 const int32_t *__restrict__ ci, int32_t *parent, int *changed) {
  bool ch = false;
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    if (!ok) return;
    const int32_t pu = parent[row], pv = parent[ci[k]];
    const int32_t lo = min(pu, pv), hi = max(pu, pv);
    if (lo < hi && parent[hi] > lo && atomicMin(&parent[hi], lo) > lo) ch = true;
  });
  if (__any(ch) && (threadIdx.x & (WAVE - 1)) == 0) atomicOr(changed, 1);
}

// shortcut: every vertex points at its root (parents strictly decrease
// along a path, so the walk ends)
__global__ void k_cc_jump(int64_t n, int32_t *parent) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    int32_t p = parent[i];
    while (true) {
      const int32_t q = parent[p];
      if (q >= p) break;
      p = q;
    }
    parent[i] = p;
  }
}

// Largest vertex index and size of every component (indexed by its root).
// A root counts itself; the other lanes of a wavefront are grouped by root,
// and each wavefront keeps the sums of the root it met first in registers:
// with one atomic pair per vertex the giant component's two words were
// contended for 8.9 ms on R-MAT 20.
__global__ void __launch_bounds__(256) k_cc_stats(int64_t n, const int32_t *parent, int32_t *maxv, int32_t *count) {
  const int lane = threadIdx.x & (WAVE - 1);
  int32_t kept = -1, kmax = -1, kcnt = 0;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = blockIdx.x * (int64_t)blockDim.x + threadIdx.x - lane; base < n; base += step) {
    const int64_t i = base + lane;
    const int32_t r = i < n ? parent[i] : -1;
    if (r == i) {
      atomicMax(&maxv[r], r);
      atomicAdd(&count[r], 1);
    }
    uint64_t left = __ballot(i < n && r != i);
    while (left) {
      const int first = __ffsll((unsigned long long)left) - 1;
      const int32_t root = __shfl(r, first, WAVE);
      const uint64_t same = __ballot(r == root) & left;
      const int32_t top = (int32_t)(base + (63 - __clzll((long long)same))), c = __popcll(same);
      if (kept < 0) kept = root;
      if (root == kept) {
        kmax = max(kmax, top);
        kcnt += c;
      } else if (lane == 0) {
        atomicMax(&maxv[root], top);
        atomicAdd(&count[root], c);
      }
      left &= ~same;
    }
  }
  if (kept >= 0 && lane == 0) {
    atomicMax(&maxv[kept], kmax);
    atomicAdd(&count[kept], kcnt);
  }
}

// the component of the largest count, among equals the one of the smallest
// label: the maximum of count << 32 | (INT32_MAX - label)
__global__ void __launch_bounds__(256) k_cc_best(int64_t n, const int32_t *count, const int32_t *maxv,
                                                 unsigned long long *key) {
  unsigned long long best = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (count[i] > 0) {
      const unsigned long long q = ((unsigned long long)count[i] << 32) | (uint32_t)(INT32_MAX - maxv[i]);
      best = best < q ? q : best;
    }
  for (int off = WAVE / 2; off >= 1; off >>= 1) {
    const unsigned long long q = __shfl_xor(best, off, WAVE);
    best = best < q ? q : best;
  }
  if ((threadIdx.x & (WAVE - 1)) == 0 && best) atomicMax(key, best);
}

// new ids are -1 (bad |= 1 otherwise) or a rank below n_out used once (bad |= 2)
__global__ void k_ids_check(int64_t n, int64_t n_out, const int32_t *ids, int32_t *seen, int *bad) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t q = ids[i];
    if (q < -1 || q >= n_out) atomicOr(bad, 1);
    else if (q >= 0 && atomicExch(&seen[q], 1) != 0) atomicOr(bad, 2);
  }
}

__global__ void k_cc_label(int64_t n, const int32_t *parent, const int32_t *maxv, int32_t *label) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    label[i] = maxv[parent[i]];
}

__global__ void k_keep_flags(int64_t n, const int32_t *parent, int32_t root, int32_t *flag) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= n;
       i += (int64_t)gridDim.x * blockDim.x)
    flag[i] = (i < n && parent[i] == root) ? 1 : 0;
}

__global__ void k_keep_ids(int64_t n, const int32_t *flag, const int32_t *scan, int32_t *new_id) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    new_id[i] = flag[i] ? scan[i] : -1;
}

// kept entries per kept row, in the order of the rows' new ids (cnt zeroed
// before): the lanes of a row count themselves, one atomic per 64 entries
__global__ void __launch_bounds__(256) k_sub_count(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                   const int32_t *__restrict__ ci,
                                                   const int32_t *__restrict__ new_id, int32_t *cnt) {
  const int lane = threadIdx.x & (WAVE - 1);
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    const uint64_t kept = __ballot(ok && new_id[ci[k]] >= 0);
    const int64_t prev = __shfl_up(row, 1, WAVE);
    const bool head = lane == 0 || prev != row;
    const uint64_t heads = __ballot(head);
    if (!head) return;
    const int32_t nr = new_id[row];
    if (nr < 0) return;
    const uint64_t above = lane == WAVE - 1 ? 0 : heads >> (lane + 1);
    const int len = above ? __ffsll((unsigned long long)above) : WAVE - lane;
    const uint64_t seg = (len == WAVE ? ~0ull : ((1ull << len) - 1)) << lane;
    const int c = __popcll(kept & seg);
    if (c) atomicAdd(&cnt[nr], c);
  });
}

// Kept rows whose entries are all kept (every row, when the kept vertices
// are whole components): entry k goes to its place in the row.
__global__ void __launch_bounds__(256) k_sub_fill_whole(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                        const int32_t *__restrict__ ci,
                                                        const double *__restrict__ v,
                                                        const int32_t *__restrict__ new_id,
                                                        const int32_t *__restrict__ orp, int32_t *oci, double *ov) {
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    if (!ok) return;
    const int32_t nr = new_id[row];
    if (nr < 0) return;
    const int32_t a = rp[row], o = orp[nr];
    if (orp[nr + 1] - o != rp[row + 1] - a) return;
    const int64_t pos = o + (k - a);
    oci[pos] = new_id[ci[k]];
    if (ov) ov[pos] = v[k];
  });
}

// the other kept rows, a wavefront each: it tests 64 rows at a time and
// compacts those that lose entries
__global__ void __launch_bounds__(256) k_sub_fill(int64_t n, const int32_t *rp, const int32_t *ci, const double *v,
                                                  const int32_t *new_id, const int32_t *orp, int32_t *oci,
                                                  double *ov) {
  const int lane = threadIdx.x & (WAVE - 1);
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int64_t nw = (int64_t)gridDim.x * blockDim.x / WAVE;
  for (int64_t r0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / WAVE * WAVE; r0 < n; r0 += nw * WAVE) {
    const int64_t rl = r0 + lane;
    const int32_t nl = rl < n ? new_id[rl] : -1;
    uint64_t todo = __ballot(nl >= 0 && orp[nl + 1] - orp[nl] != rp[rl + 1] - rp[rl]);
    while (todo) {
      const int q = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const int64_t r = r0 + q;
      int32_t o = orp[__shfl(nl, q, WAVE)];
      for (int32_t base = rp[r]; base < rp[r + 1]; base += WAVE) {
        const int32_t k = base + lane;
        const int32_t c = (k < rp[r + 1]) ? new_id[ci[k]] : -1;
        const uint64_t mk = __ballot(c >= 0);
        if (c >= 0) {
          const int32_t pos = o + __popcll(mk & lt);
          oci[pos] = c;
          if (ov) ov[pos] = v[k];
        }
        o += __popcll(mk);
      }
    }
  }
}

// Laplacian row lengths: A's row plus a diagonal slot, which k_lap_diag
// takes back from the rows whose diagonal A stores
__global__ void k_lap_len(int64_t n, const int32_t *rp, int32_t *len) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r <= n; r += (int64_t)gridDim.x * blockDim.x)
    len[r] = r < n ? rp[r + 1] - rp[r] + 1 : 0;
}
__global__ void __launch_bounds__(256) k_lap_diag(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                  const int32_t *__restrict__ ci, int32_t *len) {
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    if (ok && ci[k] == row) len[row] = rp[row + 1] - rp[row];
  });
}

// L_ij = -A_ij (j != i), L_ii = deg_i - A_ii, the diagonal inserted in
// column order when A has none (columns strictly increasing: it follows the
// last entry left of it).  Rows without entries: k_lap_empty.
__global__ void __launch_bounds__(256) k_lap_fill(int64_t n, int64_t m, const int32_t *__restrict__ rp,
                                                  const int32_t *__restrict__ ci, const double *__restrict__ v,
                                                  const double *__restrict__ deg,
                                                  const int32_t *__restrict__ orp, int32_t *oci, double *ov) {
  for_entries(n, m, rp, [&](int64_t k, int64_t row, bool ok) {
    if (!ok) return;
    const int32_t a = rp[row], b = rp[row + 1], oa = orp[row], c = ci[k];
    const bool has = orp[row + 1] - oa == b - a;  // A stores the diagonal
    const int64_t o = oa + (k - a) + (!has && c > row ? 1 : 0);
    oci[o] = c;
    ov[o] = c == row ? deg[row] - v[k] : 0.0 - v[k];
    if (has) return;
    const bool before = c > row && (k == a || ci[k - 1] < row), after = c < row && k == b - 1;
    if (before || after) {
      const int64_t od = before ? o - 1 : o + 1;
      oci[od] = (int32_t)row;
      ov[od] = deg[row];
    }
  });
}
__global__ void k_lap_empty(int64_t n, const int32_t *rp, const double *deg, const int32_t *orp, int32_t *oci,
                            double *ov) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
    if (rp[r] == rp[r + 1]) {
      oci[orp[r]] = (int32_t)r;
      ov[orp[r]] = deg[r];
    }
}

unsigned gs(int64_t work) { return grid_for(work, 256, 16384); }
// k_cc_stats: a wavefront ends with one atomic pair, so 512 workgroups at most
unsigned stat_grid(int64_t n) { return grid_for(n, 256, 512); }

// device copies of caller arrays (or views of device ones)
template <class T>
struct In {
  DevBuf<T> own;
  const T *p = nullptr;
  In(const T *src, int64_t cnt, int mem, hipStream_t s) {
    if (mem == LIGMG_MEM_DEVICE || !src) {
      p = src;
    } else {
      own.alloc(std::max<int64_t>(cnt, 1));
      to_device(own.p, src, cnt, s);
      p = own.p;
    }
  }
};

template <class T>
void out_copy(T *dst, const T *src, int64_t cnt, int mem, hipStream_t s) {
  if (cnt <= 0) return;
  if (mem == LIGMG_MEM_DEVICE) d2d(dst, src, cnt, s);
  else to_host(dst, src, cnt, s);
}

// whether two device arrays share memory (inputs that the caller also names
// as output are read to the end before it is written)
inline bool overlap(const void *a, size_t na, const void *b, size_t nb) {
  return a && b && (const char *)a < (const char *)b + nb && (const char *)b < (const char *)a + na;
}

// A caller's output array of cnt entries.  Device memory apart from the
// inputs is written in place; host memory, and device memory that overlaps
// an input, through a buffer that finish copies.  Null stays null.
template <class T>
struct Out {
  DevBuf<T> own;
  T *p, *dst = nullptr;
  int64_t cnt;
  int mem;
  Out(T *out, int64_t c, int mem_kind, bool overlaps_input) : p(out), cnt(c), mem(mem_kind) {
    if (!out || (mem == LIGMG_MEM_DEVICE && !overlaps_input)) return;
    own.alloc(std::max<int64_t>(c, 1));
    p = own.p;
    dst = out;
  }
  void finish(hipStream_t s) {
    if (dst) out_copy(dst, (const T *)p, cnt, mem, s);
  }
};

// cnt: zeroed
void sub_count(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, const int32_t *new_id, int32_t *cnt,
               hipStream_t s) {
  if (m == 0) return;
  hipLaunchKernelGGL(k_sub_count, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, new_id, cnt);
  LG_LAUNCH_CHECK();
}

void sub_fill(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, const double *v, const int32_t *new_id,
              const int32_t *orp, int32_t *oci, double *ov, hipStream_t s) {
  if (m == 0) return;
  hipLaunchKernelGGL(k_sub_fill_whole, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, v, new_id, orp, oci, ov);
  LG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sub_fill, dim3(gs(n)), dim3(256), 0, s, n, rp, ci, v, new_id, orp, oci, ov);
  LG_LAUNCH_CHECK();
}

void lap_lengths(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, int32_t *len, hipStream_t s) {
  hipLaunchKernelGGL(k_lap_len, dim3(gs(n + 1)), dim3(256), 0, s, n, rp, len);
  LG_LAUNCH_CHECK();
  if (m == 0) return;
  hipLaunchKernelGGL(k_lap_diag, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, len);
  LG_LAUNCH_CHECK();
}

void lap_fill(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, const double *v, const double *deg,
              const int32_t *orp, int32_t *oci, double *ov, hipStream_t s) {
  hipLaunchKernelGGL(k_lap_empty, dim3(gs(n)), dim3(256), 0, s, n, rp, deg, orp, oci, ov);
  LG_LAUNCH_CHECK();
  if (m == 0) return;
  hipLaunchKernelGGL(k_lap_fill, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, v, deg, orp, oci, ov);
  LG_LAUNCH_CHECK();
}

int64_t nnz_of(const int32_t *rp, int64_t n, int mem, hipStream_t s) {
  int32_t e[2];
  if (mem == LIGMG_MEM_DEVICE) {
    to_host(&e[0], rp, 1, s);
    to_host(&e[1], rp + n, 1, s);
    LG_HIP(hipStreamSynchronize(s));
  } else {
    e[0] = rp[0];
    e[1] = rp[n];
  }
  LG_CHECK(e[0] == 0 && e[1] >= 0, LIGMG_ERR_INVALID, "rowptr[0] must be 0 and rowptr[n] >= 0");
  return e[1];
}

// roots (count > 0) of the forest: the number of components
__global__ void k_cc_count_roots(int64_t n, const int32_t *count, int *ncomp) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    if (count[i] > 0) atomicAdd(ncomp, 1);
}

// hooks + shortcuts to a forest of stars whose roots are the smallest index
// of every component; changed is one word of device scratch
void cc_forest_into(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, int32_t *parent, int *changed,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_cc_init, dim3(gs(n)), dim3(256), 0, s, n, parent);
  LG_LAUNCH_CHECK();
  if (m == 0) return;
  hipLaunchKernelGGL(k_cc_first, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, parent);
  LG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_cc_jump, dim3(gs(n)), dim3(256), 0, s, n, parent);
  LG_LAUNCH_CHECK();
  for (int round = 0;; round++) {
    LG_CHECK(round < 256, LIGMG_ERR_NUMERIC, "connected components did not converge");
    fill_i32(changed, 0, 1, s);
    hipLaunchKernelGGL(k_cc_hook, dim3(edge_grid(m)), dim3(256), 0, s, n, m, rp, ci, parent, changed);
    LG_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_cc_jump, dim3(gs(n)), dim3(256), 0, s, n, parent);
    LG_LAUNCH_CHECK();
    int h = 0;
    to_host(&h, changed, 1, s);
    LG_HIP(hipStreamSynchronize(s));
    if (!h) break;
  }
}

void cc_forest(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, DevBuf<int32_t> &parent, hipStream_t s) {
  parent.alloc(n);
  DevBuf<int> changed(1);
  cc_forest_into(n, m, rp, ci, parent.p, changed.p, s);
}

// connected_components on a validated device CSR, into caller buffers:
// parent, maxv and count hold n words each, flags 2 (the forest's change
// flag, the component count); label (device, n) receives the labels.
// Returns the number of components.  Every buffer is written before it is
// read, so scratch left over from an earlier call does not matter.
int64_t cc_labels_into(int64_t n, int64_t m, const int32_t *rp, const int32_t *ci, int32_t *parent, int32_t *maxv,
                       int32_t *count, int *flags, int32_t *label, hipStream_t s) {
  cc_forest_into(n, m, rp, ci, parent, flags, s);
  fill_i32(maxv, -1, n, s);
  fill_i32(count, 0, n, s);
  fill_i32(flags + 1, 0, 1, s);
  hipLaunchKernelGGL(k_cc_stats, dim3(stat_grid(n)), dim3(256), 0, s, n, (const int32_t *)parent, maxv, count);
  LG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_cc_label, dim3(gs(n)), dim3(256), 0, s, n, (const int32_t *)parent, (const int32_t *)maxv,
                     label);
  LG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_cc_count_roots, dim3(gs(n)), dim3(256), 0, s, n, (const int32_t *)count, flags + 1);
  LG_LAUNCH_CHECK();
  int k = 0;
  to_host(&k, flags + 1, 1, s);
  LG_HIP(hipStreamSynchronize(s));
  return k;
}

}  // namespace

// pass 3 (optional): strictly increasing columns within every row.  An entry
// not above its predecessor must start a row, which only such entries search.
__global__ void k_sorted_check(int64_t n, int64_t m, const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                               int *bad) {
  bool ok = true;
  for (int64_t k = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < m; k += (int64_t)gridDim.x * blockDim.x)
    if (ci[k - 1] >= ci[k]) ok &= rp[entry_row(rp, 0, n - 1, k)] == k;
  if (!__all(ok) && (threadIdx.x & (WAVE - 1)) == 0) atomicOr(bad, 4);
}

// bad: one word of device scratch
void validate_csr_into(int64_t n, int64_t ncols, const int32_t *rp, const int32_t *ci, hipStream_t s, bool sorted,
                       int *bad) {
  int32_t m = 0;
  to_host(&m, rp + n, 1, s);
  LG_HIP(hipStreamSynchronize(s));
  LG_CHECK(m >= 0, LIGMG_ERR_INVALID, "rowptr[n] must be non-negative");
  fill_i32(bad, 0, 1, s);
  hipLaunchKernelGGL(k_rowptr_check, dim3(gs(n + 1)), dim3(256), 0, s, n, (int64_t)m, rp, bad);
  LG_LAUNCH_CHECK();
  int h = 0;
  to_host(&h, bad, 1, s);
  LG_HIP(hipStreamSynchronize(s));
  LG_CHECK(!(h & 1), LIGMG_ERR_INVALID, "rowptr must start at 0 and be non-decreasing");
  hipLaunchKernelGGL(k_colind_check, dim3(gs(m)), dim3(256), 0, s, (int64_t)m, ncols, ci, bad);
  LG_LAUNCH_CHECK();
  to_host(&h, bad, 1, s);
  LG_HIP(hipStreamSynchronize(s));
  LG_CHECK(!(h & 2), LIGMG_ERR_INVALID, "column index out of range");
  if (sorted) {
    hipLaunchKernelGGL(k_sorted_check, dim3(gs(m)), dim3(256), 0, s, n, (int64_t)m, rp, ci, bad);
    LG_LAUNCH_CHECK();
    to_host(&h, bad, 1, s);
    LG_HIP(hipStreamSynchronize(s));
    LG_CHECK(!(h & 4), LIGMG_ERR_INVALID, "columns must be sorted and unique within every row");
  }
}

void validate_csr(int64_t n, int64_t ncols, const int32_t *rp, const int32_t *ci, hipStream_t s, bool sorted) {
  DevBuf<int> bad(1);
  validate_csr_into(n, ncols, rp, ci, s, sorted, bad.p);
}

}  // namespace lg

// Scratch of ligmg_components_noalloc: parent, per-root maximum and per-root
// count (LIGMG_NOALLOC_CC_MAX_N words each), then flag words.  Each GPU the
// library runs on holds its own copy until the process ends.  Host code
// never uses this name as an address: scratch_on_device() looks the
// device's copy up once per device.
constexpr int64_t NOALLOC_CC_N = LIGMG_NOALLOC_CC_MAX_N;
constexpr int64_t NOALLOC_CC_WORDS = 3 * NOALLOC_CC_N + 64;
static __device__ __align__(256) int32_t scratch[NOALLOC_CC_WORDS];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mu;
int32_t *scratch_addr[MAX_DEVICES] = {};

// this device's copy of scratch, looked up on the first call on the device
int32_t *scratch_on_device() {
  int dev = 0;
  LG_HIP(hipGetDevice(&dev));
  LG_CHECK(dev >= 0 && dev < MAX_DEVICES, LIGMG_ERR_DEVICE, "device index out of range");
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_addr[dev]) {
    void *p = nullptr;
    LG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    scratch_addr[dev] = (int32_t *)p;
  }
  return scratch_addr[dev];
}

thread_local hipStream_t prep_stream = nullptr;
hipStream_t prep_s() {
  if (!prep_stream) LG_HIP(hipStreamCreateWithFlags(&prep_stream, hipStreamNonBlocking));
  return prep_stream;
}
int prep_fail(const lg::Error &e) {
  lg::g_last_error = e.what();
  return e.code;
}
}  // namespace

extern "C" {

int ligmg_components(int64_t n, const int32_t *rowptr, const int32_t *colind, int mem_kind, int32_t *label,
                     int64_t *ncomp) {
  if (n <= 0 || n >= INT32_MAX || !rowptr || !colind || !label) return LIGMG_ERR_INVALID;
  try {
    hipStream_t s = prep_s();
    const int64_t m = lg::nnz_of(rowptr, n, mem_kind, s);
    lg::In<int32_t> rp(rowptr, n + 1, mem_kind, s), ci(colind, m, mem_kind, s);
    lg::validate_csr(n, n, rp.p, ci.p, s, false);
    lg::DevBuf<int32_t> parent(n), maxv(n), count(n), lab(n);
    lg::DevBuf<int> flags(2);
    const int64_t k = lg::cc_labels_into(n, m, rp.p, ci.p, parent.p, maxv.p, count.p, flags.p, lab.p, s);
    lg::out_copy(label, (const int32_t *)lab.p, n, mem_kind, s);
    if (ncomp) *ncomp = k;
    LG_HIP(hipStreamSynchronize(s));
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

int ligmg_components_noalloc(int64_t n, const int32_t *rowptr, const int32_t *colind, int32_t *label,
                             int64_t *ncomp) {
  if (n <= 0 || !rowptr || !colind || !label) return LIGMG_ERR_INVALID;
  if (n > NOALLOC_CC_N) {
    lg::g_last_error = "ligmg_components_noalloc: n = " + std::to_string(n) + " is above the maximum of " +
                       std::to_string(NOALLOC_CC_N) + " vertices (use ligmg_components)";
    return LIGMG_ERR_INVALID;
  }
  try {
    // the calling thread's default stream of the current device: no stream
    // is created either
    hipStream_t s = hipStreamPerThread;
    int32_t *sc = scratch_on_device();
    int32_t *parent = sc, *maxv = sc + NOALLOC_CC_N, *count = sc + 2 * NOALLOC_CC_N;
    int *flags = (int *)(sc + 3 * NOALLOC_CC_N);
    const int64_t m = lg::nnz_of(rowptr, n, LIGMG_MEM_DEVICE, s);
    lg::validate_csr_into(n, n, rowptr, colind, s, false, flags + 2);
    const int64_t k = lg::cc_labels_into(n, m, rowptr, colind, parent, maxv, count, flags, label, s);
    if (ncomp) *ncomp = k;
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

int ligmg_largest_component(int64_t n, const int32_t *rowptr, const int32_t *colind, int mem_kind,
                            int32_t *new_id, int64_t *n_out, int64_t *nnz_out) {
  if (n <= 0 || n >= INT32_MAX || !rowptr || !colind || !new_id || !n_out || !nnz_out) return LIGMG_ERR_INVALID;
  try {
    hipStream_t s = prep_s();
    const int64_t m = lg::nnz_of(rowptr, n, mem_kind, s);
    lg::In<int32_t> rp(rowptr, n + 1, mem_kind, s), ci(colind, m, mem_kind, s);
    lg::validate_csr(n, n, rp.p, ci.p, s, false);
    lg::DevBuf<int32_t> parent, maxv(n), count(n);
    lg::cc_forest(n, m, rp.p, ci.p, parent, s);
    lg::fill_i32(maxv.p, -1, n, s);
    lg::fill_i32(count.p, 0, n, s);
    hipLaunchKernelGGL(lg::k_cc_stats, dim3(lg::stat_grid(n)), dim3(256), 0, s, n, (const int32_t *)parent.p, maxv.p,
                       count.p);
    LG_LAUNCH_CHECK();
    // the largest count; among equals the smallest label (cc.hpp:71-72:
    // max_element over counts indexed by label returns the first maximum)
    lg::DevBuf<unsigned long long> key(1);
    lg::fill_u8((uint8_t *)key.p, 0, sizeof(*key.p), s);
    hipLaunchKernelGGL(lg::k_cc_best, dim3(lg::stat_grid(n)), dim3(256), 0, s, n, (const int32_t *)count.p,
                       (const int32_t *)maxv.p, key.p);
    LG_LAUNCH_CHECK();
    unsigned long long k = 0;
    lg::to_host(&k, key.p, 1, s);
    LG_HIP(hipStreamSynchronize(s));
    int32_t best = -1;  // the root of the vertex that names the component
    lg::to_host(&best, parent.p + (INT32_MAX - (int32_t)(k & 0x7fffffffull)), 1, s);
    LG_HIP(hipStreamSynchronize(s));
    lg::DevBuf<int32_t> flag(n + 1), scan(n + 1), ids(n), cnt(n + 1);
    hipLaunchKernelGGL(lg::k_keep_flags, dim3(lg::gs(n + 1)), dim3(256), 0, s, n, (const int32_t *)parent.p, best,
                       flag.p);
    LG_LAUNCH_CHECK();
    const int64_t nk = lg::exclusive_scan_i32(flag.p, scan.p, n + 1, s);
    hipLaunchKernelGGL(lg::k_keep_ids, dim3(lg::gs(n)), dim3(256), 0, s, n, (const int32_t *)flag.p,
                       (const int32_t *)scan.p, ids.p);
    LG_LAUNCH_CHECK();
    lg::fill_i32(cnt.p, 0, nk + 1, s);
    lg::sub_count(n, m, rp.p, ci.p, ids.p, cnt.p, s);
    lg::DevBuf<int32_t> cs(nk + 1);
    const int64_t mk = lg::exclusive_scan_i32(cnt.p, cs.p, nk + 1, s);
    lg::out_copy(new_id, (const int32_t *)ids.p, n, mem_kind, s);
    LG_HIP(hipStreamSynchronize(s));
    *n_out = nk;
    *nnz_out = mk;
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

int ligmg_extract(int64_t n, const int32_t *rowptr, const int32_t *colind, const double *vals,
                  const int32_t *new_id, int64_t n_out, int mem_kind, int32_t *out_rowptr, int32_t *out_colind,
                  double *out_vals) {
  if (n <= 0 || n >= INT32_MAX || !rowptr || !colind || !new_id || n_out < 0 || !out_rowptr || !out_colind)
    return LIGMG_ERR_INVALID;
  try {
    hipStream_t s = prep_s();
    const int64_t m = lg::nnz_of(rowptr, n, mem_kind, s);
    lg::In<int32_t> rp(rowptr, n + 1, mem_kind, s), ci(colind, m, mem_kind, s), ids(new_id, n, mem_kind, s);
    lg::In<double> v(vals, m, mem_kind, s);
    lg::validate_csr(n, n, rp.p, ci.p, s, false);
    // new ids must be -1 or a rank below n_out, each rank used once
    {
      lg::DevBuf<int32_t> seen(std::max<int64_t>(n_out, 1));
      lg::DevBuf<int> bad(1);
      lg::fill_i32(seen.p, 0, n_out, s);
      lg::fill_i32(bad.p, 0, 1, s);
      hipLaunchKernelGGL(lg::k_ids_check, dim3(lg::gs(n)), dim3(256), 0, s, n, n_out, ids.p, seen.p, bad.p);
      LG_LAUNCH_CHECK();
      int h = 0;
      lg::to_host(&h, bad.p, 1, s);
      LG_HIP(hipStreamSynchronize(s));
      LG_CHECK(!(h & 1), LIGMG_ERR_INVALID, "ligmg_extract: new_id out of range");
      LG_CHECK(!(h & 2), LIGMG_ERR_INVALID, "ligmg_extract: new_id repeats a rank");
    }
    lg::DevBuf<int32_t> cnt(n_out + 1), orp(n_out + 1);
    lg::fill_i32(cnt.p, 0, n_out + 1, s);
    lg::sub_count(n, m, rp.p, ci.p, ids.p, cnt.p, s);
    const int64_t mk = lg::exclusive_scan_i32(cnt.p, orp.p, n_out + 1, s);
    const size_t i4 = sizeof(int32_t), f8 = sizeof(double);
    auto meets = [&](const void *o, size_t bytes) {
      return lg::overlap(o, bytes, rowptr, (n + 1) * i4) || lg::overlap(o, bytes, colind, m * i4) ||
             lg::overlap(o, bytes, vals, m * f8) || lg::overlap(o, bytes, new_id, n * i4);
    };
    lg::Out<int32_t> oci(out_colind, mk, mem_kind, meets(out_colind, mk * i4));
    lg::Out<double> ov(v.p ? out_vals : nullptr, mk, mem_kind, meets(out_vals, mk * f8));
    lg::sub_fill(n, m, rp.p, ci.p, v.p, ids.p, orp.p, oci.p, ov.p, s);
    lg::out_copy(out_rowptr, (const int32_t *)orp.p, n_out + 1, mem_kind, s);
    oci.finish(s);
    ov.finish(s);
    LG_HIP(hipStreamSynchronize(s));
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

int ligmg_laplacian_nnz(int64_t n, const int32_t *rowptr, const int32_t *colind, int mem_kind, int64_t *nnz_out) {
  if (n <= 0 || n >= INT32_MAX || !rowptr || !colind || !nnz_out) return LIGMG_ERR_INVALID;
  try {
    hipStream_t s = prep_s();
    const int64_t m = lg::nnz_of(rowptr, n, mem_kind, s);
    lg::In<int32_t> rp(rowptr, n + 1, mem_kind, s), ci(colind, m, mem_kind, s);
    lg::validate_csr(n, n, rp.p, ci.p, s, false);
    lg::DevBuf<int32_t> len(n + 1), orp(n + 1);
    lg::lap_lengths(n, m, rp.p, ci.p, len.p, s);
    const int64_t tot = lg::exclusive_scan_i32(len.p, orp.p, n + 1, s);
    LG_CHECK(tot < INT32_MAX, LIGMG_ERR_INVALID, "Laplacian too large for int32 indices");
    *nnz_out = tot;
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

int ligmg_adjacency_to_laplacian(int64_t n, const int32_t *rowptr, const int32_t *colind, const double *vals,
                                 int mem_kind, int32_t *out_rowptr, int32_t *out_colind, double *out_vals) {
  if (n <= 0 || n >= INT32_MAX || !rowptr || !colind || !vals || !out_rowptr || !out_colind || !out_vals)
    return LIGMG_ERR_INVALID;
  try {
    hipStream_t s = prep_s();
    const int64_t m = lg::nnz_of(rowptr, n, mem_kind, s);
    lg::In<int32_t> rp(rowptr, n + 1, mem_kind, s), ci(colind, m, mem_kind, s);
    lg::In<double> v(vals, m, mem_kind, s);
    lg::validate_csr(n, n, rp.p, ci.p, s, true);  // the diagonal is inserted in column order
    lg::DevBuf<int32_t> len(n + 1), orp(n + 1);
    lg::lap_lengths(n, m, rp.p, ci.p, len.p, s);
    const int64_t tot = lg::exclusive_scan_i32(len.p, orp.p, n + 1, s);
    lg::DevBuf<double> deg(n);
    lg::row_sums_seq(n, rp.p, v.p, deg.p, s);
    const size_t i4 = sizeof(int32_t), f8 = sizeof(double);
    auto meets = [&](const void *o, size_t bytes) {
      return lg::overlap(o, bytes, rowptr, (n + 1) * i4) || lg::overlap(o, bytes, colind, m * i4) ||
             lg::overlap(o, bytes, vals, m * f8);
    };
    lg::Out<int32_t> oci(out_colind, tot, mem_kind, meets(out_colind, tot * i4));
    lg::Out<double> ov(out_vals, tot, mem_kind, meets(out_vals, tot * f8));
    lg::lap_fill(n, m, rp.p, ci.p, v.p, deg.p, orp.p, oci.p, ov.p, s);
    lg::out_copy(out_rowptr, (const int32_t *)orp.p, n + 1, mem_kind, s);
    oci.finish(s);
    ov.finish(s);
    LG_HIP(hipStreamSynchronize(s));
    return LIGMG_OK;
  } catch (const lg::Error &e) {
    return prep_fail(e);
  }
}

}  // extern "C"
