// The coarse levels of a V-cycle as one dense matrix (collapse.hip).
#pragma once
#include <vector>

#include "hierarchy.hpp"

namespace lg {

// Whether a level is small enough to collapse.  A product with 1024^2 entries
// (8 MiB, a quarter of the L2s' 32) takes about 4 us, one with 2048^2 (32 MiB,
// read from the Infinity Cache) about 10, the levels below 50 to 150 us of
// dependent launches: R-MAT 10 solve 1.37 -> 0.70 ms, 256 x 256 grid 14.6 ->
// 12.3 ms.  Forming the matrix takes about a dozen operations of nnz * n
// multiply-adds per level (0.2 ms at 1024), so sparse levels may be twice as
// large (the grid 6.5 -> 5.8 ms, 181 x 97 x 3 columns 4.7 -> 4.2 ms, a 250 K-vertex
// gradient with its setup 39.3 -> 37.5 ms) while a dense one of 1700 vertices cost a
// single solve 0.15 ms more than it gained.
inline bool collapse_fits(int64_t n, int64_t nnz) { return n <= 1024 || (n <= 2048 && nnz <= 16 * n); }

// What the cycle does besides its operators: smoother coefficients per level
// (al[l][k] and be[l][k] of step k), the smoother, the constant correction.
struct CycleCoeffs {
  const std::vector<std::vector<double>> &al_pre, &be_pre, &al_post, &be_post;
  int pre_smooth, post_smooth;
  bool jacobi;
  double scale;  // 4/3 with the constant correction, else 1
};

// out: the row-major n x n matrix of the FP64 V-cycle from level l down
// (n = H[l].A.n).  Queues its work on s.
void collapse_cycle(const std::vector<DLevel> &H, const CycleCoeffs &C, size_t l, DevBuf<double> &out,
                    hipStream_t s);

}  // namespace lg
