// The stop filter of tolerance rounds that sum the last sweep only.
#pragma once
#include <math.h>

namespace chm {
namespace jac {

// Whether a round of `depth` sweeps over `cells` cells may hold the stop, that
// is, a sweep j whose exact residual S_j = sum floor(fl(d^2) 2^56) (saturating
// at 2^64 - 1 a cell) is at most thr.  a: the FP64 sum, in any order, of the
// last sweep's fl(d^2); m: the largest |u|.
//
// With D_j = u_j - u_{j-1}, D_{j+1} = 0.2 A D_j + e: A (a cell and its four
// neighbours) is symmetric with norm at most 5, and e is what two sweeps
// round, at most 2 x 3.8 x 2^-53 m a cell.  So |D_j| >= |D_n| - n E over the N
// cells for every earlier sweep, E = sqrt(N) 2^-48 m holding e four times over
// (0.2 is rounded up, which grows |u| and |D_j| by 2^-53 a sweep), and one sum
// of two operations per cell and round replaces n of three.  With it the exact
// S_j, which truncates less than 1 a cell, exceeds 2^56 (|D_n| - n E)^2 - N; a
// saturated term makes it more than any thr below 2^62.
__host__ __device__ inline bool last_sum_may_stop(double thr, double a,
                                                  double cells, double depth,
                                                  double m) {
  if (!(thr < 0x1.0p62)) return true;
  const double x =
      sqrt(a) * (1.0 - 0x1.0p-20) - depth * sqrt(cells) * m * 0x1.0p-48;
  return !(x > 0.0 && x * x * 0x1.0p56 * (1.0 - 0x1.0p-20) - cells >
                          thr * (1.0 + 0x1.0p-20));
}

}  // namespace jac
}  // namespace chm
