// How the workgroups of a launch share the cells of a rows x cols region in
// the kernels that touch each cell once (fill, hash, residual), with no
// division per cell.
#pragma once
#include <math.h>

namespace chm {
namespace jac {

// A thread's cells: rows row, row + row_step, ... and in each the columns
// col, col + col_step, ...
struct CellShare {
  int row, row_step, col, col_step;
};

constexpr int kCellsLog2 = 2;  // 4 cells of a row a thread, before it is split

// The smallest power of two that is at least cols, and at most threads.
__host__ __device__ inline int lanes_log2(int cols, int threads) {
  return cols >= threads ? 31 - __builtin_clz(threads)
         : cols <= 1     ? 0
                         : 32 - __builtin_clz(cols - 1);
}

// Thread t of workgroup wg of n_wg, of `threads` threads each (a power of
// two).  A workgroup takes a row at a time, or several of a region narrower
// than it is.  Of fewer rows than two turns of the workgroups each is cut into
// interleaved parts, down to four cells a thread, and each part has a team of
// workgroups, so that all have about the same to do.  (Whole rows only kept one
// workgroup busy on 1 x 2.7M cells, sixteen on 16 x 1M and half of them on
// 526 x 70506: a no-alloc solve of 2 sweeps of the first took 5117 us, now 160;
// the hash of the others 1330, now 58, and 183, now 120; of 1M x 16, where 16
// of 256 lanes had a cell, 424, now 62.  Grids of 2000 x 2000 are as fast.)
__host__ __device__ inline CellShare cell_share(int rows, int cols, int wg,
                                                int n_wg, int threads, int t) {
  if (rows <= 0 || cols <= 0) return {rows, 1, cols, 1};
  const int lg = lanes_log2(cols, threads), lanes = 1 << lg;
  const int pg = lanes_log2(threads, threads) - lg;  // 2^pg rows at a time
  const int groups = (rows + (1 << pg) - 1) >> pg;
  int segs = 1, team = n_wg, seg = 0, of_team = wg;
  const int most = cols >> (lg + kCellsLog2);
  // (an eighth of the last turn's workgroups may be idle: cut, 316 rows for
  // 316 workgroups would be eight turns of a seventh of a row)
  const bool full = groups <= n_wg ? groups > n_wg - n_wg / 8
                                   : groups > 2 * n_wg - n_wg / 8;
  if (!full && most > 1) {
    const int want = 8 * n_wg / groups;
    segs = want < most ? want : most;
    segs = segs < n_wg ? segs : n_wg;
    team = n_wg / segs;
    seg = wg / team;
    of_team = seg < segs ? wg - seg * team : groups;  // (left over)
  }
  CellShare s;
  s.row = (of_team << pg) + (t >> lg);
  s.row_step = team << pg;
  s.col = (seg << lg) + (t & (lanes - 1));
  s.col_step = segs << lg;
  return s;
}

// Workgroups that have something to do, at most `most`.
inline int cell_wgs(int rows, int cols, int threads, int most) {
  const int lg = lanes_log2(cols, threads);
  const int per = threads >> lg;
  const long long segs = cols >> (lg + kCellsLog2);
  const long long n =
      (long long)((rows + per - 1) / per) * (segs < 1 ? 1 : segs);
  return (int)(n < most ? n : most);
}

// Workgroups for a sum over the region, whose workgroups each end in one or two
// atomics on one cache line.  Those are done one after another, 9 ns each, and
// a thread's cells are too, so n workgroups take a cells / n + b n: least at a
// multiple of sqrt(cells), of which 1 / c is what runs of 64..1024 workgroups on
// 19 shapes gave: c 2.5 for the hash and the residual (one atomic), 5 for the
// hash that counts its workgroups besides.  500 x 2800: 256 workgroups take
// 30.1 and 14.6 us, 1024 37.0 and 30.8; 2800 x 2800: 54 and 39 us with 384, 45
// and 40 with 1024, which is the most: four a CU.
inline int sum_wgs(int rows, int cols, int threads, double c) {
  int n = 1024;
  const double best = sqrt((double)rows * (double)cols) / c;
  if (best < n) {
    n = best < 64 ? 64 : (int)best;
    // whole turns of whole rows where they are about as many (316 x 7627: 17.8
    // us with 316 workgroups, 19.4 with 310)
    const int per = threads >> lanes_log2(cols, threads);
    const int groups = rows / per + (rows % per > 0);
    if (5LL * groups >= 3 * n) {
      const int turns = (int)(((long long)2 * groups + n) / (2 * n));
      n = (groups - 1) / turns + 1;
    }
  }
  n = cell_wgs(rows, cols, threads, n);
  return n < 1 ? 1 : n > 1024 ? 1024 : n;  // (an empty region's sum is 0)
}

}  // namespace jac
}  // namespace chm
