// How the workgroups of a launch share the cells of a rows x cols region in
// the kernels that touch each cell once (fill, hash, residual), with no
// division per cell.
#pragma once

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
// than it is.  Where that leaves workgroups over, each row is cut into as many
// interleaved parts as there are workgroups for, down to four cells a thread.
// (A whole row to a workgroup at any shape kept one busy on 1 x 2.7M
// cells and sixteen on 16 x 1M: a no-alloc solve of 2 sweeps of 1 x 2.7M took
// 5117 us, now 160; the hash of 16 x 1M 1330, now 60; of 1M x 16, where 16 of
// 256 lanes had a cell, 424, now 64.  Grids of 2000 x 2000 are as fast.)
__host__ __device__ inline CellShare cell_share(int rows, int cols, int wg,
                                                int n_wg, int threads, int t) {
  if (rows <= 0 || cols <= 0) return {rows, 1, cols, 1};
  const int lg = lanes_log2(cols, threads), lanes = 1 << lg;
  const int pg = lanes_log2(threads, threads) - lg;  // 2^pg rows at a time
  const int groups = (rows + (1 << pg) - 1) >> pg;
  CellShare s;
  int segs = 1, group = wg, seg = 0;
  if (groups < n_wg) {
    const int most = cols >> (lg + kCellsLog2);
    if (most > 1) {
      const int have = n_wg / groups;
      segs = have < most ? have : most;
    }
    if (wg >= groups) {
      seg = wg / groups;
      group = seg < segs ? wg - seg * groups : groups;  // (none left for it)
    }
  }
  s.row = (group << pg) + (t >> lg);
  s.row_step = (groups < n_wg ? groups : n_wg) << pg;
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

}  // namespace jac
}  // namespace chm
