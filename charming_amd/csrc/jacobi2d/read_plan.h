// The pieces in which a grid goes to the host through pinned buffers.
#pragma once
#include <stddef.h>

namespace chm {
namespace jac {

// Bytes of a piece, at most (and of each of the two pinned buffers).
constexpr size_t kReadBytes = 1 << 20;

// Pieces of n_rows rows of n_cols doubles: whole rows, or parts of one where
// a row is longer than a piece, so that no grid takes more pinned memory (two
// whole rows of a grid 2^30 wide would be 17 GB).
struct ReadPlan {
  int rows, cols;  // of a piece, less at the ends
  int n_rows, n_cols, per_row, n;
  int row(int k) const { return k / per_row * rows; }
  int col(int k) const { return k % per_row * cols; }
  int rows_of(int k) const {
    return n_rows - row(k) < rows ? n_rows - row(k) : rows;
  }
  int cols_of(int k) const {
    return n_cols - col(k) < cols ? n_cols - col(k) : cols;
  }
  size_t first(int k) const { return (size_t)row(k) * n_cols + col(k); }
};
inline ReadPlan read_plan(int n_rows, int n_cols) {
  constexpr int kCells = (int)(kReadBytes / sizeof(double));
  ReadPlan p;
  p.n_rows = n_rows;
  p.n_cols = n_cols;
  p.cols = n_cols < kCells ? n_cols : kCells;
  p.rows = kCells / p.cols < n_rows ? kCells / p.cols : n_rows;
  if (p.cols < n_cols) p.rows = 1;
  p.per_row = (n_cols + p.cols - 1) / p.cols;
  p.n = (n_rows + p.rows - 1) / p.rows * p.per_row;
  return p;
}

}  // namespace jac
}  // namespace chm
