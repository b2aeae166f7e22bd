// Internal (host + device) declarations shared by the Jacobi2D translation
// units: the problem handle and the device kernels every form reuses.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "../common/status.h"
#include "chm_jacobi2d.h"
#include "stencil.h"

namespace chm {
namespace jac {

// Chare geometry of the decomposed forms: chare (r, c) covers interior rows
// [row0, row0 + bh) and columns [col0, col0 + bw) (1-based); equal blocks
// with the last row/column of chares taking the remainder.
struct ChareGeom {
  int row0, col0, bh, bw;
};

__host__ __device__ inline void split_extent(int len, int n, int r, int* start,
                                             int* size) {
  int b = len / n;
  *start = r * b;
  *size = (r == n - 1) ? len - b * (n - 1) : b;
}

// Workgroup-collective: the sum of every thread's v, in thread 0.
__device__ inline uint64_t block_sum(uint64_t v) {
  __shared__ uint64_t part[16];
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_down(v, off, 64);
  if (__lane_id() == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x / 64); w++) v += part[w];
  return v;
}

struct PersistentState;  // defined by the message-driven form

// Two pinned buffers through which a grid goes to the host, made at the first
// read and kept with the problem.
struct GridReader {
  std::mutex mu;  // reads of one problem by several threads take turns
  double* buf[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
};

struct Handle {
  chm_jacobi_problem prob;
  int form;
  int W, H;
  int64_t P;         // pitch of the global array (plain forms)
  double* grid[2];   // plain forms: u_k lives in grid[cur]
  int cur;
  hipStream_t stream;
  hipEvent_t ev0, ev1;
  uint64_t* d_acc;   // 4 x u64 scratch: hash, residual lo/hi
  chm_jacobi_tuning tune;
  // graph form
  hipGraphExec_t gexec;
  int graph_iters;
  // persistent form
  PersistentState* ps;
  GridReader* reader;
};

// Launches, on the problem's stream, what writes rows [row, row + rows) x
// columns [col, col + cols) of the grid, ring included, to `dst` (cols cells
// a row).
void persistent_gather(Handle* h, double* dst, int row, int rows, int col,
                       int cols);

// Forms implemented in other translation units.
int persistent_create(Handle* h);
int persistent_reset(Handle* h);
int persistent_solve(Handle* h, chm_jacobi_result* res);
int persistent_hash_region(Handle* h, int r0, int r1, int c0, int c1,
                           uint64_t* hash);
int persistent_phase_stats(Handle* h, double* out);
int persistent_chare_phases(Handle* h, double* out);
int persistent_chare_count(Handle* h, int* n);
void persistent_destroy(Handle* h);

}  // namespace jac
}  // namespace chm
