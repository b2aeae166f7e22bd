// Tile sides of engines whose rounds run as groups of waves (512-thread
// workgroups), where the caller gives none: what a window of 9, 5 or 3 columns
// per lane leaves after sixteen sweeps, and half of the first for little work.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "chm_jacobi2d.h"

namespace chm {
namespace eng {

// A side, and the time of a tile's round in us on a card with little else to
// do.  The rules below compare such times with each other, so that their
// ratios count: 5.7 : 2.4 : 1.3 : 1 with a task's 8 us; with every CU busy the
// rounds take 440, 169, 88 and 68 us, 6.4 : 2.5 : 1.3 : 1.
constexpr int kPipeSides[] = {544, 288, 160, 96};
constexpr double kPipeTimes[] = {300, 120, 61, 46};
constexpr int kBatchSides = 4;  // those a batch's problems may get
constexpr int kServeSides = 4;  // those a request may get

// A round of a tile of level l in us, of a problem `height` rows high (a
// partial tile takes its share of the steps; a task costs about 8 us besides).
inline double pipe_tile_us(int height, int l) {
  const int side = kPipeSides[l];
  const double h = std::min(height, side);
  return kPipeTimes[l] * (h / 2 + 38) / (side / 2 + 38) + 8;
}

// Tile sides of a batch for an engine of groups of waves (blocks[i], those
// not given already): the largest side costs least per cell (on a busy card
// 1.5 ns a cell and round at 544, 2.0 at 288, 3.4 at 160, 7.4 at 96), but a
// problem's rounds follow each other, so the one whose rounds take longest is
// cut finer while that is longer than the whole batch's work spread over the
// workgroups.  Where a problem with a tolerance stops is not known: each counts
// as many rounds as the one with the highest cap (by its own cap, one of 100
// sweeps was left in tiles of 544 beside one of 400, and where both stopped
// after 4 its two rounds with exact residuals were all the time: 6 problems of
// up to 1187 to 0.1 took 2.66 ms, 0.47 with the caps taken as equal).
inline void pick_blocks(const chm_batch_problem* probs, int n, int n_wg,
                        int64_t max_tiles, std::vector<int>& blocks) {
  struct Item {
    double latency;
    int i, level;
    bool operator<(const Item& o) const { return latency < o.latency; }
  };
  int tol_iters = 0;
  for (int i = 0; i < n; i++)
    if (probs[i].tol > 0) tol_iters = std::max(tol_iters, probs[i].iters);
  auto rounds = [&](int i) {
    return (double)(((probs[i].tol > 0 ? tol_iters : probs[i].iters) + 15) / 16);
  };
  auto tiles = [&](int i, int side) {
    return (double)((probs[i].width + side - 1) / side) *
           ((probs[i].height + side - 1) / side);
  };
  auto tile_us = [&](int i, int l) { return pipe_tile_us(probs[i].height, l); };
  double work = 0;  // us over all workgroups
  std::vector<Item> heap;
  for (int i = 0; i < n; i++) {
    if (blocks[i] > 0) {
      work += rounds(i) * tiles(i, blocks[i]) * 60;
      continue;
    }
    int l = 0;  // no side beyond the next one that holds the problem
    const int side = std::max(probs[i].width, probs[i].height);
    while (l + 1 < kBatchSides && side <= kPipeSides[l + 1]) l++;
    blocks[i] = kPipeSides[l];
    work += rounds(i) * tiles(i, kPipeSides[l]) * tile_us(i, l);
    heap.push_back({rounds(i) * tile_us(i, l), i, l});
  }
  std::make_heap(heap.begin(), heap.end());
  while (!heap.empty() && heap.front().latency > work / n_wg) {
    std::pop_heap(heap.begin(), heap.end());
    Item t = heap.back();
    heap.pop_back();
    if (t.level + 1 >= kBatchSides ||
        tiles(t.i, kPipeSides[t.level + 1]) >= (double)max_tiles)
      break;  // cannot get shorter
    const double was = rounds(t.i) * tiles(t.i, kPipeSides[t.level]) *
                       tile_us(t.i, t.level);
    t.level++;
    blocks[t.i] = kPipeSides[t.level];
    work += rounds(t.i) * tiles(t.i, kPipeSides[t.level]) *
                tile_us(t.i, t.level) - was;
    t.latency = rounds(t.i) * tile_us(t.i, t.level);
    heap.push_back(t);
    std::push_heap(heap.begin(), heap.end());
  }
}

// Tile side of a served request: a finer one where it at least halves the
// round on this request's share of the workgroups.  It costs 1.4 to 2.1 times
// as much per cell, which requests that arrive beside this one would miss.
// (The factor of two was set on one workload, a burst of 24 requests of
// 256..8192 per side, and others were not tried.)
inline int serve_block_pipe(int W, int H, int n_wg, int resident,
                            int64_t max_tiles) {
  const int64_t share = std::max<int64_t>(1, n_wg / (1 + resident));
  int best = kPipeSides[0];
  double t_best = 0;
  for (int l = 0; l < kServeSides; l++) {
    const int bs = kPipeSides[l];
    const int64_t tiles = (int64_t)((W + bs - 1) / bs) * ((H + bs - 1) / bs);
    if (l > 0 && tiles >= max_tiles) break;
    const double t =
        (double)((tiles + share - 1) / share) * pipe_tile_us(H, l);
    if (l == 0 || 2 * t <= t_best) {
      best = bs;
      t_best = t;
    }
  }
  return best;
}

}  // namespace eng
}  // namespace chm
