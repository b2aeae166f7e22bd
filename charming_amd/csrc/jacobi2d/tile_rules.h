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

constexpr int kBatchSides = 4;
constexpr int kBatchSide[kBatchSides] = {544, 288, 160, 96};
constexpr int kServeSides = 6;
constexpr int kServeSide[kServeSides] = {544, 288, 192, 160, 96, 64};

// The time of a tile's round in us, a task's 8 beside it.  The rules below
// compare such times with each other, so that their ratios count.  A batch's
// are of rounds of sixteen alone on a card, 5.7 : 2.4 : 1.3 : 1 (with every CU
// busy 440, 169, 88 and 68 us, 6.4 : 2.5 : 1.3 : 1); a request's are those of
// lone requests to a tolerance of 17 rounds, less what its tiles cost once.
constexpr double kBatchTimes[kBatchSides] = {300, 120, 61, 46};
constexpr double kServeTimes[kServeSides] = {337, 130, 93, 69, 49, 42};

// A round of a tile of `side` (a full one takes `us`) of a problem `height`
// rows high: a partial tile takes its share of the steps.
inline double pipe_tile_us(double us, int side, int height) {
  const double h = std::min(height, side);
  return us * (h / 2 + 38) / (side / 2 + 38) + 8;
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
  auto tile_us = [&](int i, int l) {
    return pipe_tile_us(kBatchTimes[l], kBatchSide[l], probs[i].height);
  };
  double work = 0;  // us over all workgroups
  std::vector<Item> heap;
  for (int i = 0; i < n; i++) {
    if (blocks[i] > 0) {
      work += rounds(i) * tiles(i, blocks[i]) * 60;
      continue;
    }
    int l = 0;  // no side beyond the next one that holds the problem
    const int side = std::max(probs[i].width, probs[i].height);
    while (l + 1 < kBatchSides && side <= kBatchSide[l + 1]) l++;
    blocks[i] = kBatchSide[l];
    work += rounds(i) * tiles(i, kBatchSide[l]) * tile_us(i, l);
    heap.push_back({rounds(i) * tile_us(i, l), i, l});
  }
  std::make_heap(heap.begin(), heap.end());
  while (!heap.empty() && heap.front().latency > work / n_wg) {
    std::pop_heap(heap.begin(), heap.end());
    Item t = heap.back();
    heap.pop_back();
    if (t.level + 1 >= kBatchSides ||
        tiles(t.i, kBatchSide[t.level + 1]) >= (double)max_tiles)
      break;  // cannot get shorter
    const double was = rounds(t.i) * tiles(t.i, kBatchSide[t.level]) *
                       tile_us(t.i, t.level);
    t.level++;
    blocks[t.i] = kBatchSide[t.level];
    work += rounds(t.i) * tiles(t.i, kBatchSide[t.level]) *
                tile_us(t.i, t.level) - was;
    t.latency = rounds(t.i) * tile_us(t.i, t.level);
    heap.push_back(t);
    std::push_heap(heap.begin(), heap.end());
  }
}

// The same for a request of `iters` sweeps, with its share of what a tile takes
// once: to be seeded and hashed and for the sums of exact residuals, 4.9 ns a
// cell (of one sweep, 11 requests of 500 x 500 took 0.53 ms in tiles of 288, now
// 0.32 in tiles of 64, 96 and 192).
inline double serve_tile_us(int l, int W, int H, int iters) {
  const int side = kServeSide[l], rounds = (iters + 15) / 16;
  return pipe_tile_us(kServeTimes[l], side, H) +
         4.9e-3 * std::min(W, side) * std::min(H, side) / std::max(1, rounds);
}

// The workgroup time of a round of the request: its tiles, those at its right
// and lower edge in their own sizes (a row of a window costs by the columns per
// lane that hold it, 3, 5 or 9).
inline double serve_request_us(int l, int W, int H, int iters) {
  const int side = kServeSide[l], rounds = std::max(1, (iters + 15) / 16);
  auto step = [](int w) { return w <= 160 ? 0.585 : w <= 288 ? 0.71 : 1.09; };
  // all columns' steps of one row of the request, and all rows' of one column
  const int cw = W / side, rw = W % side, ch = H / side, rh = H % side;
  const double row = cw * step(side) + (rw ? step(rw) : 0);
  const double col = ch * (side / 2.0 + 38) + (rh ? rh / 2.0 + 38 : 0);
  return row * col + 8.0 * (cw + (rw > 0)) * (ch + (rh > 0)) +
         4.9e-3 * W * H / rounds;
}

// What a server's resident requests take of the card.
struct ServeLoad {
  int requests = 0;
  int64_t tiles = 0;  // tasks of a round of all of them
  double us = 0;      // workgroup time of such a round
};

// What a request in `tiles` tiles of side bs adds to it.
inline double serve_round_us(int W, int H, int iters, int64_t tiles, int bs) {
  int l = 0;
  while (l + 1 < kServeSides && kServeSide[l] > bs) l++;
  return tiles * serve_tile_us(l, W, H, iters);
}

inline double clamp01(double v) { return std::min(1.0, std::max(0.0, v)); }

// Tile side of a served request: the one whose round costs least, in time of
// - the request: a tile's, or what all residents' tiles take of the card if
//   that is more (5 % more, by their waits for each other);
// - a third of a tile's where the card has no room for another such request
//   beside it, but is not overfilled many times: the last tiles then wait for
//   a turn of their own;
// - the residents, whom the request delays by the card time it takes (partial
//   tiles at their own sizes: counted full, a request a little wider than 544
//   went to tiles of 288, 250.9 requests a second of a saturated stream, now
//   253.9): three times that as the card fills from half on, and six more as it
//   fills once more, for the requests that such a load brings besides (of more
//   than sixteen residents sixteen count);
// - requests to come: three fifths of that card time.
// A finer side is over sooner where the card has room for its tiles, but costs
// 1.4 to 2.1 times as much per cell.  Ms of requests of 300 x 300 x 200 to a
// tolerance, alone, 6 and 20 at once: 0.90, 0.98, 1.57 (by each request's share
// of the workgroups, and a finer side only where it halved the round: 1.43,
// 1.44, 1.49; by the window pass: 1.13, 1.24, 2.22); of 2000 x 2000 x 200
// alone: 1.95 (2.81; 2.37).  Of 42 bursts of 1..24 drawn requests of up to 7956
// per side the weights leave none more than 2 % behind the share rule, and take
// 0.84 of its time on average; with a residents' weight of 1 and 3, 0.81, but
// one was 8 % behind.  Requests of one size submitted at once are where the
// greedy choice costs: the first take tiles that the next have no room beside.
// Of 80 bursts of 1 to 20 such the rule takes 0.83 of the share rule's time, but
// 30 are more than 3 % slower (2 of 959 x 959 x 12: 292 us, 182 in tiles of 96).
inline int serve_block_pipe(int W, int H, int iters, int n_wg,
                            const ServeLoad& load, int64_t max_tiles) {
  int best = kServeSide[0];
  double least = 0;
  for (int l = 0; l < kServeSides; l++) {
    const int bs = kServeSide[l];
    const int64_t tiles = (int64_t)((W + bs - 1) / bs) * ((H + bs - 1) / bs);
    if (l > 0 && tiles >= max_tiles) break;
    const double us = serve_tile_us(l, W, H, iters);
    const double card = tiles * us / n_wg;
    const double delay = serve_request_us(l, W, H, iters) / n_wg;
    const double full = (double)(load.tiles + tiles) / n_wg;
    const double twice = (double)(load.tiles + 2 * tiles) / n_wg;
    const double cost =
        std::max(us, 1.05 * (load.us / n_wg + card)) + 0.6 * card +
        clamp01(10 * twice - 9.5) * clamp01(2.5 - twice) * 0.35 * us +
        (3 * clamp01(2 * full - 1) + 6 * clamp01(2 * full - 2)) *
            std::min(load.requests, 16) * delay;
    if (l == 0 || cost < least) {
      best = bs;
      least = cost;
    }
  }
  return best;
}

}  // namespace eng
}  // namespace chm
