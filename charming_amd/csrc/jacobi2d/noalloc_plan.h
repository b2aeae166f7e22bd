// The launches of a no-alloc solve, as counts: a list of them would grow with
// the sweeps (8 GB for 2^31 single sweeps of a low grid) and could throw
// across the C entry.
#pragma once

namespace chm {
namespace jac {

// Sweeps per launch of `iters` >= 1 sweeps whose last one is a launch of its
// own (it leaves u_{iters-1} for the residual): sixteen, then what is left in
// fours, then single sweeps.  An even number of launches ends in the array
// it began in, so of an odd one a pass is split, which costs less than the
// copy back.  Grids lower than sixteen rows are swept one at a time (a pass
// needs the ring's rows that far apart).
struct NoallocPlan {
  int n;         // launches
  int head;      // 12 and 4 come first (2) or nothing (0)
  int full;      // then so many of sixteen
  int tail[2];   // then these, where not zero
  int operator[](int i) const {
    if (i < head) return i == 0 ? 12 : 4;
    i -= head;
    if (i < full) return 16;
    i -= full;
    return i < 2 && tail[i] > 0 ? tail[i] : 1;
  }
};

inline NoallocPlan noalloc_plan(int H, int iters) {
  NoallocPlan p = {0, 0, 0, {0, 0}};
  const int left = iters - 1;
  if (H >= 16) {
    p.full = left / 16;
    p.tail[0] = left % 16 / 4 * 4;
  }
  const int singles = left - 16 * p.full - p.tail[0] + 1;
  p.n = p.full + (p.tail[0] > 0) + singles;
  if (p.n % 2 && p.tail[0] > 4) {
    p.tail[0] -= 4;
    p.tail[1] = 4;
    p.n++;
  } else if (p.n % 2 && p.full > 0) {
    p.full--;
    p.n++;
    if (p.tail[0] > 0) {
      p.head = 2;
    } else {
      p.tail[0] = 12;
      p.tail[1] = 4;
    }
  }
  return p;
}

}  // namespace jac
}  // namespace chm
