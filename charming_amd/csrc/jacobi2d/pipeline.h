// Deep fused sweeps of a block by groups of four waves: the sweeps of a pass
// are spread over the waves of a group, which hand rows on through LDS.
//
// The window pass of stencil.h (sweep_panelD) holds all D sweeps of a
// 128-column window in one wave, so a row of the window costs each lane two
// cells per sweep: 4 of its 14 vector operations shift lanes, and 32 of the
// 128 columns are margin that a neighbouring window computes too.  Here wave
// r of a group makes sweeps r * NST + 1 .. (r + 1) * NST of a window of
// 64 * K columns (K = 3, 5 or 9 columns per lane).  A quarter of the
// sweeps leaves a wave the registers for rows 4.5 times as wide: 4 of 49
// operations shift lanes, 32 of 576 columns are margin, and a block of
// 1024 x 1024 is two windows of full height (no bands, each of which fills
// its pipeline anew).
//
// Per sweep a wave keeps two rows: c, the newest row of the sweep's input,
// and p, the sum (c + W) + E + N of the row before it, which waits for its
// south neighbour.  When a row S arrives,
//   out = (p + S) * 0.2;  p = S + W + E + c;  c = S
// (the operand order of the single sweep, so every grid is bit-identical).
// `out` is written over c, whose row just died, and is the S of the next
// sweep: the row sets rotate through the sweeps, no row is copied, and the
// step loop is unrolled by the number of sets.
//
// Wave 0 streams the input rows into LDS with kPipeRing rows in flight
// (global_load_lds: no registers are held); each link between two waves
// holds kPipeLink rows; the last wave stores a row as whole 16-byte pairs
// after turning it through LDS.  Waves wait for each other on LDS counters
// (rows made / rows used), not on workgroup barriers.
//
// What bounds it: 1024 x 1024 blocks on all 256 CUs take 1.13-1.17 ms per
// sixteen sweeps (3700-3790 Gcell/s) against 1.56-1.60 ms with sweep_panelD
// on the same card.  The vector ALU alone would need 0.69 ms at 2.4 GHz and
// memory 0.93 ms (the same pass without arithmetic); with both busy the card
// holds the clock at 1.95-2.05 GHz.  64 blocks of 512 x 512 (2.4 GHz): 263 us
// against 567; 256 of 256 x 256 (K = 5): 116 against 230; of 128 x 128
// (K = 3): 57 against 113.
// Measured and not kept (ms per sixteen sweeps of 1024 x 1024): a workgroup
// barrier per row instead of the LDS counters 1.28, three or four input rows
// 1.3-1.6, equal wave priorities 1.20 (see step()), priorities by which group
// is ahead 1.21, the groups' operations in the compiler's order 1.20.
#pragma once
#include "stencil.h"

namespace chm {
namespace jac {

typedef __attribute__((address_space(3))) double ldouble;
typedef double lpair __attribute__((ext_vector_type(2), aligned(16)));
typedef __attribute__((address_space(3))) lpair llpair;
typedef __attribute__((address_space(1))) const char gcchar;

constexpr int kPipeWaves = 4;  // waves of a group
constexpr int kPipeRing = 6;   // input rows in LDS
constexpr int kPipeLink = 2;   // rows between two waves
constexpr int kPipeMaxK = 9;   // columns per lane of the widest window
constexpr int kNoRing = 1 << 29;

// Wave-uniform copies in scalar registers.
__device__ inline int suni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int64_t suni(int64_t v) {
  const uint64_t u = (uint64_t)v;
  return (int64_t)(((uint64_t)(uint32_t)suni((int)(u >> 32)) << 32) |
                   (uint32_t)suni((int)(uint32_t)u));
}
template <class T>
__device__ inline T* suni(T* p) {
  return (T*)suni((int64_t)p);
}

// One window of a block: columns [w0, w0 + 64 K), of which [oc0, oc1) are
// written, rows [r0, r1).
struct PipeJob {
  const double* in;
  double* out;
  double* sum;         // FP64 sum of the last sweep's squared changes (or null)
  int64_t pitch;
  int w0, oc0, oc1;
  int r0, r1;
  int lo_col, hi_col;  // columns of `in` that may be read (odd .. any)
  int lo_row, hi_row;  // rows of `in` that may be read
  int top, bottom;     // rows that keep their values (kNoRing: none)
  int left, right;     // columns that keep their values (kNoRing: none)
  double ring;         // west of lane 0's columns and east of lane 63's
};

// LDS of a group (sized for the widest window).
struct alignas(128) PipeLds {
  double edge[2 * 64 * kPipeMaxK];  // the grid's ring rows above and below
  double ring[kPipeRing * 64 * kPipeMaxK];
  double link[(kPipeWaves - 1) * kPipeLink * 64 * kPipeMaxK];
  double row[64 * kPipeMaxK + 64];
  int made[kPipeWaves], used[kPipeWaves];  // rows of link i made / used
  PipeJob job;
};

// ---------------------------------------------------------------------------
// a block's windows
// ---------------------------------------------------------------------------
// A block [c0, c1) (c0 odd) of columns whose input reaches `d` columns past
// either side, or to the grid's ring column `left` (even) or `right` if that
// is nearer.  Windows start on odd columns (16-byte pairs).  `flat`: the
// ring's columns hold one value, which then need not be in a window: the lane
// shifts hand it to the end lanes (of a window that starts on left + 1, or
// ends on right - 1).  Else, and where right - 1 cannot be lane 63's last
// column, a ring column is in the window and its cells keep their values.
struct PipeCols {
  int c0, c1, left, right;
  bool flat;
};
struct PipeSplit {
  int n, first, stride, hi, win;
  bool ring_l, ring_r;
};
__host__ __device__ inline PipeSplit pipe_split(const PipeCols& b, int d,
                                                int k) {
  PipeSplit s;
  s.win = 64 * k;
  s.stride = s.win - 2 * d;
  s.ring_l = b.left >= b.c0 - d && b.left != kNoRing;
  s.ring_r = b.right < b.c1 + d;
  const int lo = s.ring_l ? b.left + (b.flat ? 1 : 0) : b.c0 - d;
  s.first = (lo & 1) ? lo : lo - 1;
  s.hi = s.ring_r ? b.right - (b.flat && (b.right & 1) ? 1 : 0) : b.c1 - 1 + d;
  const int over = s.hi - s.first + 1 - s.win;
  s.n = over <= 0 ? 1 : 1 + (over + s.stride - 1) / s.stride;
  return s;
}
// Columns per lane for a block: the fewest columns swept in all (a step has
// a fixed part of about two columns per lane).
__host__ __device__ inline int pipe_pick_k(const PipeCols& b, int d) {
  int best = 9, cost = 1 << 30;
  for (int k = 9; k >= 3; k -= (k == 9 ? 4 : 2)) {
    const int c = pipe_split(b, d, k).n * (k + 2);
    if (c < cost) {
      cost = c;
      best = k;
    }
  }
  return best;
}
// Window i of the block: fills the column fields of the job; returns which
// of the lanes' columns may be ring columns: 0 none, 2 lane 63's last one,
// 3 any.
__host__ __device__ inline int pipe_window(const PipeSplit& s, int i,
                                           const PipeCols& b, int d,
                                           PipeJob* j) {
  int w0 = s.first + i * s.stride;
  const bool last = i == s.n - 1;
  // the right ring column (or the last one before it) ends the last window
  const bool ends = last && s.ring_r && b.flat && (s.n > 1 || !s.ring_l);
  if (ends) w0 = s.hi + 1 - s.win;
  j->w0 = w0;
  j->oc0 = i == 0 ? b.c0 : s.first + i * s.stride + d;
  j->oc1 = last ? b.c1 : min(b.c1, s.first + (i + 1) * s.stride + d);
  j->left = s.ring_l && i == 0 && !b.flat ? b.left : kNoRing;
  j->right = s.ring_r && last && w0 + s.win > b.right ? b.right : kNoRing;
  if (j->left == kNoRing && j->right == kNoRing) return 0;
  return ends ? 2 : 3;
}

// ---------------------------------------------------------------------------
// pieces of a step (every lane of the wave active)
// ---------------------------------------------------------------------------
// c = t * 0.2 in the lanes of m: a masked multiply leaves the ring's cells
// as they are without a select (two scalar moves instead of two vector
// selects per cell, and no control flow for the register allocator).
__device__ inline void mul_masked(double& c, double t, uint64_t m) {
  asm("s_mov_b64 exec, %2\n\tv_mul_f64 %0, %1, %3\n\ts_mov_b64 exec, -1"
      : "+v"(c)
      : "v"(t), "s"(m), "s"(0.2));
}
// acc += d * d in the lanes of m
__device__ inline void add_sq_masked(double& acc, double d, uint64_t m) {
  asm("s_mov_b64 exec, %2\n\tv_fma_f64 %0, %1, %1, %0\n\ts_mov_b64 exec, -1"
      : "+v"(acc)
      : "v"(d), "s"(m));
}
// w = lane l-1's v, e = lane l+1's v; lane 0 keeps its w and lane 63 its e.
__device__ inline void shift_in(double& w, double& e, double v_last,
                                double v_first) {
  const long long a = __double_as_longlong(v_last), b = __double_as_longlong(v_first);
  const long long ow = __double_as_longlong(w), oe = __double_as_longlong(e);
  const int wl = __builtin_amdgcn_update_dpp((int)ow, (int)a, 0x138, 0xf, 0xf, false);
  const int wh = __builtin_amdgcn_update_dpp((int)(ow >> 32), (int)(a >> 32), 0x138, 0xf, 0xf, false);
  const int el = __builtin_amdgcn_update_dpp((int)oe, (int)b, 0x130, 0xf, 0xf, false);
  const int eh = __builtin_amdgcn_update_dpp((int)(oe >> 32), (int)(b >> 32), 0x130, 0xf, 0xf, false);
  w = __longlong_as_double(((long long)wh << 32) | (unsigned)wl);
  e = __longlong_as_double(((long long)eh << 32) | (unsigned)el);
}
template <int N>
__device__ inline void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until the LDS word at byte address a is at least `need`; `known` is
// the last value seen of it (the words only grow).  In one block of assembly
// so the loop is no control flow of the step.
__device__ inline void lds_wait_ge(int a, int need, int& known) {
  int t;
  asm volatile(
      "s_cmp_ge_i32 %0, %2\n\t"
      "s_cbranch_scc1 2f\n"
      "1:\n\t"
      "v_mov_b32 %1, %3\n\t"
      "ds_read_b32 %1, %1\n\t"
      "s_waitcnt lgkmcnt(0)\n\t"
      "v_readfirstlane_b32 %0, %1\n\t"
      "s_cmp_lt_i32 %0, %2\n\t"
      "s_cbranch_scc1 1b\n"
      "2:"
      : "+s"(known), "=&v"(t)
      : "s"(need), "s"(a)
      : "memory", "scc");
  known = suni(known);
}
// One lane stores v to the LDS word at byte address a (after the wave's
// earlier LDS accesses: LDS executes them in order).
__device__ inline void lds_post(int a, int v) {
  int x, y;
  asm volatile(
      "s_mov_b64 exec, 1\n\tv_mov_b32 %0, %2\n\tv_mov_b32 %1, %3\n\t"
      "ds_write_b32 %0, %1\n\ts_mov_b64 exec, -1"
      : "=&v"(x), "=&v"(y)
      : "s"(a), "s"(v)
      : "memory");
}
// Streaming stores by the lanes of m at byte offset o from p (the s_nop: the
// store reads its data up to two cycles after it issues).
__device__ inline void store_masked(gdouble* p, int o, lpair v, uint64_t m) {
  asm volatile(
      "s_mov_b64 exec, %3\n\tglobal_store_dwordx4 %0, %1, %2 nt\n\t"
      "s_mov_b64 exec, -1\n\ts_nop 1" ::"v"(o),
      "v"(v), "s"(p), "s"(m)
      : "memory");
}
__device__ inline void store_masked(gdouble* p, int o, double v, uint64_t m) {
  asm volatile(
      "s_mov_b64 exec, %3\n\tglobal_store_dwordx2 %0, %1, %2 nt\n\t"
      "s_mov_b64 exec, -1\n\ts_nop 1" ::"v"(o),
      "v"(v), "s"(p), "s"(m)
      : "memory");
}
// 16 bytes per lane of m from p + o to the LDS bytes lds + 16 * lane.
__device__ inline void fetch_masked(gcchar* p, int o, int lds, uint64_t m) {
  asm volatile(
      "s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\t"
      "global_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(o),
      "s"(p), "s"(lds), "s"(m)
      : "memory");
}

// c = the K doubles at LDS byte address base + at, if row == ring_row.  In
// one block of assembly, loads and wait included: a branch in the step would
// cost the register allocator copies and spills of the row sets.
template <int K>
__device__ inline void take_ring_row(double* c, int row, int ring_row, int at,
                                     int base) {
  int t;
#define CHM_HEAD "s_cmp_lg_i32 %[q], %[r]\n\ts_cbranch_scc1 1f\n\tv_add_u32 %[t], %[b], %[a]\n\t"
#define CHM_LD(N, O) "ds_read_b64 %" #N ", %[t] offset:" #O "\n\t"
#define CHM_TAIL "s_waitcnt lgkmcnt(0)\n1:"
#define CHM_IN [q] "s"(row), [r] "s"(ring_row), [a] "s"(at), [b] "v"(base)
  if constexpr (K == 3)
    asm(CHM_HEAD CHM_LD(0, 0) CHM_LD(1, 8) CHM_LD(2, 16) CHM_TAIL
                 : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), [t] "=&v"(t)
                 : CHM_IN
                 : "scc");
  else if constexpr (K == 5)
    asm(CHM_HEAD CHM_LD(0, 0) CHM_LD(1, 8) CHM_LD(2, 16) CHM_LD(3, 24)
                     CHM_LD(4, 32) CHM_TAIL
                 : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]), "+v"(c[4]),
                   [t] "=&v"(t)
                 : CHM_IN
                 : "scc");
  else
    asm(CHM_HEAD CHM_LD(0, 0) CHM_LD(1, 8) CHM_LD(2, 16) CHM_LD(3, 24)
                     CHM_LD(4, 32) CHM_LD(5, 40) CHM_LD(6, 48) CHM_LD(7, 56)
                         CHM_LD(8, 64) CHM_TAIL
                 : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]), "+v"(c[4]),
                   "+v"(c[5]), "+v"(c[6]), "+v"(c[7]), "+v"(c[8]), [t] "=&v"(t)
                 : CHM_IN
                 : "scc");
#undef CHM_HEAD
#undef CHM_LD
#undef CHM_TAIL
#undef CHM_IN
}

// ---------------------------------------------------------------------------
// one wave of a group
// ---------------------------------------------------------------------------
enum { PIPE_FIRST = 0, PIPE_MIDDLE = 1, PIPE_LAST = 2 };

// Sweeps role * NST + 1 .. (role + 1) * NST of the group's window (job in
// LDS).  COLS: the lanes' columns that may be ring columns (pipe_window).
// SUM (last wave): the FP64 sum of the
// last sweep's squared changes over the cells written is added to *job.sum.
// T only gives callers of one workgroup size a copy compiled for their
// register budget.
template <int T, int K, int NST, int COLS, int KIND, bool SUM>
__device__ __noinline__ void pipe_wave(int role, int lds_off) {
  constexpr int NS = NST + 2;  // row sets: NST, the row in, the row prefetched
  constexpr int D = kPipeWaves * NST;
  constexpr int ROW = 64 * K;
  constexpr int ROWB = ROW * (int)sizeof(double);
  role = suni(role);
  lds_off = suni(lds_off);
  typedef __attribute__((address_space(3))) PipeLds lPipeLds;
  typedef __attribute__((address_space(3))) const PipeJob lPipeJob;
  const lPipeLds* ld = (const lPipeLds*)(uintptr_t)(uint32_t)lds_off;
  lPipeJob* jp = &ld->job;
  const double* in = suni(jp->in);
  gdouble* out = (gdouble*)suni(jp->out);
  const int64_t pitch = suni(jp->pitch);
  const int w0 = suni(jp->w0), oc0 = suni(jp->oc0), oc1 = suni(jp->oc1);
  const int r0 = suni(jp->r0), r1 = suni(jp->r1);
  const int top = suni(jp->top), bottom = suni(jp->bottom);
  const int lane = __lane_id();
  // every input row, one more step for the last wave's deferred store, in
  // whole turns of the row sets
  const int n_steps = (r1 - r0 + 2 * D + 1 + NS - 1) / NS * NS;
  auto at = [&](size_t member) {
    return (ldouble*)(uintptr_t)(uint32_t)(lds_off + (int)member);
  };
  ldouble* ring = at(offsetof(PipeLds, ring));
  ldouble* links = at(offsetof(PipeLds, link));
  ldouble* row = at(offsetof(PipeLds, row));
  const int in_made = lds_off + (int)offsetof(PipeLds, made) + 4 * (role - 1);
  const int in_used = lds_off + (int)offsetof(PipeLds, used) + 4 * (role - 1);
  const int out_made = in_made + 4, out_used = in_used + 4;

  double p[NST][K], c[NS][K];
#pragma unroll
  for (int s = 0; s < NST; s++)
#pragma unroll
    for (int j = 0; j < K; j++) p[s][j] = 0;
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int j = 0; j < K; j++) c[s][j] = 0;

  // lanes whose column j takes new values
  const int col = w0 + K * lane;
  uint64_t keep[K];
  {
    const int left = suni(jp->left), right = suni(jp->right);
#pragma unroll
    for (int j = 0; j < K; j++)
      keep[j] = __ballot(!(col + j == left || col + j == right));
  }

  // a row in pieces of 128 columns, a pair per lane (the last one half a
  // piece for odd K)
  constexpr int NP = (K + 1) / 2;
  auto piece = [](int m) { return 2 * m + 1 < K ? ~0ull : 0xffffffffull; };
  // FIRST: byte offsets of this lane's pairs in an input row (pairs past the
  // columns that may be read take others: nothing depends on them)
  int goff[NP];
  if (KIND == PIPE_FIRST) {
    const int lo = suni(jp->lo_col), hi = suni(jp->hi_col);
#pragma unroll
    for (int m = 0; m < NP; m++) {
      const int cc = min(w0 + 128 * m + 2 * lane, hi - ((hi & 1) ^ 1));
      goff[m] = (kColOff + max(lo, cc)) * (int)sizeof(double);
    }
  }
  const int lo_row = suni(jp->lo_row), hi_row = suni(jp->hi_row);
  auto fetch_row = [&](int r, int to) {
    gcchar* rp = (gcchar*)(in + (int64_t)r * pitch);
#pragma unroll
    for (int m = 0; m < NP; m++)
      fetch_masked(rp, goff[m], lds_off + to + m * 1024, piece(m));
  };
  auto fetch = [&](int i, int slot) {
    fetch_row(max(lo_row, min(r0 - D + i, hi_row)),
              (int)offsetof(PipeLds, ring) + slot * ROWB);
  };
  ldouble* ring_r = ring + K * lane;
  ldouble* lin = links + (role - 1) * kPipeLink * ROW + 2 * lane;
  ldouble* lout = links + role * kPipeLink * ROW + 2 * lane;
  int k_made = 0, k_used = 0, slot_in = 0, slot_out = 0;
  // row i of this wave's input into d (rows in order)
  auto read_row = [&](double* d, int i) {
    if (KIND == PIPE_FIRST) {
      ldouble* rr = ring_r + slot_in * ROW;
#pragma unroll
      for (int j = 0; j < K; j++) d[j] = rr[j];
      slot_in = slot_in == kPipeRing - 1 ? 0 : slot_in + 1;
    } else {
      // (past the last row there is nothing to wait for or to use)
      lds_wait_ge(in_made, min(i + 1, n_steps), k_made);
      ldouble* src = lin + slot_in * ROW;
#pragma unroll
      for (int j = 0; j + 1 < K; j += 2) {
        const lpair v = *(const llpair*)(src + j * 64);
        d[j] = v.x;
        d[j + 1] = v.y;
      }
      if (K & 1) d[K - 1] = *(src + (K - 1) * 64 - lane);
      lds_post(in_used, i + 1);
      slot_in = slot_in == kPipeLink - 1 ? 0 : slot_in + 1;
    }
  };
  // LAST: the output row, turned through LDS
  ldouble* row_w = row + K * lane;
  ldouble* row_r = row + 2 * lane;
  uint64_t stm[NP], tail_m = 0;
  int tail = 0;
  uint64_t summ[K];
  double sum = 0.0;
  if (KIND == PIPE_LAST) {
#pragma unroll
    for (int m = 0; m < NP; m++) {
      const int cc = w0 + 128 * m + 2 * lane;
      stm[m] = __ballot(cc >= oc0 && cc + 1 < oc1) & piece(m);
    }
    tail_m = (oc1 - oc0) & 1;  // lane 0 stores the last column of an odd width
    tail = oc1 - 1 - w0;
    if (SUM) {
#pragma unroll
      for (int j = 0; j < K; j++)
        summ[j] = __ballot(col + j >= oc0 && col + j < oc1);
    }
  }
  if (KIND == PIPE_FIRST) {
    // (before the rows, so they are in when row 0 is)
    if (top != kNoRing) fetch_row(top, (int)offsetof(PipeLds, edge));
    if (bottom != kNoRing)
      fetch_row(bottom, (int)offsetof(PipeLds, edge) + ROWB);
#pragma unroll
    for (int f = 0; f < kPipeRing; f++) fetch(f, f);
    wait_vm<NP*(kPipeRing - 1)>();
  }
  read_row(c[0], 0);
  // row made by this wave's first sweep at step 0
  const int q0 = r0 - D - role * NST - 1;

  // the grid's ring row that the current turn may meet, where it lies in LDS
  // west of the lane's columns and east of them
  double wl = jp->ring, er = wl;
  int ring_row = kNoRing, ring_at = 0;
  const int edge_b = lds_off + (int)offsetof(PipeLds, edge) + 8 * K * lane;

  // One step: the wave's row n in, its row n out, the row sets rotated by u
  // places.  The wave's first half of a step runs at a higher priority:
  // two waves share a SIMD, and with equal priorities the older one took
  // all the issue slots it could, its group ran ahead and the other group
  // finished alone (1.20 -> 1.13-1.17 ms per sixteen sweeps of 1024 x 1024).
  auto step = [&](int u, int n) __attribute__((always_inline)) {
    const int e = (NS - u) % NS;
    __builtin_amdgcn_s_setprio(1);
    // pieces of a row in a share
    constexpr int NSH = NST > 1 ? NST - 1 : 1, PS = (NP + NSH - 1) / NSH;
    lpair hold[PS];
    double hold_t = 0;
    shift_in(wl, er, c[e][K - 1], c[e][0]);
#pragma unroll
    for (int s = 0; s < NST; s++) {
      double* S = c[(e + s) % NS];
      double* C = c[(e + s + 1) % NS];
      double* P = p[s];
      // three columns at a time, operations that depend on each other three
      // apart (a dependent FP64 operation waits 8 cycles, an independent one
      // issues after 5)
#pragma unroll
      for (int g = 0; g < K; g += 3) {
        double a[3], t[3];
#pragma unroll
        for (int x = 0; x < 3; x++)
          if (g + x < K) {
            const int j = g + x;
            a[x] = S[j] + (j ? S[j - 1] : wl);
            t[x] = P[j] + S[j];
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 3; x++)
          if (g + x < K) {
            const int j = g + x;
            a[x] = a[x] + (j < K - 1 ? S[j + 1] : er);
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 3; x++)
          if (g + x < K) P[g + x] = a[x] + C[g + x];
        __builtin_amdgcn_sched_barrier(0);
        double old[3];
        if (SUM && KIND == PIPE_LAST && s == NST - 1) {
#pragma unroll
          for (int x = 0; x < 3; x++)
            if (g + x < K) old[x] = C[g + x];
        }
#pragma unroll
        for (int x = 0; x < 3; x++)
          if (g + x < K) {
            const bool ring_j = COLS == 3 || (COLS == 2 && g + x == K - 1);
            if (ring_j)
              mul_masked(C[g + x], t[x], keep[g + x]);
            else
              C[g + x] = t[x] * 0.2;
          }
        if (SUM && KIND == PIPE_LAST && s == NST - 1) {
          const int orow = r0 - 2 * D + n;
          const uint64_t rm = (orow >= r0 && orow < r1) ? ~0ull : 0ull;
#pragma unroll
          for (int x = 0; x < 3; x++)
            if (g + x < K)
              add_sq_masked(sum, C[g + x] - old[x], summ[g + x] & rm);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      take_ring_row<K>(C, q0 + n - s, ring_row, ring_at, edge_b);
      if (s + 1 < NST) shift_in(wl, er, C[K - 1], C[0]);
      __builtin_amdgcn_sched_barrier(0);
      if (s == (NST - 1) / 2) __builtin_amdgcn_s_setprio(0);
      if (s == 0) {
        if (KIND == PIPE_FIRST) {
          // row n has been read: its slot takes row n + kPipeRing
          fetch(n + kPipeRing, slot_in == 0 ? kPipeRing - 1 : slot_in - 1);
          wait_vm<NP*(kPipeRing - 1)>();  // row n + 1 is in
        }
        read_row(c[(e + NS - 1) % NS], n + 1);
      }
      if (KIND == PIPE_LAST) {
        // the row of step n - 1 from LDS to memory, a share after each sweep
        // (read after one, stored after the next, so nothing waits for LDS)
        const int orow = r0 - 2 * D + n - 1;
        const uint64_t rm = (orow >= r0 && orow < r1) ? ~0ull : 0ull;
        gdouble* rp = out + (int64_t)orow * pitch + kColOff + w0;

        auto put = [&](int from) __attribute__((always_inline)) {
#pragma unroll
          for (int x = 0; x < PS; x++) {
            const int m = from + x;
            if (m < NP)
              store_masked(rp, 16 * lane + 1024 * m, hold[x], stm[m] & rm);
          }
        };
        if (s > 0) put((s - 1) * PS);
        if (s > 0 && s == NST - 1) store_masked(rp, 8 * tail, hold_t, tail_m & rm);
        if (s < NST - 1 || NST == 1) {
#pragma unroll
          for (int x = 0; x < PS; x++) {
            const int m = s * PS + x;
            if (m < NP) hold[x] = *(const llpair*)(row_r + 128 * m);
          }
          if (s == NST - 2 || NST == 1) hold_t = row[tail];
        }
        if (NST == 1) {  // (nothing to overlap with: read, then store)
          put(0);
          store_masked(rp, 8 * tail, hold_t, tail_m & rm);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    double* O = c[(e + NST) % NS];
    if (KIND != PIPE_LAST) {
      lds_wait_ge(out_used, n + 1 - kPipeLink, k_used);
      ldouble* dst = lout + slot_out * ROW;
#pragma unroll
      for (int j = 0; j + 1 < K; j += 2) {
        lpair v;
        v.x = O[j];
        v.y = O[j + 1];
        *(llpair*)(dst + j * 64) = v;
      }
      if (K & 1) *(dst + (K - 1) * 64 - lane) = O[K - 1];
      lds_post(out_made, n + 1);
      slot_out = slot_out == kPipeLink - 1 ? 0 : slot_out + 1;
    } else {
#pragma unroll
      for (int j = 0; j < K; j++) row_w[j] = O[j];
    }
  };
  // sweep s of step n makes row q0 + n - s: the turns that begin before tA may
  // meet the top ring row, later ones the bottom one.  The last of the former
  // ends with row top + NST + NS - 2 = top + 2 NST at most: the bottom ring row
  // lies beyond it in a grid of D = 4 NST rows or more.
  static_assert(D + 1 > NST + NS - 2, "both ring rows in one turn");
  const int tA = top != kNoRing ? top - q0 + NST : 0;
  for (int t0 = 0; t0 < n_steps; t0 += NS) {
    ring_row = t0 < tA ? top : bottom;
    ring_at = t0 < tA ? 0 : ROWB;
#pragma unroll
    for (int u = 0; u < NS; u++) step(u, t0 + u);
  }
  // fetches and stores the compiler does not know of
  if (KIND != PIPE_MIDDLE) wait_vm<0>();
  if (SUM && KIND == PIPE_LAST) {
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
    double* slot = suni(jp->sum);
    if (lane == 0 && sum != 0.0)
      __hip_atomic_fetch_add(slot, sum, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <int T, int K, int NST, int COLS, bool SUM>
__device__ __forceinline__ void pipe_group_cols(int role, int off) {
  if (role == 0)
    pipe_wave<T, K, NST, COLS, PIPE_FIRST, false>(role, off);
  else if (role < kPipeWaves - 1)
    pipe_wave<T, K, NST, COLS, PIPE_MIDDLE, false>(role, off);
  else
    pipe_wave<T, K, NST, COLS, PIPE_LAST, SUM>(role, off);
}
template <int T, int K, int NST, bool SUM>
__device__ __forceinline__ void pipe_group(int cols, int role, int off) {
  switch (cols) {
    case 0: pipe_group_cols<T, K, NST, 0, SUM>(role, off); break;
    case 2: pipe_group_cols<T, K, NST, 2, SUM>(role, off); break;
    default: pipe_group_cols<T, K, NST, 3, SUM>(role, off); break;
  }
}

// ---------------------------------------------------------------------------
// a block
// ---------------------------------------------------------------------------
// A block of an array: output columns [cols.c0, cols.c1) and rows [r0, r1),
// the grid's ring rows and columns (kNoRing where they are out of reach) and
// the part of the input that may be read (odd columns to lo_col at least).
// Ring rows, if both are in reach, are more than 2 NST rows apart (callers'
// grids have 4 NST rows at least).
struct PipeBlock {
  const double* in;
  double* out;
  int64_t pitch;
  PipeCols cols;
  int r0, r1, top, bottom;
  int lo_col, hi_col, lo_row, hi_row;
  double ring;  // the ring's value (cols.flat)
};

// The groups' LDS, one for all passes of a kernel of T-thread workgroups.
template <int T>
__device__ inline PipeLds* pipe_lds() {
  __shared__ PipeLds lds[T / 64 / kPipeWaves];
  return lds;
}

// Workgroup-collective (T threads, all waves): 4 NST fused sweeps of the
// block.  Groups take whole windows in turn; of an odd number the last one
// is halved by rows (so both groups always have as many windows to do).
template <int T, int NST, bool SUM>
__device__ __forceinline__ void pipe_block(const PipeBlock& b, double* sum) {
  constexpr int G = T / 64 / kPipeWaves;
  constexpr int D = kPipeWaves * NST;
  static_assert(G == 1 || G == 2, "one or two groups");
  const int wave = suni((int)(threadIdx.x / 64));
  const int grp = wave / kPipeWaves;
  // the second group's waves in the other order: the first and the last wave
  // have the loads and stores to do, and waves i and i + 4 share a SIMD
  const int role = grp ? kPipeWaves - 1 - wave % kPipeWaves : wave % kPipeWaves;
  const int k = pipe_pick_k(b.cols, D);
  const PipeSplit sp = pipe_split(b.cols, D, k);
  const int whole = sp.n / G * G;
  const int turns = (sp.n + G - 1) / G;
  const int rows = b.r1 - b.r0;
  typedef __attribute__((address_space(3))) PipeLds lPipeLds;
  PipeLds* my = pipe_lds<T>() + grp;
  const int off = suni((int)(uint32_t)(uintptr_t)(lPipeLds*)my);
  for (int t = 0; t < turns; t++) {
    int win = t * G + grp, ra = b.r0, rb = b.r1;
    if (t * G >= whole) {  // the odd window: half the rows each
      win = sp.n - 1;
      if (G == 2) {
        const int half = (rows + 1) / 2;
        if (grp == 0)
          rb = b.r0 + half;
        else
          ra = b.r0 + half;
      }
    }
    PipeJob j;
    const int cols = pipe_window(sp, win, b.cols, D, &j);
    j.in = b.in;
    j.out = b.out;
    j.sum = sum;
    j.ring = b.ring;
    j.pitch = b.pitch;
    j.r0 = ra;
    j.r1 = rb;
    j.lo_col = b.lo_col;
    j.hi_col = b.hi_col;
    j.lo_row = b.lo_row;
    j.hi_row = b.hi_row;
    j.top = b.top >= ra - D ? b.top : kNoRing;
    j.bottom = b.bottom < rb + D ? b.bottom : kNoRing;
    __syncthreads();  // the last turn's rows and job are done with
    if (threadIdx.x % (64 * kPipeWaves) == 0) {
      my->job = j;
      for (int i = 0; i < kPipeWaves; i++) my->made[i] = my->used[i] = 0;
    }
    __syncthreads();
    if (ra >= rb || j.oc0 >= j.oc1) continue;
    switch (k) {
      case 3: pipe_group<T, 3, NST, SUM>(cols, role, off); break;
      case 5: pipe_group<T, 5, NST, SUM>(cols, role, off); break;
      default: pipe_group<T, 9, NST, SUM>(cols, role, off); break;
    }
  }
}

}  // namespace jac
}  // namespace chm
