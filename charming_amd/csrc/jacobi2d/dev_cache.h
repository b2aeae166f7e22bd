// Device memory of the batched and served forms, kept between calls: grids
// and queues are gigabytes that a call needs for tens of milliseconds, and
// taking 16 GiB from the driver and giving it back costs 240-480 ms (a served
// burst of 24 requests, 16 GiB of pool: 470 ms, now 134; 512 problems, 17 GB of
// grids: 110-490, now 75).
//
// What is kept is bounded (an eighth of the device's memory, kBlocks blocks;
// the longest unused go first), holds no data (every user writes what it
// reads), is given back when any allocation of this library fails, when a
// block has not been used for kKeepSeconds and another is returned, and by
// chm_jacobi2d_release_memory().  A block is kept only once the work that used
// it has ended, so any stream may take it next.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <chrono>
#include <mutex>

namespace chm {
namespace jac {

struct DevBlock {
  void* p = nullptr;
  size_t bytes = 0;  // may exceed what was asked for
  int dev = 0;       // the device it is on
};

class DevCache {
 public:
  static constexpr int kAllDevices = -1;

  // (never destroyed: its blocks go with the process)
  static DevCache& get() {
    static DevCache* c = new DevCache;
    return *c;
  }

  // At least `bytes` of the current device: the smallest kept block of up to
  // a quarter and 1 MiB more, or new memory.
  hipError_t take(DevBlock* b, size_t bytes) {
    hipError_t e = hipGetDevice(&b->dev);
    if (e != hipSuccess) return e;
    {
      std::lock_guard<std::mutex> lk(mu_);
      Kept* best = nullptr;
      for (int i = 0; i < n_; i++)
        if (kept_[i].b.dev == b->dev && kept_[i].b.bytes >= bytes &&
            kept_[i].b.bytes - bytes <= bytes / 4 + (1 << 20) &&
            (!best || kept_[i].b.bytes < best->b.bytes))
          best = &kept_[i];
      if (best) {
        *b = best->b;
        *best = kept_[--n_];
        return hipSuccess;
      }
    }
    b->bytes = bytes;
    return alloc(&b->p, bytes);
  }

  // hipMalloc, with what is kept on the current device given back if it fails.
  template <class T>
  hipError_t alloc(T** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess || !release_current()) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
  }

  // Returns a block; `idle` says that nothing uses it any more.
  void put(DevBlock b, bool idle) {
    if (!b.p) return;
    size_t total = 0;
    if (!idle || hipDeviceTotalMem(&total, b.dev) != hipSuccess ||
        b.bytes > total / 8) {
      (void)hipFree(b.p);
      return;
    }
    const auto now = Clock::now();
    void* out[kBlocks + 1];
    int n_out = 0;
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (;;) {
        size_t sum = b.bytes;
        int old = -1;
        for (int i = 0; i < n_; i++) {
          if (kept_[i].b.dev != b.dev) continue;
          sum += kept_[i].b.bytes;
          if (old < 0 || kept_[i].t < kept_[old].t) old = i;
        }
        if (old < 0 || (sum <= total / 8 && n_ < kBlocks &&
                        now - kept_[old].t < std::chrono::seconds(kKeepSeconds)))
          break;
        out[n_out++] = kept_[old].b.p;
        kept_[old] = kept_[--n_];
      }
      if (n_ < kBlocks)
        kept_[n_++] = Kept{b, now};
      else
        out[n_out++] = b.p;
    }
    // (outside the lock: a free may wait for work on the device)
    for (int i = 0; i < n_out; i++) (void)hipFree(out[i]);
  }

  // Gives back what is kept on `dev` (kAllDevices: on any); false if nothing
  // was.  Not where a server runs: see serving().
  bool release(int dev) {
    void* out[kBlocks];
    int n_out = 0;
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (int i = n_ - 1; i >= 0; i--) {
        if (dev != kAllDevices && kept_[i].b.dev != dev) continue;
        if (servers(kept_[i].b.dev) > 0) continue;
        out[n_out++] = kept_[i].b.p;
        kept_[i] = kept_[--n_];
      }
    }
    for (int i = 0; i < n_out; i++) (void)hipFree(out[i]);
    return n_out > 0;
  }
  // A server's engine starts (+1) or has stopped (-1) on `dev`.  hipFree waits
  // for every kernel of the device, and this one ends only when its owner, who
  // may be the thread that frees, stops it: what is kept goes back before it
  // starts, and nothing while it runs (an allocation that fails then fails at
  // once).
  void serving(int dev, int change) {
    if (change > 0) (void)release(dev);
    std::lock_guard<std::mutex> lk(mu_);
    if (dev >= 0 && dev < kDevices) servers_[dev] += change;
  }
  // Something is kept that a running server holds back.
  bool held_back() {
    std::lock_guard<std::mutex> lk(mu_);
    for (int i = 0; i < n_; i++)
      if (servers(kept_[i].b.dev) > 0) return true;
    return false;
  }
  bool release_current() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess && release(dev);
  }

 private:
  using Clock = std::chrono::steady_clock;
  static constexpr int kBlocks = 48;
  static constexpr int kDevices = 64;
  static constexpr int kKeepSeconds = 10;
  struct Kept {
    DevBlock b;
    Clock::time_point t;
  };
  int servers(int dev) const {
    return dev >= 0 && dev < kDevices ? servers_[dev] : 0;
  }
  std::mutex mu_;
  int servers_[kDevices] = {};
  Kept kept_[kBlocks];
  int n_ = 0;
};

}  // namespace jac
}  // namespace chm
