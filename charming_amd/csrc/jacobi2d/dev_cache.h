// Device memory of the batched and served forms, kept between calls: grids
// and queues are gigabytes that a call needs for tens of milliseconds, and
// taking 16 GiB from the driver and giving it back costs 240-480 ms (a served
// burst of 24 requests, 16 GiB of pool: 470 ms, now 134; 512 problems, 17 GB of
// grids: 110-490, now 75).
//
// What is kept is bounded (an eighth of the device's memory, kBlocks blocks;
// the longest unused go first), holds no data (every user writes what it
// reads), and goes back when it has not been used for ten seconds (by a thread
// that lives while anything is kept), when an allocation made here fails,
// before a server's engine starts, and by chm_jacobi2d_release_memory().  A
// block is kept only once the work that used it has ended, so any stream may
// take it next.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <mutex>
#include <thread>

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

  // keep: how long a block is kept unused.
  explicit DevCache(std::chrono::milliseconds keep) : keep_(keep) {}

  // (never destroyed: its blocks go with the process)
  static DevCache& get() {
    static DevCache* c = new DevCache(std::chrono::seconds(10));
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
    void* out[kBlocks + 1];
    int n_out = 0;
    {
      std::lock_guard<std::mutex> lk(mu_);
      const bool reaped = start_reaper();
      while (reaped) {
        size_t sum = b.bytes;
        int old = -1;
        for (int i = 0; i < n_; i++) {
          if (kept_[i].b.dev != b.dev) continue;
          sum += kept_[i].b.bytes;
          if (old < 0 || kept_[i].t < kept_[old].t) old = i;
        }
        if (old < 0 || (sum <= total / 8 && n_ < kBlocks)) break;
        out[n_out++] = kept_[old].b.p;
        kept_[old] = kept_[--n_];
      }
      if (reaped && n_ < kBlocks)
        kept_[n_++] = Kept{b, Clock::now()};
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
    std::unique_lock<std::mutex> lk(mu_);
    if (dev >= 0 && dev < kDevices) servers_[dev] += change;
    if (change > 0) idle_.wait(lk, [this] { return !freeing_; });
  }
  // Bytes that are kept on `dev` and an allocation here could have.
  size_t available(int dev) {
    std::lock_guard<std::mutex> lk(mu_);
    size_t sum = 0;
    for (int i = 0; i < n_; i++)
      if (kept_[i].b.dev == dev && servers(dev) == 0) sum += kept_[i].b.bytes;
    return sum;
  }
  // Something is kept that a running server holds back.
  bool held_back() {
    std::lock_guard<std::mutex> lk(mu_);
    for (int i = 0; i < n_; i++)
      if (servers(kept_[i].b.dev) > 0) return true;
    return false;
  }
  // The same for the current device; true also if the reaper's frees, which
  // were under way, have ended meanwhile.
  bool release_current() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    bool some = release(dev);
    std::unique_lock<std::mutex> lk(mu_);
    for (; freeing_; some = true) idle_.wait(lk);
    return some;
  }
  // Ends the reaper (what is kept stays): for the process's exit.
  void stop() {
    std::unique_lock<std::mutex> lk(mu_);
    quit_ = true;
    wake_.notify_all();
    idle_.wait_for(lk, std::chrono::seconds(10), [this] { return !reaping_; });
  }

 private:
  using Clock = std::chrono::steady_clock;
  static constexpr int kBlocks = 48;
  static constexpr int kDevices = 64;
  struct Kept {
    DevBlock b;
    Clock::time_point t;
  };
  // With the lock held: sees to it that the reaper runs.  False where it
  // cannot (nothing is kept then).
  bool start_reaper() {
    if (reaping_ || quit_) return reaping_ && !quit_;
    // HIP's own exit handlers were registered at its first call, so this one
    // runs before them and no free meets a runtime that has gone.
    static const int at_exit = std::atexit([] { get().stop(); });
    if (at_exit != 0) return false;
    try {
      std::thread([this] { reap(); }).detach();
      reaping_ = true;
    } catch (...) {  // (no thread to be had)
    }
    return reaping_;
  }

  void reap() {
    // a free must not end a graph capture of another thread
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    std::unique_lock<std::mutex> lk(mu_);
    while (n_ > 0 && !quit_) {
      const auto now = Clock::now();
      auto next = now + keep_;
      void* out[kBlocks];
      int n_out = 0;
      for (int i = n_ - 1; i >= 0; i--) {
        if (servers(kept_[i].b.dev) > 0) kept_[i].t = now;
        if (now - kept_[i].t >= keep_) {
          out[n_out++] = kept_[i].b.p;
          kept_[i] = kept_[--n_];
        } else {
          next = std::min(next, kept_[i].t + keep_);
        }
      }
      if (n_out == 0) {
        wake_.wait_until(lk, next);
        continue;
      }
      freeing_ = true;
      lk.unlock();
      for (int i = 0; i < n_out; i++) (void)hipFree(out[i]);
      lk.lock();
      freeing_ = false;
      idle_.notify_all();
    }
    reaping_ = false;
    idle_.notify_all();
  }

  int servers(int dev) const {
    return dev >= 0 && dev < kDevices ? servers_[dev] : 0;
  }
  const std::chrono::milliseconds keep_;
  std::mutex mu_;
  std::condition_variable wake_, idle_;  // the reaper; who waits for it
  bool reaping_ = false, freeing_ = false, quit_ = false;
  int servers_[kDevices] = {};
  Kept kept_[kBlocks];
  int n_ = 0;
};

}  // namespace jac
}  // namespace chm
