"""The device memory kept between calls
(charming_amd/csrc/jacobi2d/dev_cache.h, compiled for the host against a
stand-in for the few HIP calls it makes: two devices of 800 MiB)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "charming_amd", "csrc", "jacobi2d")
HIP = r"""
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <atomic>
#include <chrono>
#include <map>
#include <mutex>
#include <thread>
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeRelaxed };
inline hipStreamCaptureMode& capture_mode() {
  static thread_local hipStreamCaptureMode m = hipStreamCaptureModeGlobal;
  return m;
}
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
struct FakeHip {
  std::mutex mu;
  size_t total = 800u << 20, used[2] = {0, 0};
  std::map<void*, std::pair<int, size_t>> blocks;
  char* next = (char*)4096;
  int frees = 0;
  bool running[2] = {false, false};  // a kernel that this thread has to stop
  bool capturing = false;            // a global capture is under way
  std::atomic<int> free_ms{0};       // how long a free takes
};
inline FakeHip& fake() { static FakeHip* f = new FakeHip; return *f; }
inline int& cur_dev() { static thread_local int d = 0; return d; }
inline hipError_t hipGetDevice(int* d) { *d = cur_dev(); return hipSuccess; }
inline hipError_t hipSetDevice(int d) { cur_dev() = d; return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  std::swap(*m, capture_mode());
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipDeviceTotalMem(size_t* t, int) {
  *t = fake().total;
  return hipSuccess;
}
template <class T>
hipError_t hipMalloc(T** p, size_t n) {
  FakeHip& f = fake();
  std::lock_guard<std::mutex> lk(f.mu);
  if (f.used[cur_dev()] + n > f.total) return hipErrorOutOfMemory;
  f.used[cur_dev()] += n;
  *p = (T*)f.next;
  f.next += n + 4096;
  f.blocks[*p] = {cur_dev(), n};
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  FakeHip& f = fake();
  std::this_thread::sleep_for(std::chrono::milliseconds(f.free_ms));
  std::lock_guard<std::mutex> lk(f.mu);
  auto it = f.blocks.find(p);
  if (it == f.blocks.end()) abort();  // freed twice, or never taken
  if (f.running[it->second.first]) abort();  // would wait for ever
  if (f.capturing && capture_mode() != hipStreamCaptureModeRelaxed) abort();
  f.used[it->second.first] -= it->second.second;
  f.blocks.erase(it);
  f.frees++;
  return hipSuccess;
}
"""
MAIN = r"""
#include "dev_cache.h"
#include <stdio.h>
#include <string>
#include <vector>
using chm::jac::DevBlock;
using chm::jac::DevCache;
#define CHECK(x) \
  do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
constexpr size_t MB = 1u << 20;
static DevBlock take(size_t bytes) {
  DevBlock b;
  CHECK(DevCache::get().take(&b, bytes) == hipSuccess);
  return b;
}
static size_t used(int dev) {
  std::lock_guard<std::mutex> lk(fake().mu);
  return fake().used[dev];
}
static void set(bool& flag, bool v) {
  std::lock_guard<std::mutex> lk(fake().mu);
  flag = v;
}
static void sleep_ms(int ms) {
  std::this_thread::sleep_for(std::chrono::milliseconds(ms));
}
// used(dev) == bytes within five seconds
static bool comes_to(int dev, size_t bytes) {
  for (int i = 0; i < 500 && used(dev) != bytes; i++) sleep_ms(10);
  return used(dev) == bytes;
}
static void keep(int dev, size_t bytes) {
  (void)hipSetDevice(dev);
  DevCache::get().put(take(bytes), true);
}
int main(int argc, char** argv) {
  const std::string what = argv[1];
%s
  CHECK(!"no such test");
}
"""
TESTS = {
    "per_device": r"""
    // a failing allocation gives back its own device's blocks, no other's
    keep(0, 40 * MB);
    keep(1, 50 * MB);
    (void)hipSetDevice(0);
    void* p = nullptr;
    CHECK(DevCache::get().alloc(&p, 790 * MB) == hipSuccess);
    CHECK(fake().used[0] == 790 * MB && fake().used[1] == 50 * MB);
    void* q = nullptr;  // nothing left to give back here: it fails
    CHECK(DevCache::get().alloc(&q, 790 * MB) == hipErrorOutOfMemory);
    CHECK(fake().used[1] == 50 * MB && fake().frees == 1);
    // all devices' when asked for
    (void)hipFree(p);
    keep(0, 30 * MB);
    CHECK(DevCache::get().release(DevCache::kAllDevices));
    CHECK(fake().used[0] == 0 && fake().used[1] == 0);
    CHECK(!DevCache::get().release(DevCache::kAllDevices));""",
    "bounds": r"""
    // at most an eighth of the device, the longest unused first, and a block
    // in the hands of one user only
    keep(0, 60 * MB);
    const DevBlock a = take(55 * MB);  // the 60 MB one
    CHECK(a.bytes == 60 * MB && fake().used[0] == 60 * MB);
    const DevBlock b = take(55 * MB);
    CHECK(b.p != a.p && fake().used[0] == 115 * MB);
    DevCache::get().put(a, true);
    DevCache::get().put(b, true);  // 115 MB > 100 MB: a goes
    CHECK(fake().used[0] == 55 * MB && fake().blocks.count(b.p));
    keep(0, 101 * MB);  // too large to keep at all
    CHECK(fake().used[0] == 55 * MB);
    DevCache::get().put(take(20 * MB), false);  // work that failed: not kept
    CHECK(fake().used[0] == 55 * MB);""",
    "server": r"""
    // what is kept goes back before a server's engine starts; while it runs a
    // failing allocation fails at once, and nothing is given back there
    keep(0, 40 * MB);
    keep(1, 50 * MB);
    (void)hipSetDevice(0);
    const DevBlock pool = take(700 * MB);
    DevCache::get().serving(0, +1);
    CHECK(fake().used[0] == 700 * MB && fake().used[1] == 50 * MB);
    fake().running[0] = true;
    keep(0, 60 * MB);  // another thread's batch ends meanwhile
    void* p = nullptr;
    CHECK(DevCache::get().alloc(&p, 90 * MB) == hipErrorOutOfMemory);
    CHECK(DevCache::get().release(DevCache::kAllDevices));  // device 1's
    CHECK(fake().used[0] == 760 * MB && fake().used[1] == 0);
    CHECK(DevCache::get().held_back() && DevCache::get().available(0) == 0);
    fake().running[0] = false;
    DevCache::get().serving(0, -1);
    DevCache::get().put(pool, true);
    CHECK(!DevCache::get().held_back());
    CHECK(DevCache::get().release(0));
    CHECK(fake().used[0] == 0);""",
    "available": r"""
    // what an allocation could have on a device counts as free there
    keep(0, 40 * MB);
    keep(0, 30 * MB);
    keep(1, 20 * MB);
    CHECK(DevCache::get().available(0) == 70 * MB);
    CHECK(DevCache::get().available(1) == 20 * MB);
    (void)hipSetDevice(0);
    const DevBlock b = take(40 * MB);
    CHECK(DevCache::get().available(0) == 30 * MB);
    void* p = nullptr;
    CHECK(DevCache::get().alloc(&p, 760 * MB) == hipSuccess);
    CHECK(DevCache::get().available(0) == 0);""",
    "timed": r"""
    // what is not used for a while goes back by itself, also under another
    // thread's graph capture, and again after all had gone
    DevCache& c = *new DevCache(std::chrono::milliseconds(400));
    for (int turn = 0; turn < 2; turn++) {
      DevBlock a, b;
      CHECK(c.take(&a, 30 * MB) == hipSuccess);
      CHECK(c.take(&b, 50 * MB) == hipSuccess);
      c.put(a, true);
      sleep_ms(200);
      set(fake().capturing, true);
      c.put(b, true);
      CHECK(used(0) == 80 * MB);
      CHECK(comes_to(0, 50 * MB) && comes_to(0, 0));
      set(fake().capturing, false);
    }
    // a block in use stays, one given to a new user too
    DevBlock d, e;
    CHECK(c.take(&d, 30 * MB) == hipSuccess);
    c.put(d, true);
    sleep_ms(200);
    CHECK(c.take(&e, 30 * MB) == hipSuccess && e.p == d.p);
    sleep_ms(600);
    CHECK(used(0) == 30 * MB);
    c.put(e, true);
    CHECK(comes_to(0, 0));""",
    "timed_server": r"""
    // not while a server runs, whose start waits for frees under way
    DevCache& c = *new DevCache(std::chrono::milliseconds(200));
    DevBlock a, b;
    CHECK(c.take(&a, 30 * MB) == hipSuccess);
    c.put(a, true);
    fake().free_ms = 300;
    sleep_ms(350);  // (its free is under way, or about to be)
    c.serving(0, +1);
    CHECK(used(0) == 0);
    set(fake().running[0], true);
    CHECK(c.take(&b, 30 * MB) == hipSuccess);
    c.put(b, true);
    sleep_ms(700);
    CHECK(used(0) == 30 * MB && c.held_back());
    set(fake().running[0], false);
    c.serving(0, -1);
    CHECK(comes_to(0, 0));""",
    "failing_meanwhile": r"""
    // an allocation that fails while the thread frees waits for it
    DevCache& c = *new DevCache(std::chrono::milliseconds(200));
    DevBlock a;
    CHECK(c.take(&a, 90 * MB) == hipSuccess);
    c.put(a, true);
    fake().free_ms = 400;
    sleep_ms(400);
    void* p = nullptr;
    CHECK(c.alloc(&p, 790 * MB) == hipSuccess);""",
    "stop": r"""
    // the thread ends on request, at once, and nothing is kept or freed by it
    // afterwards
    DevCache& c = *new DevCache(std::chrono::milliseconds(300));
    DevBlock a, b;
    CHECK(c.take(&a, 30 * MB) == hipSuccess);
    CHECK(c.take(&b, 20 * MB) == hipSuccess);
    c.put(a, true);
    const auto t0 = std::chrono::steady_clock::now();
    c.stop();
    CHECK(std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(250));
    c.put(b, true);
    CHECK(used(0) == 30 * MB);
    sleep_ms(500);
    CHECK(used(0) == 30 * MB);""",
    "threads": r"""
    // takes and returns by several threads beside the one that gives back
    DevCache& c = *new DevCache(std::chrono::milliseconds(3));
    std::vector<std::thread> ts;
    for (int t = 0; t < 6; t++)
      ts.emplace_back([&c, t] {
        (void)hipSetDevice(t & 1);
        for (int i = 0; i < 400; i++) {
          DevBlock a, b;
          CHECK(c.take(&a, (1 + (i * 7 + t) % 9) * MB) == hipSuccess);
          CHECK(c.take(&b, (1 + (i * 5 + t) % 30) * MB) == hipSuccess);
          CHECK(a.p != b.p);
          if (i % 40 == t) sleep_ms(5);
          c.put(a, true);
          c.put(b, i % 3 != 0);
          if (i % 50 == t) c.release(t & 1);
          if (i % 60 == t) {
            c.serving(t & 1, +1);
            c.serving(t & 1, -1);
          }
        }
      });
    for (auto& t : ts) t.join();
    CHECK(comes_to(0, 0) && comes_to(1, 0));""",
    "exit": r"""
    // a process may end with memory kept and its thread waiting
    keep(0, 40 * MB);""",
}


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("cache")
    os.makedirs(d / "hip")
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    body = "".join('  if (what == "%s") {%s\n    return 0;\n  }\n' % kv
                   for kv in TESTS.items())
    (d / "main.cpp").write_text(MAIN.replace("%s\n", body, 1))
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-I", str(d), "-I",
                           CSRC, str(d / "main.cpp"), "-o", str(d / "main"),
                           "-lpthread"])
    return str(d / "main")


@pytest.mark.parametrize("what", list(TESTS))
def test_cache(exe, what):
    p = subprocess.run([exe, what], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
