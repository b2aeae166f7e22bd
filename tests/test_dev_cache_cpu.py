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
#include <map>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
struct FakeHip {
  std::mutex mu;
  size_t total = 800u << 20, used[2] = {0, 0};
  std::map<void*, std::pair<int, size_t>> blocks;
  char* next = (char*)4096;
  int frees = 0;
  bool running[2] = {false, false};  // a kernel that this thread has to stop
};
inline FakeHip& fake() { static FakeHip* f = new FakeHip; return *f; }
inline int& cur_dev() { static thread_local int d = 0; return d; }
inline hipError_t hipGetDevice(int* d) { *d = cur_dev(); return hipSuccess; }
inline hipError_t hipSetDevice(int d) { cur_dev() = d; return hipSuccess; }
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
  std::lock_guard<std::mutex> lk(f.mu);
  auto it = f.blocks.find(p);
  if (it == f.blocks.end()) abort();  // freed twice, or never taken
  if (f.running[it->second.first]) abort();  // would wait for ever
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
    CHECK(DevCache::get().held_back());
    fake().running[0] = false;
    DevCache::get().serving(0, -1);
    DevCache::get().put(pool, true);
    CHECK(!DevCache::get().held_back());
    CHECK(DevCache::get().release(0));
    CHECK(fake().used[0] == 0);""",
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
