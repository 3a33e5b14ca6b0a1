"""Bookkeeping of the device blocks kept between objects (mg_block_cache.hpp), on the host against a
driver that counts: each check is one function of the program below."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include <cassert>
#include <cstdio>
#include <cstring>
#include <limits>
#include <set>
#include <thread>
#include <vector>
#include "mg_block_cache.hpp"
using namespace mgamd;

// A driver with `capacity` bytes, which refuses what it does not know as hipFree does. Of the
// temporaries' pool it knows the bytes held and not used.
struct Driver {
  using Status = int;
  static constexpr int kOk = 0, kOutOfMemory = 2, kInvalid = 1;
  static inline std::mutex mu;
  static inline size_t capacity = ~size_t{0} / 2, used = 0, idle_pool = 0, last_bytes = 0;
  static inline int device = 0, waits = 0, frees = 0, mallocs = 0;
  static inline uintptr_t next = 4096;
  static inline std::map<void*, size_t> blocks;
  static int malloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    ++mallocs;
    last_bytes = bytes;
    if (bytes > capacity || used + idle_pool + queued_pool > capacity - bytes) return kOutOfMemory;
    *p = reinterpret_cast<void*>(next);
    next += (bytes + 4096) / 4096 * 4096;
    blocks[*p] = bytes;
    used += bytes;
    return kOk;
  }
  static int free(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    auto it = blocks.find(p);
    if (it == blocks.end()) return kInvalid;
    ++frees;
    used -= it->second;
    blocks.erase(it);
    return kOk;
  }
  static int current_device(int* d) { *d = device; return kOk; }
  static bool wait() { ++waits; return true; }
  using Stream = int;  // kCapturing: one that must not be waited for
  static constexpr int kCapturing = 7;
  static inline size_t queued_pool = 0;  // freed, but work in front of the free has not finished
  static int pool_malloc(void** p, size_t bytes, Stream) {
    if (bytes <= idle_pool) idle_pool -= bytes;
    return malloc(p, bytes);
  }
  static bool settle(Stream s) {
    if (s == kCapturing) return false;
    idle_pool += queued_pool;
    queued_pool = 0;
    return true;
  }
  static void trim(int) { idle_pool = 0; }
};
using Cache = BlockCache<Driver>;
constexpr size_t kMB = 1 << 20;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

static void* take(Cache& c, size_t bytes) {
  void* p = nullptr;
  return c.alloc(bytes, &p) == Driver::kOk ? p : nullptr;
}

// A block that was freed and is kept is refused, and handed out to one caller only.
static int freed_twice() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  void* const p = take(c, kMB);
  CHECK(p && c.free(p) == Driver::kOk && Driver::frees == 0);
  CHECK(c.free(p) == Driver::kInvalid && Driver::frees == 0);
  CHECK(c.free(p) == Driver::kInvalid);
  CHECK(take(c, kMB) == p && Driver::blocks.count(p));
  CHECK(take(c, kMB) != p);
  return 0;
}
// What the cache has not handed out is the driver's.
static int foreign() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  CHECK(c.free(reinterpret_cast<void*>(12345)) == Driver::kInvalid);
  void* theirs = nullptr;
  Driver::malloc(&theirs, kMB);
  CHECK(c.free(theirs) == Driver::kOk && Driver::frees == 1);
  CHECK(c.free(theirs) == Driver::kInvalid);
  CHECK(c.free(nullptr) == Driver::kOk);
  return 0;
}
// Sizes: rounded to 512 bytes; a kept block serves what is up to an eighth smaller.
static int sizes() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  void* const p = take(c, 900);
  CHECK(Driver::blocks[p] == 1024);
  c.free(p);
  CHECK(take(c, 1024) == p);
  c.free(p);
  CHECK(take(c, 1025) != p && take(c, 512) != p && take(c, 1000) == p);
  void* const q = take(c, 9 * kMB);
  c.free(q);
  CHECK(take(c, 7 * kMB) != q && take(c, 8 * kMB) == q);
  return 0;
}
// At most the limit is kept, the oldest out first, and no block above half of it.
static int limit() {
  Cache c;
  c.add_context(0, 64 * 10 * kMB);  // 10 MB
  void* const big = take(c, 5 * kMB + 512);
  c.free(big);
  CHECK(Driver::frees == 1 && Driver::used == 0);
  std::vector<void*> p;
  for (int i = 0; i < 4; ++i) p.push_back(take(c, 3 * kMB));
  for (void* x : p) c.free(x);
  CHECK(Driver::frees == 2 && Driver::used == 9 * kMB);
  CHECK(!Driver::blocks.count(p[0]) && Driver::blocks.count(p[1]) && Driver::blocks.count(p[3]));
  return 0;
}
// Everything goes back with the device's last context; without one nothing is kept.
static int last_context() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  c.add_context(0, 64 * 100 * kMB);
  void *a = take(c, kMB), *b = take(c, kMB), *outlives = take(c, kMB);
  c.free(a);
  Driver::idle_pool = kMB;
  c.drop_context(0);
  CHECK(Driver::used == 3 * kMB && Driver::idle_pool == kMB);
  c.free(b);
  c.drop_context(0);
  CHECK(Driver::used == kMB && Driver::idle_pool == 0);
  CHECK(c.free(outlives) == Driver::kOk && Driver::used == 0);
  CHECK(c.free(outlives) == Driver::kInvalid);
  return 0;
}
// A device's blocks stay its own; one freed with another device current goes to the driver.
static int devices() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  c.add_context(1, 64 * 100 * kMB);
  void* const p = take(c, kMB);
  c.free(p);
  Driver::device = 1;
  void* const q = take(c, kMB);
  CHECK(q != p);
  Driver::device = 0;
  CHECK(take(c, kMB) == p);
  CHECK(c.free(q) == Driver::kOk && Driver::frees == 1);
  return 0;
}
// A block is kept only after a wait; the frees of a scope share one.
static int waits() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  void *a = take(c, kMB), *b = take(c, 2 * kMB), *d = take(c, 3 * kMB);
  c.free(a);
  CHECK(Driver::waits == 1);
  {
    FreeScope outer, inner;
    c.free(b);
    c.free(d);
  }
  CHECK(Driver::waits == 2);
  c.free(take(c, kMB));
  CHECK(Driver::waits == 3);
  return 0;
}
// Threads allocating and freeing: no block is handed out twice, nothing is lost.
static int threads() {
  Cache c;
  c.add_context(0, 64 * 20 * kMB);
  std::mutex mu;
  std::set<void*> out;
  bool bad = false;
  auto work = [&](int seed) {
    for (int i = 0; i < 2000; ++i) {
      void* const p = take(c, kMB * (1 + (seed + i) % 3));
      { std::lock_guard<std::mutex> lock(mu); bad |= !p || !out.insert(p).second; }
      { std::lock_guard<std::mutex> lock(mu); out.erase(p); }
      bad |= c.free(p) != Driver::kOk;
    }
  };
  std::vector<std::thread> t;
  for (int i = 0; i < 4; ++i) t.emplace_back(work, i);
  for (auto& x : t) x.join();
  CHECK(!bad && Driver::used <= 20 * kMB);
  c.drop_context(0);
  CHECK(Driver::used == 0);
  return 0;
}

// A device that is full but for kept blocks and the pool's idle memory: an object and a temporary both
// get memory once these are given back, and fail as before where that is not enough.
static int out_of_memory() {
  Cache c;
  c.add_context(0, 64 * 40 * kMB);
  Driver::capacity = 100 * kMB;
  void* p = nullptr;
  auto fill = [&] {  // 20 MB of kept blocks, 30 MB idle in the pool, 10 MB on their way there
    void *a = take(c, 10 * kMB), *b = take(c, 10 * kMB);
    c.free(a);
    c.free(b);
    Driver::idle_pool = 30 * kMB;
    Driver::queued_pool = 10 * kMB;
  };
  fill();
  CHECK(c.alloc(70 * kMB, &p) == Driver::kOk && Driver::used == 70 * kMB && Driver::idle_pool == 0);
  c.free(p);
  Driver::queued_pool = 0;
  fill();
  CHECK(c.pool_alloc(90 * kMB, 0, &p) == Driver::kOk && Driver::used == 90 * kMB);
  Driver::free(p);
  fill();
  CHECK(c.pool_alloc(101 * kMB, 0, &p) == Driver::kOutOfMemory && !p);
  CHECK(c.alloc(101 * kMB, &p) == Driver::kOutOfMemory && !p);
  fill();
  CHECK(c.pool_alloc(90 * kMB, Driver::kCapturing, &p) == Driver::kOutOfMemory);
  CHECK(Driver::idle_pool == 30 * kMB && Driver::used == 20 * kMB);  // nothing was touched
  return 0;
}

// Sizes that rounding up would wrap.
static int size_wraps() {
  Cache c;
  c.add_context(0, 64 * 100 * kMB);
  void* p = &c;
  for (size_t bytes : {SIZE_MAX, SIZE_MAX - 1, SIZE_MAX - 510}) {
    CHECK(c.alloc(bytes, &p) == Driver::kOutOfMemory && !p && Driver::mallocs == 0);
  }
  CHECK(c.alloc(SIZE_MAX - 511, &p) == Driver::kOutOfMemory && Driver::last_bytes == SIZE_MAX - 511);
  return 0;
}

int main(int, char** argv) {
#define RUN(f) if (!std::strcmp(argv[1], #f)) return f();
  RUN(freed_twice) RUN(foreign) RUN(sizes) RUN(limit) RUN(last_context) RUN(devices) RUN(waits) RUN(threads) RUN(out_of_memory) RUN(size_wraps)
  std::printf("no check %s\n", argv[1]);
  return 2;
}
"""
CHECKS = ("freed_twice", "foreign", "sizes", "limit", "last_context", "devices", "waits", "threads", "out_of_memory", "size_wraps")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("block_cache")
    (d / "check.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", str(ROOT / "matrixgraph_amd" / "csrc"), "check.cpp", "-o",
                    "check"], cwd=d, check=True)
    return d / "check"


@pytest.mark.parametrize("check", CHECKS)
def test_block_cache(program, check):
    r = subprocess.run([str(program), check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
