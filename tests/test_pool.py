"""CPU: a context's memory pool (lisa_pool.h) over a counted device of 10,000
bytes: idle blocks make room where an allocation of the context fails, a set of
blocks is taken whole or not at all, host memory that runs out is an error code,
and everything is freed once."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "lisa_pool.h"
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <map>

static std::map<void*, size_t> live;
static size_t held = 0, calls = 0, last_errors = 0;
constexpr size_t kDevice = 10000;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  ++calls;
  if (held + n > kDevice) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  live[*p] = n;
  held += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  assert(live.count(p));  // freed once, and only what was given out
  held -= live[p];
  live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetLastError() { ++last_errors; return hipSuccess; }
}
static bool no_host_memory = false;
void* operator new(size_t n) {
  if (no_host_memory) throw std::bad_alloc();
  void* p = std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main() {
  DevPool pool, other;
  DevPool* const pools[2] = {&pool, &other};
  void *a = nullptr, *b = nullptr, *c = nullptr;

  // blocks come back to requests of at least half their size
  assert(pool.take(&a, 4096) == hipSuccess && held == 4096);
  pool.give(a);
  assert(pool.take(&b, 3000) == hipSuccess && b == a && calls == 1);
  pool.give(b);

  // a growing buffer's allocation fails while the pool holds idle memory: it makes room
  DevBuf<char> buf;
  assert(buf.ensure(9000, pool) == hipSuccess && buf.p && buf.cap == 9000 && held == 9000 && pool.idle.empty());
  assert(last_errors > 0);
  assert(buf.ensure(8000, pool) == hipSuccess && held == 9000);  // grown once
  assert(buf.ensure(20000, pool) == hipErrorOutOfMemory && !buf.p && buf.cap == 0 && held == 0);

  // so do the pools of a batch's contexts
  assert(pool.take(&a, 2560) == hipSuccess && other.take(&b, 5120) == hipSuccess);
  pool.give(a);
  other.give(b);
  assert(dev_alloc(&c, 9000, pools, 2) == hipSuccess && held == 9000);
  assert(hipFree(c) == hipSuccess);
  c = &c;
  assert(dev_alloc(&c, 20000, pools, 2) == hipErrorOutOfMemory && c == nullptr);

  // all blocks of a set or none
  assert(pool.take(&a, 1024) == hipSuccess);
  void *x = &x, *y = &y, *z = &z;
  const PoolWant too_much[3] = {{&x, 2048}, {&y, 4096}, {&z, 4096}};
  assert(pool.take_all(too_much, 3) == hipErrorOutOfMemory && !x && !y && !z);
  assert(pool.used.size() == 1 && pool.used[0].p == a);
  const PoolWant fits[2] = {{&x, 2048}, {&y, 4096}};
  assert(pool.take_all(fits, 2) == hipSuccess && x && y && pool.used.size() == 3);

  // no host memory: an error from take, nothing thrown by give
  pool.used.shrink_to_fit();
  pool.idle.shrink_to_fit();
  no_host_memory = true;
  z = &z;
  const size_t before = held;
  assert(pool.take(&z, 256) == hipErrorOutOfMemory && !z && held == before);
  no_host_memory = false;
  assert(pool.take(&z, 256) == hipSuccess);
  no_host_memory = true;
  pool.give(a);
  pool.give(x);
  pool.give(y);
  pool.give(z);
  pool.give(nullptr);
  {
    PoolScratch S(pool);
    char* s = nullptr;
    assert(S.alloc(&s, 10) == hipErrorOutOfMemory && !s);
  }
  no_host_memory = false;
  assert(pool.used.empty() && pool.idle.size() == 4);

  // scratch goes back at scope exit; the least that goes over `keep` is freed, largest first
  {
    PoolScratch S(pool);
    float* s = nullptr;
    assert(S.alloc(&s, 512) == hipSuccess && s && pool.used.size() == 1);
  }
  assert(pool.used.empty());
  pool.trim(2000);
  size_t sum = 0;
  for (auto& k : pool.idle) sum += k.n;
  assert(sum <= 2000 && sum > 0 && sum == held);
  assert(pool.take(&a, 1) == hipSuccess);
  pool.release();
  other.release();
  assert(held == 0 && live.empty());
  std::puts("OK");
}
"""


HIP = """#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
extern "C" hipError_t hipMalloc(void** p, size_t n);
extern "C" hipError_t hipFree(void* p);
extern "C" hipError_t hipGetLastError();
"""


def test_pool(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime_api.h").write_text(HIP)
    src, exe = tmp_path / "pool.cpp", str(tmp_path / "pool")
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "lisa_amd", "csrc"), str(src), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout.strip() == "OK", res.stderr
