// Device memory of a context: the pool of its scene memory and build scratch, and
// the buffers that grow with its calls.  Host code only; no exception leaves it.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <new>
#include <vector>

// A block of at least `n` bytes that DevPool::take_all puts into *p.
struct PoolWant {
  void** p;
  size_t n;
};

// A context's scene memory and the scratch of its builds.  hipMalloc and
// hipFree of a scene's two dozen buffers took longer than building its trees
// (292k triangles: lisa_set_scene 4.2 ms, of which kernels and copies 1.5), and a
// program that loads or moves scenes on one context asks for the same sizes
// again: blocks go back to a list and are handed out to requests of at least
// half their size.  A block is only handed to work on the context's stream (or
// behind a copy that waits for it), so one that is given back while the stream
// still uses it is safe.  The list keeps at most kPoolFree bytes, makes room when an
// allocation of its context fails (dev_alloc), and is released with the context.
constexpr size_t kPoolFree = size_t{1} << 30;
struct DevPool {
  struct Block {
    void* p;
    size_t n;
  };
  std::vector<Block> idle, used;
  hipError_t take(void** p, size_t want) {
    *p = nullptr;
    want = (std::max<size_t>(want, 1) + 255) / 256 * 256;
    try {  // give() then needs no memory
      used.reserve(used.size() + 1);
      idle.reserve(idle.size() + used.size() + 1);
    } catch (const std::bad_alloc&) {
      return hipErrorOutOfMemory;
    }
    size_t best = idle.size();
    for (size_t i = 0; i < idle.size(); ++i)
      if (idle[i].n >= want && idle[i].n <= 2 * want + 65536 && (best == idle.size() || idle[i].n < idle[best].n))
        best = i;
    if (best < idle.size()) {
      used.push_back(idle[best]);
      idle.erase(idle.begin() + (long)best);
      *p = used.back().p;
      return hipSuccess;
    }
    hipError_t e = hipMalloc(p, want);
    if (e != hipSuccess && !idle.empty()) {
      (void)hipGetLastError();
      trim(0);
      e = hipMalloc(p, want);
    }
    if (e == hipSuccess)
      used.push_back(Block{*p, want});
    else
      *p = nullptr;
    return e;
  }
  // All of the blocks, or none of them and the error.
  hipError_t take_all(const PoolWant* wants, size_t n) {
    for (size_t i = 0; i < n; ++i) {
      const hipError_t e = take(wants[i].p, wants[i].n);
      if (e == hipSuccess) continue;
      (void)hipGetLastError();
      for (size_t k = 0; k < i; ++k) {
        give(*wants[k].p);
        *wants[k].p = nullptr;
      }
      return e;
    }
    return hipSuccess;
  }
  void give(void* p) noexcept {
    if (!p) return;
    for (size_t i = used.size(); i-- > 0;)
      if (used[i].p == p) {
        idle.push_back(used[i]);  // within the room that take() reserved
        used.erase(used.begin() + (long)i);
        return;
      }
  }
  void trim(size_t keep) noexcept {  // the largest idle blocks first
    size_t sum = 0;
    for (const Block& b : idle) sum += b.n;
    while (sum > keep) {
      size_t big = 0;
      for (size_t i = 1; i < idle.size(); ++i)
        if (idle[i].n > idle[big].n) big = i;
      sum -= idle[big].n;
      (void)hipFree(idle[big].p);
      idle.erase(idle.begin() + (long)big);
    }
  }
  void release() noexcept {
    trim(0);
    for (const Block& b : used) (void)hipFree(b.p);
    used.clear();
  }
};

// hipMalloc; where it fails, the idle blocks of the n pools are freed and it is tried
// again.
inline hipError_t dev_alloc(void** p, size_t bytes, DevPool* const* pools, size_t n) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  *p = nullptr;
  bool room = false;
  for (size_t i = 0; i < n; ++i) {
    room = room || !pools[i]->idle.empty();
    pools[i]->trim(0);
  }
  if (!room) return e;
  (void)hipGetLastError();
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) *p = nullptr;
  return e;
}

// Device buffer that only grows: reallocated when a call needs more.
template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t cap = 0;
  hipError_t ensure(size_t want, DevPool& pool) {
    if (p && want <= cap) return hipSuccess;
    (void)hipFree(p);
    p = nullptr;
    cap = 0;
    DevPool* const q = &pool;
    const hipError_t e = dev_alloc(reinterpret_cast<void**>(&p), std::max<size_t>(want, 1) * sizeof(T), &q, 1);
    if (e == hipSuccess) cap = want;
    return e;
  }
  void release() {
    (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
};

// Device scratch, given back to its pool at scope exit.
struct PoolScratch {
  DevPool& pool;
  std::vector<void*> ptrs;
  explicit PoolScratch(DevPool& p) : pool(p) {}
  PoolScratch(const PoolScratch&) = delete;
  PoolScratch& operator=(const PoolScratch&) = delete;
  ~PoolScratch() {
    for (void* p : ptrs) pool.give(p);
    pool.trim(kPoolFree);
  }
  template <typename T>
  hipError_t alloc(T** p, size_t count) {
    *p = nullptr;
    try {
      ptrs.reserve(ptrs.size() + 1);
    } catch (const std::bad_alloc&) {
      return hipErrorOutOfMemory;
    }
    void* q = nullptr;
    const hipError_t e = pool.take(&q, std::max<size_t>(count, 1) * sizeof(T));
    *p = static_cast<T*>(q);
    if (e == hipSuccess) ptrs.push_back(q);
    return e;
  }
};
