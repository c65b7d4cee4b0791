#include "pool.hpp"

#include <hip/hip_runtime.h>

#include <deque>
#include <mutex>
#include <new>
#include <string>

#include "common.hpp"

namespace avionic {

namespace {

struct Kept {
  void *p;
  size_t bytes;
  int dev;
};
struct Pool {
  std::mutex mu;
  std::deque<Kept> kept;  // oldest first
  size_t bytes = 0;
  int users = 0;
};
// Never destroyed: blocks may be given back after static destruction began.
Pool &pool() {
  static Pool *p = new Pool;
  return *p;
}
void trim_locked(Pool &g, size_t most) {
  while (g.bytes > most) {
    const Kept k = g.kept.front();
    g.kept.pop_front();
    g.bytes -= k.bytes;
    (void)hipFree(k.p);
  }
}

}  // namespace

void trim_pool(size_t most) {
  Pool &g = pool();
  std::lock_guard<std::mutex> lock(g.mu);
  trim_locked(g, most);
}

size_t pooled_bytes() {
  Pool &g = pool();
  std::lock_guard<std::mutex> lock(g.mu);
  return g.bytes;
}

template <class F>
static void *alloc_or_trim(size_t bytes, F &&alloc) {
  void *p = nullptr;
  hipError_t e = alloc(&p);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    trim_pool(0);
    e = alloc(&p);
  }
  if (e != hipSuccess)
    throw Error(-2, "device allocation of " + std::to_string(bytes) + " bytes: " + hipGetErrorString(e));
  return p;
}
void *device_alloc(size_t bytes) {
  return alloc_or_trim(bytes, [&](void **p) { return hipMalloc(p, bytes); });
}
void *device_alloc_async(size_t bytes, hipStream_t s) {
  return alloc_or_trim(bytes, [&](void **p) { return hipMallocAsync(p, bytes, s); });
}

PoolBlock::PoolBlock(size_t need, size_t waste, size_t keep) {
  AV_HIP(hipGetDevice(&dev));
  need = need > 0 ? need : 256;
  {
    // the smallest kept block that is large enough
    Pool &g = pool();
    std::lock_guard<std::mutex> lock(g.mu);
    auto best = g.kept.end();
    for (auto it = g.kept.begin(); it != g.kept.end(); ++it)
      if (it->dev == dev && it->bytes >= need && it->bytes - need <= waste &&
          (best == g.kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != g.kept.end()) {
      p = best->p;
      bytes = best->bytes;
      g.bytes -= bytes;
      g.kept.erase(best);
      return;
    }
    trim_locked(g, keep);
  }
  p = device_alloc(need);
  bytes = need;
}

PoolBlock::PoolBlock(PoolBlock &&o) noexcept : p(o.p), bytes(o.bytes), dev(o.dev) { o.p = nullptr; }
PoolBlock &PoolBlock::operator=(PoolBlock &&o) noexcept {
  if (this != &o) {
    give();
    p = o.p;
    bytes = o.bytes;
    dev = o.dev;
    o.p = nullptr;
  }
  return *this;
}

void PoolBlock::give() {
  if (!p) return;
  Pool &g = pool();
  std::lock_guard<std::mutex> lock(g.mu);
  bool keep = g.users > 0 && bytes <= kPoolBytes;
  if (keep) {
    trim_locked(g, kPoolBytes - bytes);
    try {
      g.kept.push_back(Kept{p, bytes, dev});
      g.bytes += bytes;
    } catch (const std::bad_alloc &) {  // this runs in destructors
      keep = false;
    }
  }
  if (!keep) (void)hipFree(p);
  p = nullptr;
}

PoolUser::PoolUser() {
  Pool &g = pool();
  std::lock_guard<std::mutex> lock(g.mu);
  ++g.users;
}
PoolUser::~PoolUser() {
  Pool &g = pool();
  std::lock_guard<std::mutex> lock(g.mu);
  if (--g.users == 0) trim_locked(g, 0);
}

}  // namespace avionic
