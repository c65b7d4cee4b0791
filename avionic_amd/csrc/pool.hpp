// Device memory kept between reconstructions.
//
// A reconstruction needs one block of device memory for its state; hipMalloc and
// hipFree of a dozen buffers cost more than a hundred small iterations (and
// hipFree waits for the device).  Blocks that are given back are kept, at most
// kPoolBytes per process, and handed to the next request of a like size on the
// same device.  They go back to the device when the last solver or engine is
// destroyed, when the bound is passed (oldest first), when an allocation of the
// library fails, and on request (avionic_release_memory).  Thread-safe; whoever gives a block back has waited for the streams
// that use it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace avionic {

constexpr size_t kPoolBytes = size_t(4) << 30;

// A block of the pool, or none.  Move-only; give() or the destructor returns it.
class PoolBlock {
 public:
  PoolBlock() = default;
  // Throws when the device has no such memory.  A kept block is taken when it is
  // at most `waste` bytes larger; for a new one the pool first frees kept blocks
  // down to `keep` bytes.
  explicit PoolBlock(size_t bytes) : PoolBlock(bytes, bytes / 2, kPoolBytes) {}
  PoolBlock(size_t bytes, size_t waste, size_t keep);
  PoolBlock(PoolBlock &&o) noexcept;
  PoolBlock &operator=(PoolBlock &&o) noexcept;
  ~PoolBlock() { give(); }
  void give();
  void *p = nullptr;
  size_t bytes = 0;  // at least the size asked for
  int dev = 0;
};

// hipMalloc (stream: hipMallocAsync on it) that empties the pool and tries again
// when memory runs out; every device allocation of the library goes through them.
void *device_alloc(size_t bytes);
void *device_alloc_async(size_t bytes, hipStream_t stream);

// Owners of blocks: the pool is emptied when the last one ends.
struct PoolUser {
  PoolUser();
  ~PoolUser();
  PoolUser(const PoolUser &) = delete;
  PoolUser &operator=(const PoolUser &) = delete;
};
size_t pooled_bytes();
// Frees kept blocks, oldest first, until at most `most` bytes are kept.
void trim_pool(size_t most);

// Part of a block.
struct DevView {
  void *p = nullptr;
  size_t bytes = 0;
  template <typename T>
  T *as() const { return (T *)p; }
};
// Sizes collected first, then one block cut into 256-byte aligned parts.
struct PoolLayout {
  static constexpr int kMost = 20;
  DevView *view[kMost];
  int n = 0;
  size_t total = 0;
  void add(DevView &v, size_t bytes) {
    v.bytes = bytes;
    view[n++] = &v;
    total += (bytes + 255) / 256 * 256;
  }
  void cut(const PoolBlock &b) {
    char *p = (char *)b.p;
    for (int i = 0; i < n; ++i) {
      view[i]->p = p;
      p += (view[i]->bytes + 255) / 256 * 256;
    }
  }
};

}  // namespace avionic
