// Device memory of a context, kept for its later buffers.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>

#include "mxc_gpu.h"

namespace mxg {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

// hipMalloc on the current device; when it fails, once more after the device's
// pools have given their kept blocks back to the runtime.
hipError_t device_malloc(void** p, size_t bytes);

// A factorization or a level's construction allocates and frees 50 to 500 arrays,
// and hipFree alone (which waits for the device) took 13 of the 54 ms of a
// preconditioner set-up at N = 32768 and 8 of the 22.5 ms of a factorization at N =
// 131072.
//
// Blocks go back to the context they came from and every use of them is ordered
// by that context's stream, so a block may be handed out again while the kernels
// that used it last are still queued. The pools of a device keep at most a
// thirty-second of its memory between them; beyond that the blocks kept longest go,
// whichever pool has them (with the newest ones going instead, what an earlier,
// larger object had left filled the pools for good: a factorization at N = 131072
// took 38 ms instead of 10 after ten other problems). Kept blocks are given back
// when the context goes, and when any allocation of this library on the device
// fails. hipFree is never called with a lock held: it waits for the device, and a
// context that is being made or another thread's allocation would wait with it.
class DevPool {
 public:
  explicit DevPool(int device);
  ~DevPool();
  DevPool(const DevPool&) = delete;
  DevPool& operator=(const DevPool&) = delete;
  // at least `bytes` bytes; *cap receives the block's size
  void* take(size_t bytes, size_t* cap);
  void give(void* p, size_t cap) noexcept;
  // bytes kept for reuse by the pools of a device
  static size_t kept_on(int device);
  // the pool the calling thread's buffers come from (set by PoolScope)
  static std::shared_ptr<DevPool>& current();

 private:
  friend struct KeptBlocks;
  struct Block {
    void* p;
    unsigned long long age;
  };
  const int device_;
  std::multimap<size_t, Block> free_;  // by size; under the lock of all pools
};

// Buffers allocated by this thread within the scope come from the pool.
struct PoolScope {
  std::shared_ptr<DevPool> before;
  explicit PoolScope(const std::shared_ptr<DevPool>& p) : before(DevPool::current()) { DevPool::current() = p; }
  ~PoolScope() { DevPool::current() = before; }
  PoolScope(const PoolScope&) = delete;
  PoolScope& operator=(const PoolScope&) = delete;
};

}  // namespace mxg
