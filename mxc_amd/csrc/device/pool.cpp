// The pools' bookkeeping. Host code alone, so that it is also built and tested
// without a GPU, against counting stand-ins for the runtime's calls.
#include "pool.hpp"

#include <iterator>
#include <mutex>

namespace mxg {

// What all pools keep, device by device, oldest first.
struct KeptBlocks {
  typedef std::multimap<size_t, DevPool::Block> Sizes;
  struct Device {
    size_t bytes = 0, most = 0;
    std::map<unsigned long long, std::pair<DevPool*, Sizes::iterator>> by_age;
  };
  std::mutex mu;
  std::map<int, Device> devices;
  unsigned long long age = 0;

  // never destroyed: buffers may be released while the process ends
  static KeptBlocks& get() {
    static KeptBlocks* k = new KeptBlocks;
    return *k;
  }

  // The rest with the lock held.

  void keep(DevPool* pool, void* p, size_t cap) {
    Device& d = devices[pool->device_];
    const unsigned long long a = age++;
    const auto it = pool->free_.emplace(cap, DevPool::Block{p, a});
    try {
      d.by_age.emplace(a, std::make_pair(pool, it));
    } catch (...) {
      pool->free_.erase(it);
      throw;
    }
    d.bytes += cap;
  }
  void* drop(DevPool* pool, Sizes::iterator it) {
    Device& d = devices[pool->device_];
    void* p = it->second.p;
    d.bytes -= it->first;
    d.by_age.erase(it->second.age);
    pool->free_.erase(it);
    return p;
  }
  void* drop_oldest(Device& d) {
    const auto& first = d.by_age.begin()->second;
    return drop(first.first, first.second);
  }
};

namespace {
// Frees one block after the other that next(), called with the lock held, gives
// up, until it gives none.
template <class Next>
void free_while(Next next) {
  KeptBlocks& K = KeptBlocks::get();
  for (;;) {
    void* p = nullptr;
    {
      std::lock_guard<std::mutex> lk(K.mu);
      p = next(K);
    }
    if (!p) return;
    (void)hipFree(p);
  }
}
}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || DevPool::kept_on(device) == 0) return e;
  (void)hipGetLastError();
  free_while([device](KeptBlocks& K) -> void* {
    KeptBlocks::Device& d = K.devices[device];
    return d.by_age.empty() ? nullptr : K.drop_oldest(d);
  });
  return hipMalloc(p, bytes);
}

DevPool::DevPool(int device) : device_(device) {
  size_t free_b = 0, total = 0;
  if (hipMemGetInfo(&free_b, &total) != hipSuccess) total = 0;
  KeptBlocks& K = KeptBlocks::get();
  std::lock_guard<std::mutex> lk(K.mu);
  K.devices[device].most = total / 32;
}

DevPool::~DevPool() {
  free_while([this](KeptBlocks& K) -> void* { return free_.empty() ? nullptr : K.drop(this, free_.begin()); });
}

void* DevPool::take(size_t bytes, size_t* cap) {
  // whole 512 bytes, above a megabyte whole 64 KB: arrays whose sizes differ
  // little from one object to the next share blocks
  const size_t unit = bytes > (size_t(1) << 20) ? size_t(65536) : size_t(512);
  const size_t need = (bytes + unit - 1) / unit * unit;
  {
    KeptBlocks& K = KeptBlocks::get();
    std::lock_guard<std::mutex> lk(K.mu);
    const auto it = free_.lower_bound(need);
    if (it != free_.end() && it->first <= need + need / 4 + 4096) {
      *cap = it->first;
      return K.drop(this, it);
    }
  }
  void* p = nullptr;
  const hipError_t e = device_malloc(&p, need);
  if (e != hipSuccess)
    throw Error(MXG_ERR_NOMEM, "hipMalloc of " + std::to_string(need) + " bytes failed: " + hipGetErrorString(e));
  *cap = need;
  return p;
}

void DevPool::give(void* p, size_t cap) noexcept {
  bool kept = false;
  try {
    KeptBlocks& K = KeptBlocks::get();
    std::lock_guard<std::mutex> lk(K.mu);
    if (cap <= K.devices[device_].most) {
      K.keep(this, p, cap);
      kept = true;
    }
  } catch (...) {  // no memory for the entry: the block goes
  }
  if (!kept) {
    (void)hipFree(p);
    return;
  }
  free_while([this](KeptBlocks& K) -> void* {
    KeptBlocks::Device& d = K.devices[device_];
    return d.bytes > d.most ? K.drop_oldest(d) : nullptr;
  });
}

size_t DevPool::kept_on(int device) {
  KeptBlocks& K = KeptBlocks::get();
  std::lock_guard<std::mutex> lk(K.mu);
  const auto it = K.devices.find(device);
  return it == K.devices.end() ? 0 : it->second.bytes;
}

std::shared_ptr<DevPool>& DevPool::current() {
  static thread_local std::shared_ptr<DevPool> p;
  return p;
}

}  // namespace mxg
