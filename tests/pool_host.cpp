// The device layer's memory pools (pool.cpp) and stream forks (fork.hpp) against
// counting stand-ins for the runtime's calls: pool_host CASE exits 0 when the case
// holds.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <random>
#include <thread>
#include <vector>

#include "fork.hpp"
#include "pool.hpp"

using mxg::DevPool;

namespace {
std::mutex mu;
std::map<void*, std::pair<int, size_t>> live;  // device and size of the blocks the stand-in has handed out
std::map<int, size_t> used;
size_t capacity = size_t(1) << 40;             // of a device
constexpr size_t TOTAL = size_t(1) << 20;      // the device memory that hipMemGetInfo reports: pools keep 32 KB
thread_local int device = 0;
std::string events;                            // the event calls so far
std::function<void()> on_free;                 // called within hipFree

void check(bool ok, const char* what) {
  if (ok) return;
  std::fprintf(stderr, "failed: %s\n", what);
  std::fflush(stderr);
  std::_Exit(1);
}
size_t blocks_on(int d) {
  std::lock_guard<std::mutex> lk(mu);
  size_t n = 0;
  for (auto& b : live) n += b.second.first == d;
  return n;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  if (used[device] + bytes > capacity) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  live[*p] = {device, bytes};
  used[device] += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (on_free) on_free();
  std::lock_guard<std::mutex> lk(mu);
  const auto it = live.find(p);
  check(it != live.end(), "a block freed twice, or never handed out");
  used[it->second.first] -= it->second.second;
  live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = device == 2 ? 4 * TOTAL : TOTAL;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  events += "record " + std::to_string((size_t)e) + " on " + std::to_string((size_t)s) + ";";
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  events += std::to_string((size_t)s) + " waits for " + std::to_string((size_t)e) + ";";
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
}

namespace {
void* take(DevPool& p, size_t bytes, size_t* cap) { return p.take(bytes, cap); }

// Blocks come back, the smallest that fits; more than a quarter too large does not.
void reuse() {
  DevPool p(0);
  size_t ca, cb, c;
  void *a = take(p, 1000, &ca), *b = take(p, 9000, &cb);
  check(ca == 1024 && cb == 9216, "sizes in units");
  p.give(a, ca);
  p.give(b, cb);
  check(DevPool::kept_on(0) == ca + cb, "bytes kept");
  check(take(p, 600, &c) == a && c == ca, "the smallest block that fits");
  void* d = take(p, 600, &c);
  check(d != b && c == 1024, "a block far too large stays");
  check(take(p, 9001, &c) == b, "the block of the size");
  p.give(a, ca);
  p.give(b, cb);
  p.give(d, 1024);
}

// Beyond a thirty-second of the device's memory the blocks kept longest go, whichever pool has them.
void oldest_go() {
  DevPool p(0), q(0);
  size_t c;
  std::vector<void*> v;
  for (int i = 0; i < 10; i++) v.push_back(take(i % 2 ? p : q, 4096, &c));
  for (int i = 0; i < 10; i++) (i % 2 ? p : q).give(v[i], 4096);
  check(DevPool::kept_on(0) == 32768 && blocks_on(0) == 8, "eight blocks kept");
  {
    std::lock_guard<std::mutex> lk(mu);
    check(!live.count(v[0]) && !live.count(v[1]) && live.count(v[2]) && live.count(v[9]), "the oldest two went");
  }
  size_t big;
  void* w = take(p, 40000, &big);
  p.give(w, big);
  check(DevPool::kept_on(0) == 32768 && blocks_on(0) == 8, "a block beyond the limit is not kept");
}

// A failed allocation gives the device's kept blocks back and is tried again.
void failing_allocation() {
  DevPool p(0);
  size_t c;
  void* a = take(p, 16384, &c);
  p.give(a, c);
  capacity = 20000;
  void* b = nullptr;
  check(mxg::device_malloc(&b, 18000) == hipSuccess && DevPool::kept_on(0) == 0, "tried again without the kept blocks");
  bool thrown = false;
  try {
    (void)take(p, 18000, &c);
  } catch (const mxg::Error& e) {
    thrown = e.code == MXG_ERR_NOMEM;
  }
  check(thrown, "an error when it does not fit then either");
  (void)hipFree(b);
}

// hipFree is called with no lock held: other threads make contexts and take blocks meanwhile.
void free_without_locks() {
  DevPool p(0);
  size_t c;
  std::vector<void*> v;
  for (int i = 0; i < 12; i++) v.push_back(take(p, 4096, &c));
  int calls = 0;
  on_free = [&] {
    calls++;
    auto done = std::make_shared<std::atomic<bool>>(false);
    std::thread([done, &p] {
      { DevPool other(0); }
      (void)DevPool::kept_on(0);
      (void)p;
      *done = true;
    }).detach();
    for (int i = 0; i < 200 && !*done; i++) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    check(*done, "another thread's context waited for hipFree");
  };
  for (void* b : v) p.give(b, 4096);  // the last four make older ones go
  check(calls == 4, "blocks went while others were given");
  capacity = 0;
  void* b = nullptr;
  check(mxg::device_malloc(&b, 1) != hipSuccess && calls == 12, "the rest for a failing allocation");
  capacity = size_t(1) << 40;
  {
    DevPool q(0);
    void* x = take(q, 512, &c);
    q.give(x, c);
  }
  check(calls == 13, "and at the end of a pool");
  on_free = nullptr;
}

// Each device has its limit, and its pools do not make room for another's.
void per_device() {
  auto on = [](int d) {
    device = d;
    return std::make_unique<DevPool>(d);
  };
  auto p2 = on(2), p0 = on(0), p1 = on(1);
  size_t c;
  auto fill = [&](DevPool& p, int d, int n) {
    device = d;
    std::vector<void*> v;
    for (int i = 0; i < n; i++) v.push_back(take(p, 4096, &c));
    for (void* b : v) p.give(b, 4096);
  };
  fill(*p0, 0, 8);
  check(DevPool::kept_on(0) == 32768, "device 0 full");
  fill(*p1, 1, 8);
  check(DevPool::kept_on(0) == 32768 && DevPool::kept_on(1) == 32768, "device 1 full, device 0 as it was");
  fill(*p2, 2, 20);
  check(DevPool::kept_on(2) == 20 * 4096, "a larger device keeps more");
  device = 1;
  capacity = 32768 + 100;
  void* b = nullptr;
  check(mxg::device_malloc(&b, 20000) == hipSuccess, "room on device 1");
  check(DevPool::kept_on(1) == 0 && DevPool::kept_on(0) == 32768, "made by device 1 alone");
  (void)hipFree(b);
}

// Contexts at work, made and gone in several threads.
void threads() {
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; t++)
    ts.emplace_back([t] {
      device = t % 2;
      std::mt19937 rng(t);
      for (int round = 0; round < 40; round++) {
        auto p = std::make_shared<DevPool>(device);
        mxg::PoolScope scope(p);
        std::vector<std::pair<void*, size_t>> v;
        for (int i = 0; i < 60; i++) {
          if (v.size() < 4 || rng() % 2) {
            size_t c;
            void* b = DevPool::current()->take(1 + rng() % 9000, &c);
            v.push_back({b, c});
          } else {
            std::swap(v[rng() % v.size()], v.back());
            p->give(v.back().first, v.back().second);
            v.pop_back();
          }
        }
        for (auto& b : v) p->give(b.first, b.second);
      }
    });
  for (auto& t : ts) t.join();
  check(live.empty() && DevPool::kept_on(0) == 0 && DevPool::kept_on(1) == 0, "everything given back");
}

// The first stream (1) waits for the second (2) once, also when the work in between ends in an error.
void forks() {
  const auto first = (hipStream_t)1, second = (hipStream_t)2;
  const auto fork = (hipEvent_t)3, join = (hipEvent_t)4;
  const std::string begin = "record 3 on 1;2 waits for 3;", end = "record 4 on 2;1 waits for 4;";
  for (int stop = 0; stop < 3; stop++) {  // at the second stream's work, after it, not at all
    events.clear();
    try {
      mxg::Fork f(first, second, fork, join);
      if (stop == 0) throw 0;
      f.done();
      if (stop == 1) throw 0;
      f.wait();
    } catch (int) {
    }
    check(events == begin + end, events.c_str());
  }
}
}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> cases{{"reuse", reuse}, {"oldest_go", oldest_go},
                                                {"failing_allocation", failing_allocation},
                                                {"free_without_locks", free_without_locks},
                                                {"per_device", per_device}, {"threads", threads},
                                                {"forks", forks}};
  check(argc == 2 && cases.count(argv[1]), "a case by name");
  cases.at(argv[1])();
  std::lock_guard<std::mutex> lk(mu);
  check(live.empty(), "every block given back at the end");
  return 0;
}
