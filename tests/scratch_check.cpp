// Host driver for tests/test_scratch.py: the scratch pool (mpqc_amd/csrc/scratch.hpp) on a made-up
// device of 40 GiB that counts its allocations and refuses what does not fit.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <random>
#include <thread>

#include "../mpqc_amd/csrc/scratch.hpp"

namespace {
constexpr size_t kDevice = (size_t)40 << 30, GiB = (size_t)1 << 30;
std::mutex m;
std::map<void*, size_t> live;
size_t used = 0, next_address = 4096;
thread_local hipError_t last = hipSuccess;

void check(bool ok, const char* what) {
  std::printf("%s %s\n", ok ? "ok" : "FAILED", what);
  if (!ok) std::exit(1);
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(m);
  if (used + bytes > kDevice) return last = hipErrorOutOfMemory;
  *p = (void*)next_address;
  next_address += (bytes + 4095) / 4096 * 4096;
  live[*p] = bytes;
  used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(m);
  const auto it = live.find(p);
  if (it == live.end()) std::abort();  // freed twice, or never allocated
  used -= it->second;
  live.erase(it);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipMemGetInfo(size_t* free, size_t* total) {
  std::lock_guard<std::mutex> lk(m);
  *free = kDevice - used;
  *total = kDevice;
  return hipSuccess;
}
}

int main() {
  using namespace mpqc_hip;
  {
    auto a = std::make_unique<ScratchCache>();
    ScratchCache b;
    size_t got = 0;
    void* p = a->get(3 * GiB, &got);
    a->put(p, got);
    check(used == 3 * GiB, "a returned block is kept");
    check(device_available() == kDevice, "kept blocks count as available");
    void* q = b.get(3 * GiB, &got);
    check(q != p && used == 6 * GiB, "no other cache gets it");
    void* r = a->get(3 * GiB - (64 << 20), &got);
    check(r == p && got == 3 * GiB, "its own cache gets it for a request of about its size");
    a->put(r, got);
    b.put(q, 3 * GiB);
    check(used == 6 * GiB, "each cache keeps its own");
    p = a->get(2 * GiB, &got);
    a->put(p, got);
    check(used == 5 * GiB && device_available() == kDevice, "but at most 4 GiB");
    {
      std::vector<std::unique_ptr<ScratchCache>> many;
      for (int k = 0; k < 10; ++k) {
        many.push_back(std::make_unique<ScratchCache>());
        p = many.back()->get(4 * GiB, &got);
        many.back()->put(p, got);
      }
      check(used <= 32 * GiB && used >= 28 * GiB, "all caches together keep at most 32 GiB");
    }
    check(used == 0, "the longest-kept blocks made room");
    p = a->get(3 * GiB, &got);
    a->put(p, got);
    void* big = b.get(39 * GiB, &got);
    check(big && used == 39 * GiB, "an allocation gets what other caches keep before it fails");
    void* none = &got;
    check(device_malloc(&none, 2 * GiB) == hipErrorOutOfMemory && !none && hipGetLastError() == hipSuccess,
          "one that cannot fit fails and leaves no error behind");
    b.put(big, got);
    check(used == 0, "a block larger than the pool is not kept");
    p = a->get(GiB, &got);
    a->put(p, got);
    a->keep(false);
    check(used == 0, "keep(false) gives the kept blocks back");
    p = a->get(GiB, &got);
    a->put(p, got);
    check(used == 0, "and keeps no more");
    a->keep(true);
    p = a->get(GiB, &got);
    a->put(p, got);
    a.reset();
    check(used == 0, "a cache gives its blocks back with itself");
  }
  std::vector<std::thread> threads;
  for (int t = 0; t < 4; ++t)
    threads.emplace_back([t] {
      std::mt19937 rng(t);
      ScratchCache c;
      for (int k = 0; k < 2000; ++k) {
        std::vector<std::pair<void*, size_t>> held;
        for (int n = (int)(rng() % 4); n >= 0; --n) {
          size_t got = 0;
          try {
            void* p = c.get((size_t)(1 + rng() % 1000) << 20, &got);
            held.push_back({p, got});
          } catch (const std::bad_alloc&) {  // (four threads may want more than the device has)
          }
        }
        for (auto& h : held) c.put(h.first, h.second);
      }
    });
  for (auto& t : threads) t.join();
  check(used == 0 && live.empty() && ScratchPool::instance().kept == 0, "four threads leave nothing behind");
  return 0;
}
