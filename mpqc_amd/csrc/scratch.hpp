// Device temporaries of a context's calls, kept between calls.
//
// The AO -> MO transform and the (T) correction need gigabytes of temporaries.
// hipMalloc and hipFree of blocks of that size map and unmap every page: 85 to 180 ms
// per transform call at 144 basis functions against 15 ms of kernels.  A context keeps
// the blocks its calls return, at most kKeep bytes of them, and all contexts of the process together
// at most kKeepAll.  It frees them with itself or when its option "keep_scratch" is set to 0, and every
// context's go back before an allocation of the library fails (device_malloc), whichever context
// or thread it is made for.  Every user of a block queues its work on its context's one stream, so that context may
// hand a block on while kernels still use it; no other one gets it, and hipFree waits for them.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <new>
#include <vector>

namespace mpqc_hip {

// The kept blocks of all contexts, the longest kept first.
struct ScratchPool {
  static constexpr size_t kKeep = (size_t)4 << 30, kKeepAll = (size_t)32 << 30;
  struct Block {
    const void* owner;
    void* p;
    size_t bytes;
  };
  std::mutex m;
  std::vector<Block> blocks;
  size_t kept = 0;

  static ScratchPool& instance() {
    static ScratchPool* const pool = new ScratchPool;  // (contexts may outlive static objects)
    return *pool;
  }

  // frees the blocks of `owner`, or everyone's (owner null); whether there was one
  bool release(const void* owner) {
    std::lock_guard<std::mutex> lk(m);
    const size_t before = blocks.size();
    for (size_t k = 0; k < blocks.size();)
      if (!owner || blocks[k].owner == owner) drop(k);
      else ++k;
    return blocks.size() != before;
  }

  void drop(size_t k) {  // (under the lock)
    (void)hipFree(blocks[k].p);
    kept -= blocks[k].bytes;
    blocks.erase(blocks.begin() + (long)k);
  }
};

// hipMalloc that gives the kept blocks back before it fails
inline hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (ScratchPool::instance().release(nullptr)) e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
  }
  return e;
}

// Bytes of the current device that an allocation can get: the free ones, and those kept above
// (so that a choice made by it does not depend on which calls came before).
inline size_t device_available() {
  size_t free = 0, total = 0;
  if (hipMemGetInfo(&free, &total) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  ScratchPool& pool = ScratchPool::instance();
  std::lock_guard<std::mutex> lk(pool.m);
  return free + pool.kept;
}

// One context's part of the pool.
class ScratchCache {
 public:
  ScratchCache() = default;
  ScratchCache(const ScratchCache&) = delete;
  ScratchCache& operator=(const ScratchCache&) = delete;
  ~ScratchCache() { clear(); }

  // at least `bytes` bytes; *got is the block's size (for put())
  void* get(size_t bytes, size_t* got) {
    bytes = std::max<size_t>(bytes, 256);
    {
      ScratchPool& pool = ScratchPool::instance();
      std::lock_guard<std::mutex> lk(pool.m);
      int best = -1;  // the smallest kept block that fits without wasting more than an eighth
      for (size_t k = 0; k < pool.blocks.size(); ++k) {
        const ScratchPool::Block& b = pool.blocks[k];
        if (b.owner == this && b.bytes >= bytes && b.bytes <= bytes + bytes / 8 + ((size_t)1 << 20) &&
            (best < 0 || b.bytes < pool.blocks[(size_t)best].bytes))
          best = (int)k;
      }
      if (best >= 0) {
        const ScratchPool::Block b = pool.blocks[(size_t)best];
        pool.blocks.erase(pool.blocks.begin() + best);
        pool.kept -= b.bytes;
        *got = b.bytes;
        return b.p;
      }
    }
    void* p = nullptr;
    if (device_malloc(&p, bytes) != hipSuccess) throw std::bad_alloc();
    *got = bytes;
    return p;
  }

  void put(void* p, size_t bytes) {
    if (!p) return;
    if (!keep_ || bytes > ScratchPool::kKeep) {
      (void)hipFree(p);
      return;
    }
    ScratchPool& pool = ScratchPool::instance();
    std::lock_guard<std::mutex> lk(pool.m);
    size_t mine = 0;
    for (const ScratchPool::Block& b : pool.blocks) mine += b.owner == this ? b.bytes : 0;
    for (size_t k = 0; mine + bytes > ScratchPool::kKeep;) {  // the longest-kept ones go first
      if (pool.blocks[k].owner == this) {
        mine -= pool.blocks[k].bytes;
        pool.drop(k);
      } else {
        ++k;
      }
    }
    while (pool.kept + bytes > ScratchPool::kKeepAll) pool.drop(0);
    pool.blocks.push_back({this, p, bytes});
    pool.kept += bytes;
  }

  void clear() { (void)ScratchPool::instance().release(this); }

  void keep(bool on) {
    keep_ = on;
    if (!on) clear();
  }

 private:
  bool keep_ = true;
};

// n doubles from a cache, returned to it on scope exit
struct ScratchBuf {
  double* p = nullptr;
  ScratchBuf(ScratchCache& c, size_t n) : cache_(c) {
    if (n) p = (double*)c.get(n * sizeof(double), &bytes_);
  }
  ~ScratchBuf() { cache_.put(p, bytes_); }
  ScratchBuf(const ScratchBuf&) = delete;
  ScratchBuf& operator=(const ScratchBuf&) = delete;

 private:
  ScratchCache& cache_;
  size_t bytes_ = 0;
};

}  // namespace mpqc_hip
