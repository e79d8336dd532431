// Device temporaries of a context's calls, kept between calls.
//
// The AO -> MO transform and the (T) correction need gigabytes of temporaries.
// hipMalloc and hipFree of blocks of that size map and unmap every page: 85 to 180 ms
// per transform call at 144 basis functions against 15 ms of kernels.  A context keeps
// the blocks its calls return, at most kKeep bytes of them, and frees them with itself, or
// when one of its allocations would fail otherwise.  Every user of a block queues its work on the
// context's one stream, so a block may be handed on while kernels still use it.
#pragma once

#include <algorithm>
#include <new>
#include <vector>

#include "common.hpp"

namespace mpqc_hip {

class ScratchCache {
 public:
  static constexpr size_t kKeep = (size_t)4 << 30;
  ScratchCache() = default;
  ScratchCache(const ScratchCache&) = delete;
  ScratchCache& operator=(const ScratchCache&) = delete;
  ~ScratchCache() { clear(); }

  // at least `bytes` bytes; *got is the block's size (for put())
  void* get(size_t bytes, size_t* got) {
    bytes = std::max<size_t>(bytes, 256);
    int best = -1;  // the smallest kept block that fits without wasting more than an eighth
    for (size_t k = 0; k < free_.size(); ++k)
      if (free_[k].bytes >= bytes && free_[k].bytes <= bytes + bytes / 8 + ((size_t)1 << 20) &&
          (best < 0 || free_[k].bytes < free_[(size_t)best].bytes))
        best = (int)k;
    if (best >= 0) {
      const Block b = free_[(size_t)best];
      free_.erase(free_.begin() + best);
      kept_ -= b.bytes;
      *got = b.bytes;
      return b.p;
    }
    void* p = nullptr;
    if (allocate(&p, bytes) != hipSuccess) throw std::bad_alloc();
    *got = bytes;
    return p;
  }

  void put(void* p, size_t bytes) {
    if (!p) return;
    if (bytes > kKeep) {
      (void)hipFree(p);
      return;
    }
    while (kept_ + bytes > kKeep) {  // the longest-kept block goes first
      (void)hipFree(free_.front().p);
      kept_ -= free_.front().bytes;
      free_.erase(free_.begin());
    }
    free_.push_back({p, bytes});
    kept_ += bytes;
  }

  // hipMalloc that gives the kept blocks back before it fails
  hipError_t allocate(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess && !free_.empty()) {
      (void)hipGetLastError();
      clear();
      e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      *p = nullptr;
    }
    return e;
  }

  void clear() {
    for (const Block& b : free_) (void)hipFree(b.p);
    free_.clear();
    kept_ = 0;
  }

 private:
  struct Block {
    void* p;
    size_t bytes;
  };
  std::vector<Block> free_;
  size_t kept_ = 0;
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
