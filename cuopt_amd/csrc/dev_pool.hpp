// dev_pool.hpp -- device memory kept from one solve for the next.
//
// Unmapping is what a solve's large arrays cost: hipFree of about 80 arrays took 7.1 ms of
// a 130 ms solve at 70 k x 1 M (2 M nonzeros), 12.2 ms of 105 ms at 1 M x 2 M (16 M).  With the
// store these solves went 130 -> 116 ms and 120 -> 106 ms, a skewed 500 k x 1 M one 197 -> 177 ms;
// at 2 000 x 5 000 no array is large enough.
//
// A solve takes its arrays of at least kPoolMin bytes through a lease.  Within the solve a
// released array goes back to the lease and may serve a later one: all of a solve's work
// is on one stream, so the order of the launches orders the uses too.  When the solve
// ends (its stream is idle) the lease hands its blocks to a process-wide store, which
// keeps at most kPoolCap bytes, the oldest freed first, and none that the last kPoolAge
// solves, batches among them, left unused; it is emptied by cuOptAmdReleaseMemory, when an
// allocation fails, and when a differentiable operator is made, whose program goes on with
// other work.  It outlives the handles: freeing with the last of them would only move the cost
// to a caller that makes its handles anew for each solve.  Contents are never reused:
// an array from the store is as undefined as one from hipMalloc.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <list>
#include <mutex>

namespace cuopt_amd {

constexpr size_t kPoolMin = 256 << 10;    // below it hipFree takes a few microseconds
constexpr size_t kPoolCap = 2ull << 30;   // under 1 % of the card's memory; 4 GiB was no faster at 1 M x 2 M
constexpr long kPoolAge   = 8;           // solves that an unused block is kept for

struct PoolBlock {
  void* p      = nullptr;
  size_t bytes = 0;
  int dev      = 0;
  long solve   = 0;  // the solve that gave it to the store
};

// Whether a block of `have` bytes may serve a request of `want`: at most a quarter is unused.
inline bool pool_fits(size_t have, size_t want) { return have >= want && have - want <= want / 4; }

// The smallest block of device dev that serves `bytes`, taken out of blocks; null if none does.
inline PoolBlock pool_take(std::list<PoolBlock>& blocks, size_t bytes, int dev)
{
  auto best = blocks.end();
  for (auto it = blocks.begin(); it != blocks.end(); ++it)
    if (it->dev == dev && pool_fits(it->bytes, bytes) && (best == blocks.end() || it->bytes < best->bytes)) best = it;
  if (best == blocks.end()) return PoolBlock{};
  const PoolBlock b = *best;
  blocks.erase(best);
  return b;
}

inline void pool_free(std::list<PoolBlock>& blocks)
{
  for (const PoolBlock& b : blocks) (void)hipFree(b.p);
  blocks.clear();
}

class PoolStore {
 public:
  // Never destroyed: at exit the HIP runtime may be gone first.
  static PoolStore& get()
  {
    static PoolStore* s = new PoolStore;
    return *s;
  }
  PoolBlock take(size_t bytes, int dev)
  {
    std::lock_guard<std::mutex> lock(mu_);
    const PoolBlock b = pool_take(blocks_, bytes, dev);
    held_ -= b.bytes;
    return b;
  }
  // Takes over the idle blocks of a lease.
  void give(std::list<PoolBlock>& blocks)
  {
    std::list<PoolBlock> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      ++solves_;
      for (PoolBlock& b : blocks) {
        held_ += b.bytes;
        b.solve = solves_;
      }
      blocks_.splice(blocks_.end(), blocks);
      while (!blocks_.empty() && (held_ > kPoolCap || blocks_.front().solve + kPoolAge < solves_)) {
        held_ -= blocks_.front().bytes;
        out.splice(out.end(), blocks_, blocks_.begin());
      }
    }
    pool_free(out);
  }
  // A batch solve, which takes its memory elsewhere, ages the blocks as a solve does.
  void age()
  {
    std::list<PoolBlock> none;
    give(none);
  }
  void trim()
  {
    std::list<PoolBlock> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      out.swap(blocks_);
      held_ = 0;
    }
    pool_free(out);
  }

 private:
  std::mutex mu_;
  std::list<PoolBlock> blocks_;  // oldest first
  size_t held_ = 0;
  long solves_ = 0;
};

// hipMalloc, tried again with an emptied store if it fails.  A failure is returned, not left
// for the next hipGetLastError: the caller may go on with less.
inline hipError_t pool_malloc(void** p, size_t bytes)
{
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    PoolStore::get().trim();
    e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();
  }
  return e;
}

// The blocks of one solve.  It outlives every array that took from it, and its stream is
// idle when it ends.
class PoolLease {
 public:
  explicit PoolLease(bool keep = true) : keep_(keep) {}
  PoolLease(const PoolLease&)            = delete;
  PoolLease& operator=(const PoolLease&) = delete;
  ~PoolLease()
  {
    if (keep_) PoolStore::get().give(free_);
    else pool_free(free_);
  }
  // After an error whose cause may still use the blocks, they are freed (which waits).
  void drop() { keep_ = false; }

  hipError_t alloc(size_t bytes, hipStream_t s, PoolBlock& b)
  {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    b = pool_take(free_, bytes, dev);
    if (!b.p) b = PoolStore::get().take(bytes, dev);
    if (b.p) return hipSuccess;
    b.bytes      = bytes;
    b.dev        = dev;
    hipError_t e = pool_malloc(&b.p, bytes);
    if (e == hipErrorOutOfMemory && !free_.empty()) {
      (void)hipGetLastError();
      (void)hipStreamSynchronize(s);
      pool_free(free_);
      e = hipMalloc(&b.p, bytes);
      if (e != hipSuccess) (void)hipGetLastError();
    }
    if (e != hipSuccess) b = PoolBlock{};
    return e;
  }
  void release(const PoolBlock& b) noexcept
  {
    try {
      free_.push_back(b);
    } catch (...) {
      (void)hipFree(b.p);
    }
  }

  // The lease from which this thread's arrays are taken.
  struct Current {
    PoolLease* lease   = nullptr;
    hipStream_t stream = nullptr;
  };
  static Current& current()
  {
    static thread_local Current c;
    return c;
  }
  class Scope {
   public:
    Scope(PoolLease& l, hipStream_t s) : saved_(current()) { current() = Current{&l, s}; }
    ~Scope() { current() = saved_; }
    Scope(const Scope&)            = delete;
    Scope& operator=(const Scope&) = delete;

   private:
    Current saved_;
  };

 private:
  std::list<PoolBlock> free_;
  bool keep_;
};

}  // namespace cuopt_amd
