// Device memory of one context, kept for its next call.
//
// A one-shot solve allocates some thirty arrays, and hipFree waits for everything that runs on the
// device: a server's large requests, each with a context of its own, waited 25 to 40 ms each for
// one another's kernels and for the serving kernel.  Freed blocks of up to max_block bytes go to a
// list by size instead and are used again, by arrays of up to an eighth less.  The memory beyond what
// the arrays in use need -- blocks on the list, and the ends of larger blocks in use -- stays within
// the limit; what does not is given back at once, the rest with the context, or when an allocation
// fails: then every context of the process gives its list back first.  A context
// belongs to one host thread at a time, and its calls end with their stream idle: a block on the
// list has no work in flight.  The lock is for handles that another thread destroys (a garbage
// collector's), as hipFree allowed, also while a call on other handles of the context runs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <map>
#include <mutex>
#include <set>
#include <unordered_map>
#include <vector>

namespace mf {

class DevPool {
 public:
  DevPool() {
    std::lock_guard<std::mutex> lock(registry().mutex);
    registry().pools.insert(this);
  }
  ~DevPool() {
    std::lock_guard<std::mutex> lock(registry().mutex);
    registry().pools.erase(this);
  }
  DevPool(const DevPool &) = delete;
  DevPool &operator=(const DevPool &) = delete;

  hipError_t alloc(void **p, size_t bytes) {
    const size_t need = (bytes + 511) / 512 * 512;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = kept_.lower_bound(need);
      if (it != kept_.end() && it->first <= need + need / 8) {
        *p = it->second;
        used_[*p] = Block{it->first, need};
        spare_ -= need;
        kept_.erase(it);
        return hipSuccess;
      }
    }
    hipError_t e = hipMalloc(p, need);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      trim_all();
      e = hipMalloc(p, need);
    }
    if (e == hipSuccess) {
      std::lock_guard<std::mutex> lock(mutex_);
      used_[*p] = Block{need, need};
    }
    return e;
  }

  // p: from alloc, with no device work on it in flight.
  void release(void *p) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = used_.find(p);
      if (it != used_.end()) {
        const Block b = it->second;
        used_.erase(it);
        if (b.size <= max_block_ && spare_ + b.need <= limit_) {
          kept_.emplace(b.size, p);
          spare_ += b.need;
          return;
        }
        spare_ -= b.size - b.need;
      }
    }
    (void)hipFree(p);
  }

  // The largest blocks go first.
  void set_limit(size_t limit, size_t max_block) {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      limit_ = limit;
      max_block_ = max_block;
      while (!kept_.empty() && (spare_ > limit_ || std::prev(kept_.end())->first > max_block_)) {
        const auto it = std::prev(kept_.end());
        out.push_back(it->second);
        spare_ -= it->first;
        kept_.erase(it);
      }
    }
    for (void *p : out) (void)hipFree(p);
  }

  void trim() {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (const auto &b : kept_) {
        out.push_back(b.second);
        spare_ -= b.first;
      }
      kept_.clear();
    }
    for (void *p : out) (void)hipFree(p);
  }

 private:
  struct Block {
    size_t size, need;
  };
  struct Registry {
    std::mutex mutex;
    std::set<DevPool *> pools;
  };
  static Registry &registry() {
    static Registry *r = new Registry;  // (outlives every context)
    return *r;
  }
  static void trim_all() {
    std::lock_guard<std::mutex> lock(registry().mutex);
    for (DevPool *q : registry().pools) q->trim();
  }

  std::mutex mutex_;
  std::multimap<size_t, void *> kept_;        // by size
  std::unordered_map<void *, Block> used_;
  size_t spare_ = 0;  // bytes held and not needed
  size_t limit_ = size_t(256) << 20;
  size_t max_block_ = size_t(32) << 20;
};

}  // namespace mf
