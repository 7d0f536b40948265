// Device memory of one context, kept for its next call.
//
// A one-shot solve allocates some thirty arrays, and hipFree waits for everything that runs on the
// device: a server's large requests, each with a context of its own, waited 25 to 40 ms each for
// one another's kernels and for the serving kernel.  Freed blocks of up to max_block bytes go to a
// list by size instead and are used again, by arrays of up to an eighth less.  The memory beyond what
// the arrays in use need -- blocks on the list, and the ends of larger blocks in use -- stays within
// the limit: the blocks longest on the list are given back for a new one, the rest with the context,
// or when an allocation fails: then every context of the process gives its list back first.  A context
// belongs to one host thread at a time, and its calls end with their stream idle: a block on the
// list has no work in flight.  The lock is for handles that another thread destroys (a garbage
// collector's), as hipFree allowed, also while a call on other handles of the context runs.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
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
      for (auto it = kept_.lower_bound(need); it != kept_.end() && it->first <= need + need / 8; ++it) {
        if (it->second.empty()) continue;
        *p = it->second.back();
        it->second.pop_back();
        blocks_[*p].need = need;
        spare_ -= need;
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
      blocks_[*p] = Block{need, need, 0};
    }
    return e;
  }

  // p: from alloc, with no device work on it in flight.
  void release(void *p) {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = blocks_.find(p);
      if (it == blocks_.end()) {
        out.push_back(p);
      } else {
        Block &b = it->second;
        spare_ += b.need;
        b.released = ++releases_;
        kept_[b.size].push_back(p);
        if (b.size > max_block_ || b.need > limit_) give_back(kept_.find(b.size), p, out);
        shrink(out);
      }
    }
    for (void *x : out) (void)hipFree(x);
  }

  void set_limit(size_t limit, size_t max_block) {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      limit_ = limit;
      max_block_ = max_block;
      for (auto it = kept_.upper_bound(max_block_); it != kept_.end(); ++it)
        while (!it->second.empty()) give_back(it, it->second.back(), out);
      shrink(out);
    }
    for (void *p : out) (void)hipFree(p);
  }

  void trim() {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (auto it = kept_.begin(); it != kept_.end(); ++it)
        while (!it->second.empty()) give_back(it, it->second.back(), out);
      kept_.clear();
    }
    for (void *p : out) (void)hipFree(p);
  }

 private:
  struct Block {
    size_t size, need;
    unsigned long long released;  // when it went to the list
  };
  using Kept = std::map<size_t, std::vector<void *>>;

  // Takes p off the list (lock held).
  void give_back(Kept::iterator it, void *p, std::vector<void *> &out) {
    std::vector<void *> &v = it->second;
    v.erase(std::find(v.begin(), v.end(), p));
    spare_ -= it->first;
    blocks_.erase(p);
    out.push_back(p);
  }

  // Gives the oldest blocks back until the limit holds, or none is left (lock held).
  void shrink(std::vector<void *> &out) {
    while (spare_ > limit_) {
      auto oldest = kept_.end();
      void *p = nullptr;
      unsigned long long when = ~0ull;
      for (auto it = kept_.begin(); it != kept_.end(); ++it)
        for (void *x : it->second)
          if (blocks_[x].released < when) {
            when = blocks_[x].released;
            oldest = it;
            p = x;
          }
      if (!p) return;
      give_back(oldest, p, out);
    }
  }

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
  Kept kept_;                                // by size
  std::unordered_map<void *, Block> blocks_;  // every block, in use or kept
  size_t spare_ = 0;                         // bytes held and not needed
  unsigned long long releases_ = 0;
  size_t limit_ = size_t(256) << 20;
  size_t max_block_ = size_t(32) << 20;
};

}  // namespace mf
