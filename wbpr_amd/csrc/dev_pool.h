// Device memory of one context, kept for its next call.
//
// A one-shot solve allocates some thirty arrays, and hipFree waits for everything that runs on the
// device: a server's large requests, each with a context of its own, waited 25 to 40 ms each for
// one another's kernels and for the serving kernel.  Freed blocks of up to kMaxBlock bytes go to a
// list by size instead and are used again; at most `limit` bytes are kept, larger blocks and
// what is beyond the limit are given back at once, the rest with the context.  A context
// belongs to one host thread at a time, and its calls end with their stream idle: a block on the
// list has no work in flight.  The lock is for handles that another thread destroys (a garbage
// collector's), as hipFree allowed, also while a call on other handles of the context runs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace mf {

class DevPool {
 public:
  size_t limit = size_t(256) << 20;

  hipError_t alloc(void **p, size_t bytes) {
    const size_t size = rounded(bytes);
    std::lock_guard<std::mutex> lock(mutex_);
    auto it = kept_.find(size);
    if (it != kept_.end() && !it->second.empty()) {
      *p = it->second.back();
      it->second.pop_back();
      kept_bytes_ -= size;
      return hipSuccess;
    }
    hipError_t e = hipMalloc(p, size);
    if (e == hipErrorOutOfMemory && kept_bytes_ > 0) {
      (void)hipGetLastError();
      trim_locked();
      e = hipMalloc(p, size);
    }
    if (e == hipSuccess) size_[*p] = size;
    return e;
  }

  // p: from alloc, with no device work on it in flight.
  void release(void *p) {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto it = size_.find(p);
    if (it != size_.end() && it->second <= kMaxBlock && kept_bytes_ + it->second <= limit) {
      kept_[it->second].push_back(p);
      kept_bytes_ += it->second;
      return;
    }
    if (it != size_.end()) size_.erase(it);
    (void)hipFree(p);
  }

  void trim() {
    std::lock_guard<std::mutex> lock(mutex_);
    trim_locked();
  }

 private:
  void trim_locked() {
    for (auto &q : kept_)
      for (void *p : q.second) {
        size_.erase(p);
        (void)hipFree(p);
      }
    kept_.clear();
    kept_bytes_ = 0;
  }

  static constexpr size_t kMaxBlock = size_t(32) << 20;

  // Up to an eighth more, so that graphs of about one size share blocks.
  static size_t rounded(size_t bytes) {
    if (bytes > kMaxBlock) return bytes;
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
  }

  std::mutex mutex_;
  std::map<size_t, std::vector<void *>> kept_;
  std::unordered_map<void *, size_t> size_;
  size_t kept_bytes_ = 0;
};

}  // namespace mf
