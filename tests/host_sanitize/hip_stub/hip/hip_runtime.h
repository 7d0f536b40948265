// hipMalloc and hipFree of a device with `hip_capacity` bytes, for tests of host code.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };

inline size_t hip_capacity = 0, hip_held = 0, hip_allocations = 0;
inline std::map<void *, size_t> hip_blocks;

inline hipError_t hipMalloc(void **p, size_t bytes) {
  if (hip_held + bytes > hip_capacity) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  hip_blocks[*p] = bytes;
  hip_held += bytes;
  ++hip_allocations;
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  const auto it = hip_blocks.find(p);
  if (it == hip_blocks.end()) std::abort();  // freed twice, or never allocated
  hip_held -= it->second;
  hip_blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
