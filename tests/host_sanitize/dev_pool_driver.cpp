// The block list of a context (wbpr_amd/csrc/dev_pool.h) on a device of hip_stub's.
#include "../../wbpr_amd/csrc/dev_pool.h"

#include <cstdio>
#include <random>
#include <vector>

#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) {                                              \
      std::printf("line %d: %s\n", __LINE__, #x);            \
      return 1;                                              \
    }                                                        \
  } while (0)

static int random_calls(size_t limit, size_t max_block, unsigned seed) {
  hip_capacity = size_t(1) << 40;
  std::mt19937 rng(seed);
  mf::DevPool pool;
  pool.set_limit(limit, max_block);
  std::vector<std::pair<void *, size_t>> used;
  size_t need = 0;
  for (int i = 0; i < 20000; ++i) {
    if (used.empty() || rng() % 2) {
      const size_t bytes = 1 + rng() % (size_t(1) << (9 + rng() % 16));
      void *p = nullptr;
      CHECK(pool.alloc(&p, bytes) == hipSuccess);
      for (const auto &u : used) CHECK(u.first != p);
      CHECK(hip_blocks.at(p) >= bytes);
      used.emplace_back(p, (bytes + 511) / 512 * 512);
      need += used.back().second;
    } else {
      const size_t k = rng() % used.size();
      need -= used[k].second;
      pool.release(used[k].first);
      used[k] = used.back();
      used.pop_back();
    }
    CHECK(hip_held <= need + limit);  // whatever the sizes and their order
    if (i % 5000 == 4999) {
      limit /= 4;
      pool.set_limit(limit, max_block);
    }
  }
  for (const auto &u : used) pool.release(u.first);
  CHECK(hip_held <= limit);
  pool.trim();
  CHECK(hip_held == 0 && hip_blocks.empty());
  return 0;
}

// What one context keeps does not make another's allocation fail.
static int allocation_beside_another() {
  hip_capacity = 100 << 20;
  mf::DevPool a, b;
  void *p[3], *q = nullptr;
  for (void *&x : p) CHECK(a.alloc(&x, 20 << 20) == hipSuccess);
  for (void *x : p) a.release(x);
  CHECK(hip_held == 60 << 20);
  CHECK(b.alloc(&q, 80 << 20) == hipSuccess);
  CHECK(hip_held == 80 << 20);
  CHECK(a.alloc(&p[0], 30 << 20) == hipErrorOutOfMemory);
  b.release(q);  // larger than the blocks that are kept
  CHECK(hip_held == 0);
  CHECK(a.alloc(&p[0], 30 << 20) == hipSuccess);
  a.release(p[0]);
  a.trim();
  CHECK(hip_held == 0);
  return 0;
}

// A block is used again by arrays of up to an eighth less.
static int fits() {
  hip_capacity = size_t(1) << 40;
  mf::DevPool pool;
  void *p, *q;
  CHECK(pool.alloc(&p, 9 << 16) == hipSuccess);
  pool.release(p);
  CHECK(pool.alloc(&q, 8 << 16) == hipSuccess && q == p);
  pool.release(q);
  CHECK(pool.alloc(&q, (8 << 16) - 512) == hipSuccess && q != p);
  pool.release(q);
  pool.trim();
  CHECK(hip_held == 0);
  return 0;
}

// A full list makes room for what is used now: the second round of the same sizes allocates nothing.
static int a_full_list_makes_room() {
  hip_capacity = size_t(1) << 40;
  mf::DevPool pool;
  pool.set_limit(64 << 20, 32 << 20);
  void *p[6];
  for (size_t bytes : {size_t(10) << 20, size_t(8) << 20}) {
    for (int round = 0; round < 2; ++round) {
      const size_t before = hip_allocations;
      for (void *&x : p) CHECK(pool.alloc(&x, bytes) == hipSuccess);
      CHECK(round == 0 || hip_allocations == before);
      for (void *x : p) pool.release(x);
      CHECK(hip_held <= 64 << 20);
    }
  }
  pool.trim();
  CHECK(hip_held == 0);
  return 0;
}

int main() {
  for (unsigned seed = 0; seed < 8; ++seed)
    if (random_calls(size_t(1) << (18 + seed), size_t(1) << (16 + 2 * seed), seed)) return 1;
  return allocation_beside_another() || fits() || a_full_list_makes_room();
}
