// Kernels that solve whole instances inside one workgroup (wg_solve.h), and their launches.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "wg_launch.h"
#include "wg_solve.h"

using namespace mfk;

namespace mf {

// Sums over the workgroup into the report, by its first thread.
__device__ __forceinline__ void write_report(WgReport *rep, const WgOutcome &o, const WgStats &st) {
  __shared__ unsigned long long tot[7];
  if (threadIdx.x < 7) tot[threadIdx.x] = 0;
  __syncthreads();
  const long long part[7] = {st.active,   st.slots,     st.pushes,   st.relabels,
                             st.bfs_verts, st.bfs_slots, o.source_out};
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    const long long sum = tile_sum<64>(part[q]);
    if ((threadIdx.x & 63) == 0) atomicAdd(&tot[q], (unsigned long long)sum);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  rep->value = o.value;
  rep->status = o.status;
  rep->rounds = o.rounds;
  rep->cycles = o.cycles;
  rep->levels = o.levels;
  rep->active = (long long)tot[0];
  rep->slots = (long long)tot[1];
  rep->pushes = (long long)tot[2];
  rep->relabels = (long long)tot[3];
  rep->bfs_verts = (long long)tot[4];
  rep->bfs_slots = (long long)tot[5];
  rep->source_out = (long long)tot[6];
  rep->t_relabel = o.t_relabel;
  rep->t_cycle = o.t_cycle;
}

// A single graph.  Its heights and excesses go to global memory at the end, where the read-back
// entry points, or a global relabel that goes on from an abandoned one, expect them.
// WIDE: the first global relabel may give up.
template <class L, int KIND, bool WIDE>
__global__ __launch_bounds__(kWgThreads) void k_wg_solve(L g, WgSingle a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ WgShared S;
  WgSolver<L, KIND, kWgThreads> w{g, S, 0, a.n, a.s, a.t};
  w.st = WgStats{0, 0, 0, 0, 0, 0};
  w.carve(lds, a.lds_bytes, a.h, a.e);
  const WgOutcome o = w.solve(a.ratio, a.max_cycles, a.max_rounds,
                              WIDE ? a.wide : kWgNeverWide);
  for (int v = (int)threadIdx.x; v < a.n; v += kWgThreads) {
    a.h[v] = w.h[v];
    if constexpr (KIND == kWgBoth) a.e[v] = w.e[v];
  }
  if (threadIdx.x == 0) a.values[0] = o.value;
  write_report(a.report, o, w.st);
}

int wg_single_kind(int32_t n, int lds_limit) {
  const int kind = wg_kind(n, (long long)lds_limit - kWgStaticLds);
  return kind == kWgGlobal ? -1 : kind;
}

// (The attribute is the kernel's, not the launch's: every thread sets the same value, not its own
// launch's size, which another thread's smaller graph could lower before the launch.)
template <class L, int KIND, bool WIDE>
static hipError_t launch_single(hipStream_t st, const L &g, const WgSingle &a, int lds_limit) {
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void *>(k_wg_solve<L, KIND, WIDE>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds_limit - kWgStaticLds);
  if (e != hipSuccess) return e;
  k_wg_solve<L, KIND, WIDE><<<1, kWgThreads, a.lds_bytes, st>>>(g, a);
  return hipGetLastError();
}

template <class L>
hipError_t wg_single_launch(hipStream_t st, const L &g, WgSingle a, int kind, int lds_limit) {
  const long long all = wg_state_bytes(kind, a.n) + 2LL * wg_item_bytes(kind) * a.n;
  a.lds_bytes = (int)std::min<long long>((all + 15) / 16 * 16, lds_limit - kWgStaticLds);
  if (a.wide.from > 0)
    return kind == kWgBoth ? launch_single<L, kWgBoth, true>(st, g, a, lds_limit)
                           : launch_single<L, kWgHeights, true>(st, g, a, lds_limit);
  return kind == kWgBoth ? launch_single<L, kWgBoth, false>(st, g, a, lds_limit)
                         : launch_single<L, kWgHeights, false>(st, g, a, lds_limit);
}
template hipError_t wg_single_launch(hipStream_t, const LayoutBCSR &, WgSingle, int, int);
template hipError_t wg_single_launch(hipStream_t, const LayoutBCSR2 &, WgSingle, int, int);
template hipError_t wg_single_launch(hipStream_t, const LayoutRCSR &, WgSingle, int, int);

// ---- batches ----

constexpr int kWgSmallThreads = 256;
static_assert(wg_state_bytes(kWgBoth, kWgSmallVertices) + 4LL * kWgMinList <=
                  163840 / 4 - kWgStaticLds,
              "a small instance fits a quarter of 160 KB with its excesses");

template <int KIND, int BS>
__device__ __forceinline__ void batch_one(const LayoutBCSR &g, const WgBatch &a, char *lds,
                                          WgShared &S, int inst) {
  const int vb = a.vbase[inst];
  WgSolver<LayoutBCSR, KIND, BS> w{g, S, vb, a.nver[inst], a.src[inst] - vb, a.snk[inst] - vb};
  w.st = WgStats{0, 0, 0, 0, 0, 0};
  w.carve(lds, a.lds_bytes, a.h, a.e);
  const WgOutcome o = w.solve(a.ratio, a.max_cycles, a.max_rounds, kWgNeverWide);
  if (threadIdx.x == 0) {
    a.values[inst] = o.value;
    a.status[inst] = o.status;
  }
  block_flush(w.st.active, w.st.slots, w.st.pushes, w.st.relabels, a.stats, ST_ACTIVE);
  block_flush(w.st.bfs_verts, w.st.bfs_slots, 0, 0, a.stats, ST_BFS_VERTS);
}

template <int BS>
__global__ __launch_bounds__(BS) void k_wg_batch(LayoutBCSR g, WgBatch a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ WgShared S;
  __shared__ int s_next;
  for (;;) {
    if (threadIdx.x == 0) s_next = atomicAdd(a.next, 1);
    __syncthreads();
    const int i = s_next;
    __syncthreads();
    if (i >= a.k) break;
    const int inst = a.order[i];
    const int kind = BS == kWgSmallThreads ? (int)kWgBoth : wg_kind(a.nver[inst], a.lds_bytes);
    if (kind == kWgBoth) batch_one<kWgBoth, BS>(g, a, lds, S, inst);
    else if (kind == kWgHeights) batch_one<kWgHeights, BS>(g, a, lds, S, inst);
    else batch_one<kWgGlobal, BS>(g, a, lds, S, inst);
  }
}

bool wg_batch_takes(int32_t n, int lds_limit) {
  return wg_kind(n, (long long)lds_limit - kWgStaticLds) >= 0;
}

template <int BS>
static hipError_t launch_batch(hipStream_t st, const LayoutBCSR &g, const WgBatch &a, int grid) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_wg_batch<BS>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, a.lds_bytes);
  if (e != hipSuccess) return e;
  k_wg_batch<BS><<<grid, BS, a.lds_bytes, st>>>(g, a);
  return hipGetLastError();
}

hipError_t wg_batch_launch(hipStream_t st, const LayoutBCSR &g, WgBatch a, int large, int num_cu,
                           int lds_limit) {
  const int k = a.k;
  hipError_t e = hipSuccess;
  if (large > 0) {
    a.k = large;
    a.lds_bytes = (lds_limit - kWgStaticLds) & ~15;
    e = launch_batch<kWgThreads>(st, g, a, std::min(large, num_cu));
  }
  if (e == hipSuccess && k > large) {
    a.order += large;
    a.k = k - large;
    a.next += 1;
    a.lds_bytes = (lds_limit / 4 - kWgStaticLds) & ~15;
    e = launch_batch<kWgSmallThreads>(st, g, a, std::min(k - large, 4 * num_cu));
  }
  return e;
}

}  // namespace mf
