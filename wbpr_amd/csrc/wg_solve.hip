// Kernels that solve whole instances inside one workgroup (wg_solve.h), and their launches.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "wg_launch.h"
#include "wg_solve.h"

using namespace mfk;

namespace mf {

// Sums over the workgroup into the report (host memory), by its first thread.
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
// entry points expect them.
template <class L, int KIND>
__global__ __launch_bounds__(kWgThreads) void k_wg_solve(L g, WgSingle a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ WgShared S;
  WgSolver<L, KIND, kWgThreads> w{g, S, 0, a.n, a.s, a.t};
  w.st = WgStats{0, 0, 0, 0, 0, 0};
  w.carve(lds, a.lds_bytes, a.e);
  const WgOutcome o = w.solve(a.ratio, a.max_cycles, a.max_rounds, a.wide);
  if (o.status != 3) {
    for (int v = (int)threadIdx.x; v < a.n; v += kWgThreads) {
      a.h[v] = w.h[v];
      if constexpr (KIND == kWgBoth) a.e[v] = w.e[v];
    }
    if (threadIdx.x == 0) a.values[0] = o.value;
  }
  write_report(a.report, o, w.st);
}

int wg_single_kind(int32_t n, int lds_limit) {
  const long long room = (long long)lds_limit - kWgStaticLds;
  for (int kind : {(int)kWgBoth, (int)kWgHeights}) {
    if (n > kWgMaxHeights) continue;
    const long long lists = 2LL * kWgItemBytes * std::min<int32_t>(n, kWgMinList);
    if (wg_state_bytes(kind, n) + lists <= room) return kind;
  }
  return -1;
}

template <class L, int KIND>
static hipError_t launch_single(hipStream_t st, const L &g, const WgSingle &a) {
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void *>(k_wg_solve<L, KIND>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, a.lds_bytes);
  if (e != hipSuccess) return e;
  k_wg_solve<L, KIND><<<1, kWgThreads, a.lds_bytes, st>>>(g, a);
  return hipGetLastError();
}

template <class L>
hipError_t wg_single_launch(hipStream_t st, const L &g, WgSingle a, int kind, int lds_limit) {
  const long long all = wg_state_bytes(kind, a.n) + 2LL * kWgItemBytes * a.n;
  a.lds_bytes = (int)std::min<long long>((all + 15) / 16 * 16, lds_limit - kWgStaticLds);
  return kind == kWgBoth ? launch_single<L, kWgBoth>(st, g, a)
                         : launch_single<L, kWgHeights>(st, g, a);
}
template hipError_t wg_single_launch(hipStream_t, const LayoutBCSR &, WgSingle, int, int);
template hipError_t wg_single_launch(hipStream_t, const LayoutBCSR2 &, WgSingle, int, int);
template hipError_t wg_single_launch(hipStream_t, const LayoutRCSR &, WgSingle, int, int);

}  // namespace mf
