// Launches of the kernels that solve whole instances inside one workgroup (wg_solve.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace mfk {
enum WgKind { kWgBoth = 0, kWgHeights = 1, kWgGlobal = 2 };  // see wg_solve.h

// When the first global relabel gives a solve up: once more than `levels` frontiers held more than
// `from` vertices (0: never); on layouts that read two lines for a slot also at one of more than
// `most` -- of more than `most_short` where the sink takes a 64th less than the source gives.
struct WgWide {
  int from, levels, most, most_short;
};
constexpr WgWide kWgNeverWide{0, 0, 0, 0};
}

namespace mf {

// What a solve did.
struct WgReport {
  long long value;
  int status;  // WgOutcome::status
  int rounds, cycles, levels;
  long long active, slots, pushes, relabels, bfs_verts, bfs_slots, source_out;
  long long t_relabel, t_cycle;  // ticks of the 100 MHz wall clock
};

struct WgSingle {
  int *h, *e;          // n entries each, written at the end; e must be zero unless it is in LDS
  int n, s, t;
  float ratio;         // cycle time / relabel time per round
  int max_cycles;      // cycles per round
  long long max_rounds;
  mfk::WgWide wide;
  long long *values;   // [0] receives the value
  WgReport *report;    // device memory
  int lds_bytes;       // (set by the launch)
};

constexpr int kWgStaticLds = 4096;  // LDS kept back for the kernels' static arrays

// How a graph of n vertices is held (a WgKind), or -1: its state does not fit lds_limit.
int wg_single_kind(int32_t n, int lds_limit);
template <class L>
hipError_t wg_single_launch(hipStream_t st, const L &g, WgSingle a, int kind, int lds_limit);

// A batch: every instance of order[0, k) inside one workgroup of a persistent grid.
struct WgBatch {
  int *h, *e;            // global arrays over all vertices; the excesses must be zero
  const int *vbase, *nver, *src, *snk;
  const int *order;      // instances, largest first
  int k;
  int *next;             // queue heads of the launches, zero
  long long *values;
  int *status;           // per instance: WgOutcome::status
  unsigned long long *stats;
  float ratio;
  int max_cycles;
  long long max_rounds;
  int lds_bytes;         // (set by the launch)
};

// Instances of more vertices take kWgThreads threads and a CU's whole LDS each; the others
// kWgSmallThreads and a quarter of it, four to a CU.
constexpr int kWgSmallVertices = 4096;

// Whether the batch kernels take an instance of n vertices.
bool wg_batch_takes(int32_t n, int lds_limit);
// Instances order[0, large) with a CU each, then order[large, k) four to a CU.  Largest first: the
// first launch ends on its smallest instances, so the second need not overlap it.  a.next: two
// words.
hipError_t wg_batch_launch(hipStream_t st, const mfk::LayoutBCSR &g, WgBatch a, int large,
                           int num_cu, int lds_limit);

}  // namespace mf
