// Launches of the kernels that solve whole instances inside one workgroup (wg_solve.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mf {

// What a solve did, written by its kernel into host memory.
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
  int wide;            // > 0: give up when a frontier of the first relabel is wider
  long long *values;   // [0] receives the value
  WgReport *report;    // host memory the device writes
  int lds_bytes;       // (set by the launch)
};

constexpr int kWgStaticLds = 4096;  // LDS kept back for the kernels' static arrays
constexpr int kWgMinList = 2048;    // list entries an instance's LDS has room for at least

// How a graph of n vertices is held (a WgKind), or -1: its state does not fit lds_limit.
int wg_single_kind(int32_t n, int lds_limit);
template <class L>
hipError_t wg_single_launch(hipStream_t st, const L &g, WgSingle a, int kind, int lds_limit);

}  // namespace mf
