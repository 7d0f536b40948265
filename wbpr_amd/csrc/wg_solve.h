// One instance solved entirely inside one workgroup, with its vertex state in LDS.
//
// Long-path graphs and small graphs leave the grid-wide kernels idle: a push-relabel cycle with
// a few hundred active vertices, or a BFS level with a few dozen, costs a launch (or a
// device-wide round trip) and a chain of memory round trips whatever its size.  Here a cycle or
// a level costs a workgroup barrier, heights and excesses are LDS reads and LDS atomics, and
// only the residual slots are in global memory: two dependent round trips (slot range, slot
// records) per discharge, from the caches of one CU, against about sixteen per grid-wide cycle.
//
// Kinds of instance (WgKind), by what fits one CU's 160 KB of LDS:
//   kWgBoth     heights (16 bits: at most n + 1) and excesses (32 bits) in LDS, up to about 24,700
//               vertices;
//   kWgHeights  heights in LDS, excesses in global memory, up to about 63,000 vertices;
//   kWgGlobal   both in global memory, up to kWgMaxVertices (batched instances: a single graph of
//               that size has the whole grid).
// The rest of the LDS holds two vertex lists (BFS frontiers, then cycle worklists).  A list that
// outgrows its part loses nothing: the next level or cycle finds its vertices by their height or
// excess instead of by the list.
#pragma once

#include <cstddef>
#include <type_traits>

#include "kernels.h"
#include "wg_launch.h"

namespace mfk {

constexpr int kWgThreads = 1024;      // workgroup of the instances that fill a CU's LDS
constexpr int kWgMaxHeights = 65533;  // vertices whose heights (0 .. n + 1) fit 16 bits
constexpr int kWgMaxVertices = 1 << 19;  // the bitmap alone takes 64 KB of LDS then
// Vertices of more residual slots than this are discharged by a whole wave, and expanded by the
// whole workgroup in the BFS; the others by tiles of 8 or 2 lanes.
constexpr int kWgHubSlots = 96;
constexpr int kWgHubCap = 256;        // hubs waiting at a time; the others stay in the worklist
constexpr int kWgMinList = 2048;      // list entries an instance's LDS has room for at least
constexpr int kWgClockMask = 7;       // the clock is read every 8th cycle
// kWgHeights, kWgGlobal: entries of the table that sums a pass's pushes by target (at most one push per
// 2-lane tile, so at most a quarter full)
constexpr int kWgTable = 2048;

__host__ __device__ constexpr int wg_bits_words(int n) { return (n + 63) / 64 * 2; }
// LDS bytes of an instance's vertex state without the lists
__host__ __device__ constexpr long long wg_state_bytes(int kind, long long n) {
  return (kind == kWgBoth ? 4 * n : 8 * kWgTable) + (kind == kWgGlobal ? 0 : (2 * n + 3) / 4 * 4) +
         4LL * wg_bits_words((int)n);
}
// bytes of a list entry: a local vertex id
__host__ __device__ constexpr int wg_item_bytes(int kind) { return kind == kWgGlobal ? 4 : 2; }
// The kind of an instance of n vertices in `room` bytes of LDS, or -1.
__host__ __device__ constexpr int wg_kind(long long n, long long room) {
  for (int kind = kWgBoth; kind <= kWgGlobal; ++kind) {
    if (n > (kind == kWgGlobal ? kWgMaxVertices : kWgMaxHeights)) continue;
    const long long items = n < kWgMinList ? n : kWgMinList;
    if (wg_state_bytes(kind, n) + 2 * wg_item_bytes(kind) * items <= room) return kind;
  }
  return -1;
}

struct alignas(8) WgShared {
  int cnt[3];   // items of the list a cycle or level reads (q % 3), fills ((q + 1) % 3), clears
  int nhub[3];  // hubs waiting, same rotation
  int chunk;    // items of the chunk list while an overflowed worklist is walked
  int flag;     // a source was reached
  int stop[2];
  int hub[2][kWgHubCap];
};

struct WgStats {
  unsigned active, slots, pushes, relabels, bfs_verts, bfs_slots;
};

// What one solve did and how it ended.
struct WgOutcome {
  long long value;
  int status;  // 0 ok, 1 round limit, 2 a source was reached (invariant broken), 3 too wide: the
               // vertices up to `levels` have their heights, the others n
  int rounds, cycles, levels;
  long long source_out;         // this thread's part of the preflow
  long long t_relabel, t_cycle;  // wall_clock64 ticks
};

template <int T>
__device__ __forceinline__ unsigned tile_minu(unsigned v) {
  if constexpr (T > 1) {
    int a, b;
    xpair<T / 2>((int)tile_minu<T / 2>(v), a, b);
    return min((unsigned)a, (unsigned)b);
  }
  return v;
}

template <class L, int KIND, int BS>
struct WgSolver {
  // heights and list entries; a lane's lowest (height, slot)
  using HT = typename std::conditional<KIND == kWgGlobal, int, unsigned short>::type;
  using Key = typename std::conditional<KIND == kWgGlobal, unsigned long long, unsigned>::type;
  static constexpr int kSlotBits = KIND == kWgGlobal ? 32 : 16;
  static constexpr Key kNone = ~(Key)0;

  const L &g;
  WgShared &S;
  int vb, n, s, t;  // first vertex (ids in the slots), vertices, source and sink (local ids)
  HT *h;            // heights, local ids
  int *e;           // excesses, local ids
  unsigned *bits;   // BFS: reached; an overflowed worklist: its vertices
  HT *lists;        // two lists of cap entries
  int *tkey, *tsum; // kWgHeights, kWgGlobal: the table of a pass's pushes (key -1: empty)
  int cap;
  WgStats st;

  struct Range {
    int b0, d0, b1, d;  // slot i of the vertex: b0 + i below d0, else b1 + (i - d0); d slots
    __device__ __forceinline__ int seg(int i) const { return L::kSeg == 2 && i >= d0; }
    __device__ __forceinline__ int at(int i) const {
      return (L::kSeg == 2 && i >= d0) ? b1 + (i - d0) : b0 + i;
    }
  };
  __device__ __forceinline__ Range range(int u) const {
    const int2 r0 = g.range(vb + u, 0);
    Range r{r0.x, r0.y - r0.x, 0, r0.y - r0.x};
    if constexpr (L::kSeg == 2) {
      const int2 r1 = g.range(vb + u, 1);
      r.b1 = r1.x;
      r.d += r1.y - r1.x;
    }
    return r;
  }

  // Divides the dynamic LDS among the state arrays; the lists take what is left.
  __device__ __forceinline__ void carve(char *lds, int lds_bytes, int *gh, int *ge) {
    char *p = lds;
    if constexpr (KIND == kWgBoth) {
      e = reinterpret_cast<int *>(p);
      p += 4 * n;
    } else {
      e = ge + vb;
      tkey = reinterpret_cast<int *>(p);
      tsum = tkey + kWgTable;
      p += 8 * kWgTable;
    }
    bits = reinterpret_cast<unsigned *>(p);
    p += 4 * wg_bits_words(n);
    if constexpr (KIND == kWgGlobal) {
      h = reinterpret_cast<HT *>(gh + vb);
    } else {
      h = reinterpret_cast<HT *>(p);
      p += (2 * n + 3) / 4 * 4;
    }
    cap = min(n, (int)((lds + lds_bytes - p) / (2 * wg_item_bytes(KIND))));
    lists = reinterpret_cast<HT *>(p);
  }
  // (an array of two pointers, indexed at run time, would put the whole object in scratch memory)
  __device__ __forceinline__ HT *list(int q) const { return lists + (q & 1) * cap; }

  __device__ __forceinline__ void append(HT *l, int *cnt, int v) {
    const int pos = atomicAdd(cnt, 1);  // past the capacity only counted: see overflowed lists
    if (pos < cap) l[pos] = (HT)v;
  }

  // v[b] of every lane with want[b], with one counter update for the wave's active lanes.
  template <int B>
  __device__ __forceinline__ void append_all(HT *l, int *cnt, const int (&v)[B],
                                             const bool (&want)[B]) {
    unsigned long long m[B];
    int total = 0;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      m[b] = __ballot(want[b]);
      total += __popcll(m[b]);
    }
    if (total == 0) return;
    int base = 0;
    if ((int)__lane_id() == __ffsll((long long)__ballot(1)) - 1) base = atomicAdd(cnt, total);
    base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int pos = base + (int)__builtin_amdgcn_mbcnt_hi(
                                 (unsigned)(m[b] >> 32),
                                 __builtin_amdgcn_mbcnt_lo((unsigned)m[b], 0u));
      if (want[b] && pos < cap) l[pos] = (HT)v[b];
      base += __popcll(m[b]);
    }
  }

  // ---- push-relabel ------------------------------------------------------------------------

  // u, taken by a narrow tile, has too many slots for it: it waits for a wave.  Without room it
  // stays in the worklist.
  __device__ __forceinline__ void defer(int u, int *hubs, int *nhub, HT *out, int *ocnt) {
    const int pos = atomicAdd(nhub, 1);
    if (pos < kWgHubCap) hubs[pos] = u;
    else append(out, ocnt, u);
  }

  // One discharge step of each vertex of a list, by tiles of T lanes with B slots in flight each, a
  // pass of the whole workgroup (BS / T vertices) at a time.  A pass first finds every vertex's
  // lowest residual neighbour and writes the relabels; then, behind a barrier, pushes along the
  // arcs that still lead down.  No height changes while pushes run, so u -> w and w -> u never
  // push in one pass: a pair of residuals has one writer and is updated by plain stores.  (A
  // global atomic is performed in the memory-side cache and drops the line from L2, so that every
  // later read of the slot would miss.)
  template <int T, int B>
  __device__ __forceinline__ void discharge_narrow(const HT *in, int cnt, HT *out, int *ocnt,
                                                   int *hubs, int *nhub) {
    constexpr int N = BS / T;
    const int lane = (int)threadIdx.x % T;
    for (int i0 = 0; i0 < cnt; i0 += N) {
      const int i = i0 + (int)threadIdx.x / T;
      const int u = in[min(i, cnt - 1)];
      const int hu = h[u], eu = e[u];  // nothing changes excesses in this half of the pass
      const Range r = range(u);
      bool go = i < cnt && hu < n && eu > 0;
      if (go && r.d > kWgHubSlots) {
        if (lane == 0) defer(u, hubs, nhub, out, ocnt);
        go = false;
      }
      Key best = kNone;
      int bw = 0, bres = 0;
      if (go) {
        for (int x0 = lane; x0 < r.d; x0 += T * B) {
          int w[B], res[B];
#pragma unroll
          for (int b = 0; b < B; ++b) {  // past the end: the last slot again, left out below
            const int x = min(x0 + b * T, r.d - 1);
            int key;
            g.scan(r.seg(x), r.at(x), w[b], res[b], key);
          }
          Key k[B];
#pragma unroll
          for (int b = 0; b < B; ++b) {
            w[b] -= vb;
            k[b] = ((Key)(unsigned)h[w[b]] << kSlotBits) | (unsigned)(x0 + b * T);
          }
#pragma unroll
          for (int b = 0; b < B; ++b) {
            if (x0 + b * T < r.d && res[b] > 0 && w[b] != u && k[b] < best) {
              best = k[b];
              bw = w[b];
              bres = res[b];
            }
          }
        }
      }
      Key low;
      if constexpr (KIND == kWgGlobal) low = tile_min<T>(best);
      else low = tile_minu<T>(best);
      const int hmin = (int)(low >> kSlotBits);
      const bool dead = low == kNone || hmin + 1 >= n;
      const int hnew = dead ? n : max(hu, hmin + 1);
      const bool winner = go && !dead && best == low;  // one lane: keys are unique
      typename L::Pair pair;
      if (winner) {
        const int x = (int)(best & (((Key)1 << kSlotBits) - 1));
        pair = g.pair(r.seg(x), r.at(x));
      }
      if (go && lane == 0) {
        st.active++;
        st.slots += r.d;
        if (hnew > hu) {
          h[u] = (HT)hnew;
          st.relabels++;
        }
      }
      go = go && !dead && lane == 0;  // u's excess is its first lane's to lower
      __syncthreads();
      const bool push = winner && (int)h[bw] < hnew;
      const int d = tile_sum32<T>(push ? min(eu, bres) : 0);
      if (push) {
        g.push_pair(pair, bres, d);
        st.pushes++;
      }
      const int item[2] = {u, bw};
      bool want[2] = {go && eu - d > 0, false};
      if constexpr (KIND == kWgBoth) {
        if (push) want[1] = atomicAdd(&e[bw], d) == 0 && bw != t;
        if (go) want[0] = atomicSub(&e[u], d) - d > 0;
      } else {
        const int made = push ? table_add(bw, d) : -1;
        if (go && d > 0) e[u] = eu - d;
        __syncthreads();
        if (made >= 0) {
          const int old = e[bw];
          e[bw] = old + tsum[made];
          want[1] = old == 0 && bw != t;
          tkey[made] = -1;
          tsum[made] = 0;
        }
      }
      append_all(out, ocnt, item, want);
      if (i0 + N < cnt) __syncthreads();
    }
  }

  // kWgHeights, kWgGlobal: d more for w in this pass.  Excesses in global memory take no atomics (see above):
  // a pass's pushes are summed by target here, and the lane whose push made the entry, which gets
  // its index (the others -1), adds the sum to e(w) behind the next barrier.
  __device__ __forceinline__ int table_add(int w, int d) {
    int x = (int)(((unsigned)w * 2654435761u) >> 21);  // 11 bits: kWgTable entries
    for (;; x = (x + 1) & (kWgTable - 1)) {
      const int key = atomicCAS(&tkey[x], -1, w);
      if (key != -1 && key != w) continue;
      atomicAdd(&tsum[x], d);
      return key == -1 ? x : -1;
    }
  }

  // One step of a hub by a wave: push along every arc lower than h(u) until the excess is placed
  // (discharge_multi's rules).  Only hubs push meanwhile and no height changes, so plain stores do
  // here too.  Returns the height u moves to when a full scan found no lower arc, which the
  // caller writes once every hub has pushed, or -1.
  __device__ __forceinline__ int push_hub(int u, int lane, HT *out, int *ocnt) {
    constexpr int B = 4;
    const int hu = h[u];
    const int eu = tile_first<64>(lane == 0 ? e[u] : 0);  // grows meanwhile: one read for the wave
    if (hu >= n || eu <= 0) return -1;  // uniform in the wave
    const Range r = range(u);
    int hmin = n + 1;
    long long placed = 0;
    int scanned = 0;
    for (int c = 0; c < r.d && placed < eu; c += 64 * B) {
      int w[B], res[B], hw[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int i = c + lane + b * 64;
        w[b] = vb + u;
        res[b] = 0;
        int key;
        if (i < r.d) g.scan(r.seg(i), r.at(i), w[b], res[b], key);
      }
      long long want = 0;
#pragma unroll
      for (int b = 0; b < B; ++b) {
        w[b] -= vb;
        if (w[b] == u) res[b] = 0;
        hw[b] = res[b] > 0 ? (int)h[w[b]] : n + 1;
        hmin = min(hmin, hw[b]);
        if (hw[b] < hu) want += res[b];
      }
      scanned += min(r.d - c, 64 * B);
      const long long sum = tile_sum<64>(want);
      const long long left = eu - placed;
      long long d = max(0LL, min(want, left - (tile_scan<64>(want) - want)));
#pragma unroll
      for (int b = 0; b < B; ++b) {
        if (d <= 0 || res[b] <= 0 || hw[b] >= hu) continue;
        const int x = (int)min(d, (long long)res[b]);
        d -= x;
        const int i = c + lane + b * 64;
        const int old = atomicAdd(&e[w[b]], x);
        g.push_pair(g.pair(r.seg(i), r.at(i)), res[b], x);
        st.pushes++;
        if (old == 0 && w[b] != t) append(out, ocnt, w[b]);
      }
      placed += min(left, sum);
    }
    if (lane == 0) {
      st.active++;
      st.slots += scanned;
      if (placed > 0 && atomicSub(&e[u], (int)placed) - placed > 0) append(out, ocnt, u);
    }
    if (placed > 0) return -1;
    hmin = -tile_max<64>(-hmin) + 1;
    return min(hmin, n);
  }

  // The hubs waiting, a wave each.
  __device__ __forceinline__ void discharge_hubs(const int *hubs, int cnt, HT *out, int *ocnt) {
    cnt = min(cnt, kWgHubCap);
    for (int i0 = 0; i0 < cnt; i0 += BS / 64) {
      const int i = i0 + (int)threadIdx.x / 64, lane = (int)threadIdx.x & 63;
      const int hnew = i < cnt ? push_hub(hubs[i], lane, out, ocnt) : -1;
      __syncthreads();
      if (hnew >= 0 && lane == 0) {
        h[hubs[i]] = (HT)hnew;
        st.relabels++;
        if (hnew < n) append(out, ocnt, hubs[i]);
      }
      __syncthreads();
    }
  }

  // The narrowest tiles issue the fewest instructions per vertex, the widest read a vertex's slots in
  // the fewest steps: the widest that still take the list in one pass.
  __device__ __forceinline__ void discharge_list(const HT *in, int cnt, HT *out, int *ocnt,
                                                 int *hubs, int *nhub) {
    if (cnt <= BS / 8) discharge_narrow<8, 2>(in, cnt, out, ocnt, hubs, nhub);
    else if (cnt <= BS / 4) discharge_narrow<4, 4>(in, cnt, out, ocnt, hubs, nhub);
    else discharge_narrow<2, 6>(in, cnt, out, ocnt, hubs, nhub);
  }

  // The cycle of a worklist that outgrew its list: the vertices with excess and a height below n
  // are marked in the bitmap first (a vertex activated during the cycle waits for the next, as
  // with a list), then walked a list's length at a time.  The hubs waiting are among them.
  __device__ __forceinline__ void discharge_marked(HT *chunk, HT *out, int *ocnt, int *hubs,
                                                   int *nhub) {
    const int tid = (int)threadIdx.x;
    for (int v0 = 0; v0 < n; v0 += BS) {
      const int v = v0 + tid;
      const bool act = v < n && v != t && (int)h[v] < n && e[v] > 0;
      const unsigned long long m = __ballot(act);
      if ((tid & 63) == 0 && v < n) {
        bits[v / 32] = (unsigned)m;
        bits[v / 32 + 1] = (unsigned)(m >> 32);
      }
    }
    const int words = wg_bits_words(n), step = max(cap / 32, 1);
    for (int w0 = 0; w0 < words; w0 += step) {
      if (tid == 0) {
        S.chunk = 0;
        *nhub = 0;
      }
      __syncthreads();
      for (int w = w0 + tid; w < min(words, w0 + step); w += BS)
        for (unsigned m = bits[w]; m; m &= m - 1)
          append(chunk, &S.chunk, w * 32 + __ffs((int)m) - 1);
      __syncthreads();
      discharge_list(chunk, min(S.chunk, cap), out, ocnt, hubs, nhub);
      __syncthreads();
      discharge_hubs(hubs, *nhub, out, ocnt);  // (its count: every thread reads it after the barrier)
      __syncthreads();
    }
  }

  // ---- global relabel ----------------------------------------------------------------------

  // Lanes lane, lane + step, ... expand frontier vertex u of height level.  check: the source's
  // arcs are saturated, so a residual arc out of it to a vertex that reaches the sink is an error.
  template <int B>
  __device__ __forceinline__ void expand(int u, const Range &r, int lane, int step, int level,
                                         bool check, HT *out, int *ocnt) {
    for (int i0 = lane; i0 < r.d; i0 += step * B) {
      int w[B], idx[B], rin[B];
      unsigned old[B];
      bool claim[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {  // past the end: the last slot again, left out below
        const int i = min(i0 + b * step, r.d - 1);
        g.bfs_slot(r.seg(i), r.at(i), w[b], idx[b]);
      }
#pragma unroll
      for (int b = 0; b < B; ++b) old[b] = bits[(w[b] - vb) >> 5];
#pragma unroll
      for (int b = 0; b < B; ++b) {  // (u itself is marked: a loop is never followed)
        w[b] -= vb;
        const bool go = i0 + b * step < r.d && (w[b] == s ? check : !((old[b] >> (w[b] & 31)) & 1u));
        rin[b] = 0;
        if (go) rin[b] = g.bfs_rin(r.seg(min(i0 + b * step, r.d - 1)), idx[b]);
      }
#pragma unroll
      for (int b = 0; b < B; ++b) {
        old[b] = ~0u;
        if (rin[b] > 0) old[b] = atomicOr(&bits[w[b] >> 5], 1u << (w[b] & 31));
      }
#pragma unroll
      for (int b = 0; b < B; ++b) {
        claim[b] = !((old[b] >> (w[b] & 31)) & 1u);
        if (claim[b]) h[w[b]] = (HT)(level + 1);
        if (rin[b] > 0 && w[b] == s) S.flag = 1;  // residual path from the source
      }
      append_all(out, ocnt, w, claim);
    }
  }

  template <int T, int B>
  __device__ __forceinline__ void expand_vertex(int u, int lane, int level, bool check, HT *out,
                                                int *ocnt, int *hubs, int *nhub) {
    const Range r = range(u);
    if (lane == 0) {
      st.bfs_verts++;
      st.bfs_slots += r.d;
    }
    if (r.d > kWgHubSlots) {
      int pos = 0;
      if (lane == 0) {
        pos = atomicAdd(nhub, 1);
        if (pos < kWgHubCap) hubs[pos] = u;
      }
      pos = tile_first<T>(pos);
      if (pos < kWgHubCap) return;
    }
    expand<B>(u, r, lane, T, level, check, out, ocnt);
  }

  // Whether less than 63 / 64 of the capacity out of the source goes into the sink.
  __device__ __forceinline__ bool short_sink() {
    const int tid = (int)threadIdx.x;
    auto *surplus = reinterpret_cast<unsigned long long *>(S.hub[0]);  // (no hubs yet)
    static_assert(offsetof(WgShared, hub) % 8 == 0, "a 64-bit word");
    if (tid == 0) *surplus = 0;
    __syncthreads();
    long long sum = 0;
    Range r = range(s);
    for (int i = tid; i < r.d; i += BS) {
      int w, res, key;
      g.scan(r.seg(i), r.at(i), w, res, key);
      if (w - vb != s) sum += 63LL * res;
    }
    r = range(t);
    for (int i = tid; i < r.d; i += BS) {
      int w, idx;
      g.bfs_slot(r.seg(i), r.at(i), w, idx);
      if (w - vb != t) sum -= 64LL * g.bfs_rin(r.seg(i), idx);
    }
    sum = tile_sum<64>(sum);
    if (__lane_id() == 0) atomicAdd(surplus, (unsigned long long)sum);
    __syncthreads();
    return (long long)*surplus > 0;
  }

  // Heights from a BFS over reverse residual arcs: distances to the sink, n where it cannot be
  // reached.  Returns the levels; from > 0 gives up (see WgWide), before anything outside LDS has been
  // written: -1 - level, the heights up to that level set.
  __device__ __forceinline__ int relabel(int from, int levels, int most, bool check) {
    const int tid = (int)threadIdx.x;
    for (int v = tid; v < n; v += BS) h[v] = (HT)(v == s ? n + 1 : (v == t ? 0 : n));
    for (int w = tid; w < wg_bits_words(n); w += BS) {
      unsigned m = 0;
      if (w == s / 32) m |= 1u << (s & 31);
      if (w == t / 32) m |= 1u << (t & 31);
      bits[w] = m;
    }
    if (tid < 3) {
      S.cnt[tid] = tid == 0 ? 1 : 0;
      S.nhub[tid] = 0;
    }
    if (tid == 0) {
      S.flag = 0;
      list(0)[0] = (HT)t;
    }
    __syncthreads();
    int level = 0;
    for (;; ++level) {
      const int cnt = S.cnt[level % 3];
      if (cnt == 0) break;
      if (from > 0 && cnt > from) {
        if constexpr (!L::kOneLine)
          if (cnt > most) return -1 - level;
        if (levels-- == 0) return -1 - level;
      }
      if (tid == 0) {
        S.cnt[(level + 2) % 3] = 0;
        // (filled in the level that uses it, and read after that level's barrier: the next level's
        // counter, which no thread has read since two barriers ago)
        S.nhub[(level + 1) % 3] = 0;
      }
      const HT *in = list(level);
      HT *out = list(level + 1);
      int *ocnt = &S.cnt[(level + 1) % 3];
      int *hubs = S.hub[0], *nhub = &S.nhub[level % 3];
      if (cnt > cap) {  // the list overflowed: its vertices by their height
        for (int v = tid / 2; v < n; v += BS / 2)
          if ((int)h[v] == level)
            expand_vertex<2, 4>(v, tid % 2, level, check, out, ocnt, hubs, nhub);
      } else if (cnt <= BS / 8) {
        for (int i = tid / 8; i < cnt; i += BS / 8)
          expand_vertex<8, 2>(in[i], tid % 8, level, check, out, ocnt, hubs, nhub);
      } else if (cnt <= BS / 4) {
        for (int i = tid / 4; i < cnt; i += BS / 4)
          expand_vertex<4, 4>(in[i], tid % 4, level, check, out, ocnt, hubs, nhub);
      } else {
        for (int i = tid / 2; i < cnt; i += BS / 2)
          expand_vertex<2, 6>(in[i], tid % 2, level, check, out, ocnt, hubs, nhub);
      }
      __syncthreads();
      const int nh = min(*nhub, kWgHubCap);
      for (int i = 0; i < nh; ++i)
        expand<4>(hubs[i], range(hubs[i]), tid, BS, level, check, out, ocnt);
      if (nh) __syncthreads();
    }
    return level;
  }

  // ---- the whole solve ---------------------------------------------------------------------

  // The residuals hold the capacities and every excess is zero on entry.  Every thread of the
  // workgroup calls this and returns the same outcome (source_out aside).
  __device__ __forceinline__ WgOutcome solve(float ratio, int max_cycles, long long max_rounds,
                                             const WgWide &wide) {
    const int tid = (int)threadIdx.x;
    int most = 0;
    if constexpr (!L::kOneLine)
      if (wide.from > 0) most = short_sink() ? wide.most_short : wide.most;
    WgOutcome o{0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (KIND == kWgBoth) {
      for (int v = tid; v < n; v += BS) e[v] = 0;
    } else {
      for (int x = tid; x < kWgTable; x += BS) {
        tkey[x] = -1;
        tsum[x] = 0;
      }
    }
    for (long long round = 0;; ++round) {
      if (round >= max_rounds) {
        o.status = 1;
        break;
      }
      const long long t0 = (long long)wall_clock64();
      const int levels = relabel(round == 0 ? wide.from : 0, wide.levels, most, round > 0);
      if (levels < 0) {
        o.status = 3;
        o.levels = -1 - levels;
        o.t_relabel = (long long)wall_clock64() - t0;
        break;
      }
      o.levels += levels;
      o.rounds++;
      if (S.flag) {
        o.status = 2;
        break;
      }
      if (round == 0) {
        // preflow: saturate the source's arcs.  After the first BFS, which does not go through
        // the source: a solve that gives up there has changed nothing.
        const Range r = range(s);
        for (int i = tid; i < r.d; i += BS) {
          int w, res, key;
          g.scan(r.seg(i), r.at(i), w, res, key);
          if (res > 0 && w - vb != s) {
            g.push_pair(g.pair(r.seg(i), r.at(i)), res, res);
            atomicAdd(&e[w - vb], res);
            o.source_out += res;
          }
        }
      }
      __syncthreads();
      // the first worklist: reached vertices with excess (counters 1 and 2 are cleared here,
      // every thread read the last level's count before the barrier above)
      if (tid < 3) {
        S.cnt[tid] = 0;
        S.nhub[tid] = 0;
      }
      __syncthreads();
      for (int v = tid; v < n; v += BS)
        if (v != t && (int)h[v] < n && e[v] > 0) append(list(0), &S.cnt[0], v);
      __syncthreads();
      const long long t1 = (long long)wall_clock64();
      o.t_relabel += t1 - t0;
      if (S.cnt[0] == 0) break;
      // One barrier a cycle: after it a thread reads only counters that the next cycle leaves alone.
      int cnt = S.cnt[0], nh = 0;
      for (int q = 0; q < max_cycles; ++q) {
        HT *in = list(q), *out = list(q + 1);
        int *ocnt = &S.cnt[(q + 1) % 3];
        if (tid == 0) {
          S.cnt[(q + 2) % 3] = 0;
          S.nhub[(q + 2) % 3] = 0;
          S.stop[q & 1] = (q & kWgClockMask) == kWgClockMask &&
                          (double)((long long)wall_clock64() - t1) >=
                              (double)ratio * (double)(t1 - t0);
        }
        if (cnt > cap) {
          __syncthreads();  // every thread has read the hub counter this cycle rewrites
          discharge_marked(in, out, ocnt, S.hub[q & 1], &S.nhub[q % 3]);
        } else {
          discharge_hubs(S.hub[q & 1], nh, out, ocnt);
          discharge_list(in, cnt, out, ocnt, S.hub[(q & 1) ^ 1], &S.nhub[(q + 1) % 3]);
        }
        __syncthreads();
        o.cycles++;
        cnt = S.cnt[(q + 1) % 3];
        nh = S.nhub[(q + 1) % 3];
        if (cnt + nh == 0 || S.stop[q & 1]) break;
      }
      __syncthreads();
      o.t_cycle += (long long)wall_clock64() - t1;
    }
    __syncthreads();
    o.value = e[t];
    return o;
  }
};

}  // namespace mfk
