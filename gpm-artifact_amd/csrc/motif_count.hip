// Motif4 by counting identities (the counting formulation of gpm_pattern).
//
// Non-induced counts of the six connected 4-vertex shapes:
//   N_star    = sum_v C(d_v, 3)
//   N_path    = sum_{edges uv} (d_u - 1)(d_v - 1) - 3T
//   N_paw     = sum_v t_v (d_v - 2)            (tailed triangle)
//             = 1/2 sum_{edges uv} c_uv (d_u + d_v - 4)
//   N_cycle   = 4-cycles, counted per max-rank corner (below)
//   N_diamond = sum_{edges e} C(c_e, 2)        (c_e = triangles on e)
//   N_K4      = 4-cliques of the degree-oriented DAG
// The edge sums take every undirected edge once, at its lower-ranked end; c_e
// comes from streaming the neighbours' lists past each vertex's (below).
// and the induced counts by inclusion-exclusion over how many copies of
// each shape a larger shape holds:
//   I_K4 = N_K4
//   I_diamond = N_diamond - 6 I_K4
//   I_cycle   = N_cycle - I_diamond - 3 I_K4
//   I_paw     = N_paw - 4 I_diamond - 12 I_K4
//   I_path    = N_path - 2 I_paw - 4 I_cycle - 6 I_diamond - 12 I_K4
//   I_star    = N_star - I_paw - 2 I_diamond - 4 I_K4
//
// 4-cycles: with rank = position in (degree, id) order, every 4-cycle has a
// unique top corner u of maximal rank; its wedges u-v-w with v, w below u
// land on the opposite corner w.  The walk runs on the graph relabelled by
// rank with sorted lists, so the ends w in a range of ranks are a part of each
// list (binary search, no rank lookups).  For each root u and band of ranks a
// block counts, for every w of the band, the wedges reaching it in LDS, and sums
// C(cnt_w, 2) over the band (cycles_kernel); roots of few wedges use a hash table.
#include <algorithm>
#include <numeric>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>

#include "graph_dev.hpp"

using namespace gpm;

namespace {

constexpr int kBlock = 256;
// 4-cycle corners, roots of kCycHeavy wedges and more: one block per CU whose
// LDS holds the counters of a band of ranks, 16-bit ones where the root has less
// than 65536 lower neighbours (no counter can pass that).
constexpr int kCycBlock = 1024;
constexpr uint32_t kCycWords = 39936;  // 156 KiB of counters
constexpr uint32_t kCycHeavy = 2048;
// A root's last task covers every rank below its other tasks: a band in LDS and
// the ranks further down in HBM.  Roots of so many wedges have their first band
// (89 % of the wedges on R-MAT scale 19), and their second (another 8 %), as tasks
// of their own before it.
constexpr uint64_t kCycBand1 = 1u << 14, kCycBand2 = 1u << 17;
// Lighter roots: a hash table of their wedges' ends.
constexpr int kLightBlock = 256;
constexpr uint32_t kLightSlots = 4096;
static_assert(kLightSlots >= 2 * kCycHeavy, "load factor at most 1/2");
// 64-entry windows of a list in flight per wave.
constexpr uint32_t kCycWindows = 4;
constexpr uint32_t kCycShort = 2;  // lists of so many entries are the lanes' own

// The wedges u - v - x with lo <= x < hi (hi <= u), v one of the n_below first
// neighbours of u.  Ranks from band on have their counters in LDS.
struct CycleTask {
  uint32_t u, n_below, lo, hi, band;
};

// Blocks of 256 threads for `threads` threads, at most 32 per CU (the
// kernels stride over the rest).
unsigned grid_of(const gpm_graph* g, uint64_t threads) {
  const uint64_t want = (threads + 255) / 256;
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(want, (uint64_t)device_cus(g) * 32));
}

// ---------------------------------------------------- triangles per edge
//
// tri[e] of the entry e = (v, x), x > v, of the rank-relabelled graph is c_e.  A
// triangle u < v < x lies on three entries.  A block that holds N+(v) as bits and
// a counter per position counts both (v, .) entries of the triangles v is the
// lowest of, from the lists of its higher neighbours, and the (v, x) entry of
// those it is the middle of, from the lists of its lower ones: all in LDS.  (One
// global atomic per entry and triangle, three in all, had bound this: about 50
// per ns on the chip.)  Triangles whose lowest vertex has kTriPairs higher
// neighbours or fewer are found by searching its pairs, with atomics.

constexpr uint32_t kTriPairs = 16;
// Ids with a bit in LDS, counters in LDS (N+ longer than that: global atomics),
// and neighbours of v whose lists one task streams.
constexpr uint32_t kTriIdBits = 65536, kTriIdWords = kTriIdBits / 32;
constexpr uint32_t kTriCounters = 1024;
constexpr uint32_t kTriLists = 1024;

// Entries [begin, end) of v's list: the lists of these neighbours.
struct TriangleTask {
  uint32_t v, begin, end;
};

// Block per task (statically interleaved, in decreasing degree).  R-MAT scale
// 19: the edge sums take 5.3 ms, 11.6 ms with three global atomics a triangle.
__global__ __launch_bounds__(kBlock) void stream_triangles_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const uint32_t* __restrict__ below, uint32_t n, const TriangleTask* __restrict__ tasks,
    uint32_t n_tasks, uint32_t* __restrict__ tri) {
  constexpr uint32_t kWaves = kBlock / kWave, kPer = kTriIdWords / kBlock;
  __shared__ uint32_t s_bits[kTriIdWords];
  __shared__ uint16_t s_pre[kTriIdWords];
  __shared__ uint32_t s_cnt[kTriCounters];
  __shared__ uint32_t s_low, s_wsum[kWaves];
  const uint32_t lane = lane_id(), w = uniform(threadIdx.x / kWave);
  const uint32_t id_base = n > kTriIdBits ? n - kTriIdBits : 0u;
  for (uint32_t i = threadIdx.x; i < kTriIdWords; i += kBlock) s_bits[i] = 0u;
  for (uint32_t i = threadIdx.x; i < kTriCounters; i += kBlock) s_cnt[i] = 0u;
  for (uint32_t q = blockIdx.x; q < n_tasks; q += gridDim.x) {
    const uint32_t v = uniform(tasks[q].v), begin = uniform(tasks[q].begin),
                   end = uniform(tasks[q].end);
    const uint32_t vb = uniform(off[v]), sb = vb + uniform(below[v]);
    const uint32_t d = uniform(off[v + 1]) - sb;
    const uint32_t* S = adj + sb;
    if (threadIdx.x == 0) s_low = 0;
    __syncthreads();
    uint32_t low = 0;
    for (uint32_t i = threadIdx.x; i < d; i += kBlock) {
      const uint32_t t = S[i] - id_base;
      if (S[i] < id_base)
        ++low;
      else
        atomicOr(&s_bits[t >> 5], 1u << (t & 31));
    }
    if (low) atomicAdd(&s_low, low);
    __syncthreads();
    const uint32_t nlow = uniform(s_low);
    {
      // Ids of S before every bitmap word (at most kTriIdBits - 32: 16 bits hold it).
      uint32_t c[kPer], sum = 0;
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) sum += c[k] = (uint32_t)__popc(s_bits[kPer * threadIdx.x + k]);
      const uint32_t incl = wave_incl_scan(sum);
      if (lane == kWave - 1) s_wsum[w] = incl;
      __syncthreads();
      uint32_t at = incl - sum;
      for (uint32_t k = 0; k < w; ++k) at += s_wsum[k];
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) {
        s_pre[kPer * threadIdx.x + k] = (uint16_t)at;
        at += c[k];
      }
    }
    __syncthreads();
    auto count = [&](uint32_t pos, uint32_t triangles) {  // on entry `pos` of S
      if (pos < kTriCounters)
        atomicAdd(&s_cnt[pos], triangles);
      else
        atomicAdd(&tri[sb + pos], triangles);
    };
    for (uint32_t c0 = begin; c0 < end; c0 += kBlock) {
      // Lane l holds the list of neighbour c0 + kWaves l + w.
      const uint32_t mine = c0 + kWaves * lane + w;
      uint32_t b = 0, len = 0;
      if (mine < end) {
        const uint32_t y = adj[vb + mine];
        b = off[y] + below[y];
        len = off[y + 1] - b;
        // Lower neighbours with few higher ones search their pairs.
        if (y < v && len <= kTriPairs) len = 0;
      }
      uint64_t todo = wave_ballot(len != 0u);
      uint32_t cb = 0, cn = 0, ct = 0, ci = 0, x[kCycWindows];
      auto next = [&]() {  // moves on to the next batch of windows; false after the last
        ct += kCycWindows * kWave;
        if (ct < cn) return true;
        if (!todo) return false;
        const uint32_t j = (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1;
        cb = __builtin_amdgcn_readlane(b, j);
        cn = __builtin_amdgcn_readlane(len, j);
        ci = c0 + kWaves * j + w;
        ct = 0;
        return true;
      };
      auto load = [&](uint32_t (&y)[kCycWindows]) {
#pragma unroll
        for (uint32_t k = 0; k < kCycWindows; ++k) {
          const uint32_t p = ct + k * kWave + lane;
          y[k] = p < cn ? adj[cb + p] : kEmpty;  // past every id and bitmap word
        }
      };
      bool more = next();
      if (more) load(x);
      while (more) {
        uint32_t y[kCycWindows];
        const uint32_t entry = vb + ci;  // of v's list: the neighbour being streamed
        uint32_t hits = 0;  // of the wave: one addition to the streamed neighbour's count
        more = next();
        if (more) load(y);
#pragma unroll
        for (uint32_t k = 0; k < kCycWindows; ++k) {
          const uint32_t t = x[k] - id_base;
          uint32_t pos = kEmpty;
          if (t < kTriIdBits) {
            const uint32_t word = s_bits[t >> 5];
            if ((word >> (t & 31)) & 1u)
              pos = nlow + s_pre[t >> 5] + (uint32_t)__popc(word & ((1u << (t & 31)) - 1u));
          } else if (nlow && x[k] < id_base) {
            const uint32_t p = upper_index(S, nlow, x[k]);
            if (p > 0 && S[p - 1] == x[k]) pos = p - 1;
          }
          if (pos != kEmpty) count(pos, 1u);
          hits += (uint32_t)__popcll(wave_ballot(pos != kEmpty));
        }
        if (entry >= sb && hits && lane == 0) count(entry - sb, hits);
#pragma unroll
        for (uint32_t k = 0; k < kCycWindows; ++k) x[k] = y[k];
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < d; i += kBlock) {
      if (S[i] >= id_base) s_bits[(S[i] - id_base) >> 5] = 0u;
      if (i < kTriCounters && s_cnt[i]) {
        atomicAdd(&tri[sb + i], s_cnt[i]);
        s_cnt[i] = 0u;
      }
    }
  }
}

// 16 lanes per vertex v with 2 <= |N+(v)| <= kTriPairs: the pairs of N+(v), at
// distance k around the circle of its ids, searched in the lower one's list.
__global__ __launch_bounds__(kBlock) void pair_triangles_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const uint32_t* __restrict__ below, uint32_t n, uint32_t* __restrict__ tri) {
  constexpr int G = kTriPairs;
  const uint32_t sub = threadIdx.x & (G - 1);
  const uint32_t ngrp = gridDim.x * (kBlock / G);
  for (uint32_t v = (blockIdx.x * kBlock + threadIdx.x) / G; wave_ballot(v < n) != 0ull; v += ngrp) {
    const uint32_t sb = v < n ? off[v] + below[v] : 0u;
    uint32_t d = v < n ? off[v + 1] - sb : 0u;
    if (d > kTriPairs) d = 0;
    if (wave_ballot(d >= 2) == 0ull) continue;
    const bool act = sub < d;
    const uint32_t s = act ? adj[sb + sub] : 0u;
    const uint32_t b = act ? off[s] + below[s] : 0u, len = act ? off[s + 1] - b : 0u;
    for (uint32_t k = 1; wave_ballot(k <= d / 2) != 0ull; ++k) {
      uint32_t j = sub + k;
      if (j >= d) j -= d;
      const uint32_t sj = __shfl(s, (int)j, G), bj = __shfl(b, (int)j, G), nj = __shfl(len, (int)j, G);
      const bool pair = act && (2 * k < d || (2 * k == d && sub < k));
      const bool up = s < sj;  // this lane's list is the one searched
      const uint32_t key = up ? sj : s;
      uint32_t lo = up ? b : bj, m = pair ? (up ? len : nj) : 0u;
      const bool any = m != 0u;
      while (m > 1) {
        const uint32_t half = m >> 1;
        lo = adj[lo + half] <= key ? lo + half : lo;
        m -= half;
      }
      if (any && adj[lo] == key) {
        atomicAdd(&tri[sb + sub], 1u);
        atomicAdd(&tri[sb + j], 1u);
        atomicAdd(&tri[lo], 1u);
      }
    }
  }
}

// The same counts where lists are one-sided, hold a vertex twice or itself: a wave per
// entry (u, v) with v > u walks the shorter of both ends' upper lists and searches the
// longer (last of equal entries).  Three atomics a triangle, so mirrored lists take the
// kernels above.
__global__ __launch_bounds__(kBlock) void entry_triangles_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const uint32_t* __restrict__ below, uint32_t n, uint64_t m, uint32_t* __restrict__ tri) {
  const uint32_t lane = lane_id();
  const uint64_t nw = (uint64_t)gridDim.x * kBlock / kWave;
  auto upper = [&](uint32_t v, uint32_t* b, uint32_t* len) {  // entries above v
    const uint32_t end = off[v + 1];
    for (*b = off[v] + below[v]; *b < end && adj[*b] == v;) ++*b;
    *len = end - *b;
  };
  for (uint64_t e = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave; e < m; e += nw) {
    const uint32_t u = upper_index(off, n + 1, (uint32_t)e) - 1, v = adj[e];
    if (v <= u) continue;
    uint32_t ab, na, bb, nb;
    upper(u, &ab, &na);
    upper(v, &bb, &nb);
    if (na > nb) {
      uint32_t t = ab;
      ab = bb;
      bb = t;
      t = na;
      na = nb;
      nb = t;
    }
    uint32_t hits = 0;
    for (uint32_t i = lane; i < na; i += kWave) {
      const uint32_t w = adj[ab + i], p = upper_index(adj + bb, nb, w);
      if (p > 0 && adj[bb + p - 1] == w) {
        atomicAdd(&tri[ab + i], 1u);
        atomicAdd(&tri[bb + p - 1], 1u);
        ++hits;
      }
    }
    hits = wave_sum_u32(hits);
    if (lane == 0 && hits) atomicAdd(&tri[e], hits);
  }
}

// Edge sums over the undirected edges {v, x} (each once: x > v), from the per-edge
// triangle counts c and the degrees; one wave per v:
//   out[0] += 2c                      (sum: 6T)
//   out[2] += c (d_v + d_x - 4)       (sum: 2 N_paw)
//   out[3] += c (c - 1)               (sum: 2 N_diamond)
//   out[4] += 2 (d_v - 1)(d_x - 1)    (sum: 2 x the path edge sum)
__global__ __launch_bounds__(kBlock) void edge_stats_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const uint32_t* __restrict__ below, const uint32_t* __restrict__ tri, uint32_t n,
    unsigned long long* __restrict__ out) {
  uint64_t s6t = 0, spaw = 0, sdia = 0, spath = 0;
  const uint32_t nw = gridDim.x * blockDim.x / kWave;
  for (uint32_t v = (blockIdx.x * blockDim.x + threadIdx.x) / kWave; v < n; v += nw) {
    const uint32_t b = off[v], end = off[v + 1];
    const uint64_t da = end - b;
    for (uint32_t e = b + below[v] + lane_id(); e < end; e += kWave) {
      const uint32_t x = adj[e];
      if (x == v) continue;
      const uint64_t c = tri[e], db = off[x + 1] - off[x];
      s6t += 2 * c;
      spaw += c ? c * (da + db - 4) : 0;
      sdia += c * (c - (c ? 1 : 0));
      spath += 2 * (da - 1) * (db - 1);
    }
  }
  block_add(&out[0], s6t);
  block_add(&out[2], spaw);
  block_add(&out[3], sdia);
  block_add(&out[4], spath);
}

// out[1] += sum_v C(d_v, 3).
__global__ __launch_bounds__(kBlock) void star_sum_kernel(const uint32_t* __restrict__ off,
                                                          uint32_t n,
                                                          unsigned long long* __restrict__ out) {
  uint64_t acc = 0;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    const uint64_t d = off[v + 1] - off[v];
    acc += d >= 3 ? d * (d - 1) * (d - 2) / 6 : 0;
  }
  block_add(&out[1], acc);
}

// Entries of the sorted list a[0..n) below key.
__device__ __forceinline__ uint32_t count_below(const uint32_t* __restrict__ a, uint32_t n,
                                                uint32_t key) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (a[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Number of a's first n entries (sorted) below each of two keys, side by side.
__device__ __forceinline__ void count_below2(const uint32_t* __restrict__ a, uint32_t n,
                                             uint32_t key0, uint32_t key1, uint32_t* below0,
                                             uint32_t* below1) {
  uint32_t lo0 = 0, lo1 = 0, hi0 = n, hi1 = n;
  while (lo0 < hi0 || lo1 < hi1) {
    const uint32_t m0 = (lo0 + hi0) >> 1, m1 = (lo1 + hi1) >> 1;
    const uint32_t x0 = lo0 < hi0 ? a[m0] : 0u, x1 = lo1 < hi1 ? a[m1] : 0u;
    if (lo0 < hi0) (x0 < key0 ? lo0 : hi0) = x0 < key0 ? m0 + 1 : m0;
    if (lo1 < hi1) (x1 < key1 ? lo1 : hi1) = x1 < key1 ? m1 + 1 : m1;
  }
  *below0 = lo0;
  *below1 = lo1;
}

// Calls f(x) for every wedge end x of the task, the middle vertices dealt out
// over the block's waves one by one (whole groups of 64 left most waves idle on
// roots of a few hundred): the lanes find the bounds of their lists' parts, then
// the wave streams one part after another, 64 consecutive entries a load and the
// next windows loaded before the last are handled.  Parts of up to kCycShort entries
// are left to the lanes that found them: a hub over 200000 vertices of two neighbours
// is one block's, which loaded them for one lane's work at a time (K(2, 200000): 4.8 ms
// in windows alone, 1.2 ms; R-MAT scale 19: 6.9 and 6.6 ms).  With 4 or 8 entries
// R-MAT scale 19 gains more (6.5, 6.3 ms), but graphs of even degrees lose (100000
// vertices of degree 16: 0.44 ms with 0 - 2, 0.46 and 0.51 ms).
template <int BS, typename F>
__device__ __forceinline__ void for_wedges(const uint32_t* __restrict__ off,
                                           const uint32_t* __restrict__ adj, const CycleTask& t,
                                           F&& f) {
  const uint32_t lane = lane_id(), w = uniform(threadIdx.x / kWave);
  const uint32_t* mid = adj + uniform(off[t.u]);
  for (uint32_t c0 = 0; c0 < t.n_below; c0 += BS) {
    const uint32_t mine = c0 + BS / kWave * lane + w;
    uint32_t b = 0, len = 0;
    if (mine < t.n_below) {
      const uint32_t v = mid[mine];
      b = off[v];
      uint32_t first, end;
      count_below2(adj + b, off[v + 1] - b, t.lo, t.hi, &first, &end);
      b += first;
      len = end - first;
    }
    for (uint32_t i = 0; i < kCycShort; ++i)
      if (len <= kCycShort && i < len) f(adj[b + i]);
    uint64_t todo = wave_ballot(len > kCycShort);
    uint32_t cb = 0, cn = 0, ct = 0, x[kCycWindows];
    auto next = [&]() {  // moves on to the next batch of windows; false after the last
      ct += kCycWindows * kWave;
      if (ct < cn) return true;
      if (!todo) return false;
      const uint32_t j = (uint32_t)__builtin_ctzll(todo);
      todo &= todo - 1;
      cb = __builtin_amdgcn_readlane(b, j);
      cn = __builtin_amdgcn_readlane(len, j);
      ct = 0;
      return true;
    };
    auto load = [&](uint32_t (&y)[kCycWindows]) {
#pragma unroll
      for (uint32_t q = 0; q < kCycWindows; ++q) {
        const uint32_t p = ct + q * kWave + lane;
        y[q] = p < cn ? adj[cb + p] : kEmpty;
      }
    };
    bool more = next();
    if (more) load(x);
    while (more) {
      uint32_t y[kCycWindows];
      more = next();
      if (more) load(y);
#pragma unroll
      for (uint32_t q = 0; q < kCycWindows; ++q)
        if (x[q] != kEmpty) f(x[q]);
#pragma unroll
      for (uint32_t q = 0; q < kCycWindows; ++q) x[q] = y[q];
    }
  }
}

// One task per block at a time (queue, heaviest roots first): increments the LDS
// counters of the task's ranks from t.band on, then sums C(count, 2) over them and
// clears them on the way.  Lower ranks count in HBM (the block's n counters at
// `counters`): the increments' previous values sum to C(count, 2) there, and a
// second walk clears them.  R-MAT scale 19 (2.2e9 wedges, 98 % of them below 7100
// roots): 6.6 ms with the light roots, against 42.7 ms for one 256-thread block
// per CU that searched the owner of every wedge, kept 40000 32-bit counters in
// LDS and listed the touched ones.  What is left is latency: a group's list
// bounds are some 20 dependent loads, and 16 waves share the CU.  Cutting the
// heaviest roots into narrower bands lost (7.3 - 9.4 ms): the queue's order ends
// evenly without it.
// kMirrored: no list holds a vertex twice, which could pass a counter of 16 bits.
template <bool kMirrored>
__global__ __launch_bounds__(kCycBlock) void cycles_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj, uint32_t n,
    const CycleTask* __restrict__ tasks, uint32_t n_tasks, unsigned int* __restrict__ queue,
    uint32_t* __restrict__ counters, unsigned long long* __restrict__ out) {
  __shared__ __align__(16) uint32_t s_cnt[kCycWords];
  __shared__ uint32_t s_task;
  uint64_t acc = 0;
  for (uint32_t i = threadIdx.x; i < kCycWords; i += kCycBlock) s_cnt[i] = 0u;
  while (true) {
    if (threadIdx.x == 0) s_task = atomicAdd(queue, 1u);
    __syncthreads();
    const uint32_t q = uniform(s_task);
    __syncthreads();
    if (q >= n_tasks) break;
    CycleTask t = tasks[q];
    t.u = uniform(t.u);
    t.n_below = uniform(t.n_below);
    t.lo = uniform(t.lo);
    t.hi = uniform(t.hi);
    t.band = uniform(t.band);
    const uint32_t half = kMirrored && t.n_below < 65536u ? 1u : 0u;  // counters of 16 bits
    const uint32_t words = (t.hi - t.band + half) >> half;
    uint32_t* cnt = counters + (uint64_t)blockIdx.x * n;
    if (t.lo == t.band) {
      for_wedges<kCycBlock>(off, adj, t, [&](uint32_t x) {
        const uint32_t i = x - t.band;
        atomicAdd(&s_cnt[i >> half], 1u << (half & i) * 16);
      });
    } else {
      for_wedges<kCycBlock>(off, adj, t, [&](uint32_t x) {
        const uint32_t i = x - t.band;
        if (x >= t.band)
          atomicAdd(&s_cnt[i >> half], 1u << (half & i) * 16);
        else
          acc += wg_atomic_add(&cnt[x], 1u);
      });
      __threadfence_block();
    }
    __syncthreads();
    uint4* v = reinterpret_cast<uint4*>(s_cnt);
    for (uint32_t i = threadIdx.x; 4 * i < words; i += kCycBlock) {
      const uint4 c = v[i];
      if (c.x | c.y | c.z | c.w) {
        v[i] = make_uint4(0u, 0u, 0u, 0u);
        for (uint32_t k : {c.x, c.y, c.z, c.w}) {
          const uint64_t lo = half ? k & 0xFFFFu : k, hi = half ? k >> 16 : 0u;
          acc += lo * (lo - (lo != 0)) / 2 + hi * (hi - (hi != 0)) / 2;
        }
      }
    }
    if (t.lo < t.band) {
      CycleTask low = t;
      low.hi = t.band;
      for_wedges<kCycBlock>(off, adj, low, [&](uint32_t x) { cnt[x] = 0u; });
      __threadfence_block();
    }
    __syncthreads();
  }
  block_add(out, acc);
}

// Block per root of fewer than kCycHeavy wedges (statically interleaved).
__global__ __launch_bounds__(kLightBlock) void light_cycles_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const CycleTask* __restrict__ tasks, uint32_t n_tasks, unsigned long long* __restrict__ out) {
  __shared__ uint32_t s_key[kLightSlots];
  __shared__ uint32_t s_cnt[kLightSlots];
  constexpr uint32_t mask = kLightSlots - 1;
  uint64_t acc = 0;
  for (uint32_t q = blockIdx.x; q < n_tasks; q += gridDim.x) {
    CycleTask t = tasks[q];
    t.u = uniform(t.u);
    t.n_below = uniform(t.n_below);
    t.lo = uniform(t.lo);
    t.hi = uniform(t.hi);
    for (uint32_t i = threadIdx.x; i < kLightSlots; i += kLightBlock) {
      s_key[i] = kEmpty;
      s_cnt[i] = 0u;
    }
    __syncthreads();
    for_wedges<kLightBlock>(off, adj, t, [&](uint32_t x) {
      uint32_t h = hslot(x, mask);
      while (true) {
        const uint32_t old = atomicCAS(&s_key[h], kEmpty, x);
        if (old == kEmpty || old == x) break;
        h = (h + 1) & mask;
      }
      acc += atomicAdd(&s_cnt[h], 1u);
    });
    __syncthreads();
  }
  block_add(out, acc);
}

// below[u] = neighbours of u of lower rank.
__global__ __launch_bounds__(kBlock) void lower_counts_kernel(const uint32_t* __restrict__ off,
                                                              const uint32_t* __restrict__ adj,
                                                              uint32_t n,
                                                              uint32_t* __restrict__ below) {
  for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < n; u += gridDim.x * blockDim.x)
    below[u] = count_below(adj + off[u], off[u + 1] - off[u], u);
}

// wedges[u] += for every entry (u, v), v < u, the entries below u of v's list (zero on
// entry): exactly what for_wedges visits from u, whether or not v's list holds u, since
// light_cycles_kernel's table relies on it.  *mirrored += those entries that v's list
// answers and that u's holds once: half of all entries where every edge is in both lists
// and none is twice in one or a loop.  One lane per entry, so that hubs' lists are
// spread over the chip; a wave within one list adds up first.
__global__ __launch_bounds__(kBlock) void wedge_totals_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj, uint32_t n, uint64_t m,
    unsigned long long* __restrict__ wedges, unsigned long long* __restrict__ mirrored) {
  const uint32_t lane = lane_id();
  const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
  uint64_t answered = 0;
  for (uint64_t e0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; e0 < m; e0 += step) {
    const uint64_t e = e0 + lane;
    uint32_t u = kEmpty, c = 0;
    if (e < m) {
      u = upper_index(off, n + 1, (uint32_t)e) - 1;  // the last vertex whose list is not past e
      const uint32_t v = adj[e];
      if (v < u) {
        const uint32_t b = off[v], len = off[v + 1] - b;
        c = count_below(adj + b, len, u);
        if (c < len && adj[b + c] == u && (e == off[u] || adj[e - 1] != v)) ++answered;
      }
    }
    if (wave_ballot(u != uniform(u)) == 0ull) {
      const uint64_t sum = wave_sum_u64(c);
      if (lane == 0 && sum) atomicAdd(&wedges[u], (unsigned long long)sum);
    } else if (c) {
      atomicAdd(&wedges[u], (unsigned long long)c);
    }
  }
  block_add(mirrored, answered);
}

__global__ void zero_u32_kernel(unsigned int* p, uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

// keys[e] = rank(u) << 32 | rank(x) for every adjacency entry e = (u, x).
__global__ __launch_bounds__(kBlock) void rank_keys_kernel(const uint32_t* __restrict__ off,
                                                           const uint32_t* __restrict__ adj,
                                                           const uint32_t* __restrict__ rank,
                                                           uint32_t n, uint64_t* __restrict__ keys) {
  const uint32_t lane = lane_id();
  const uint32_t nw = gridDim.x * blockDim.x / kWave;
  for (uint32_t v = (blockIdx.x * blockDim.x + threadIdx.x) / kWave; v < n; v += nw) {
    const uint64_t hi = (uint64_t)rank[v] << 32;
    const uint32_t b = off[v], e = off[v + 1];
    for (uint32_t i = b + lane; i < e; i += kWave) keys[i] = hi | rank[adj[i]];
  }
}

__global__ void low_words_kernel(const uint64_t* __restrict__ keys, uint64_t m,
                                 uint32_t* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
       i += (uint64_t)gridDim.x * blockDim.x)
    out[i] = (uint32_t)keys[i];
}

// The graph relabelled by degree rank (position in (degree, id) order),
// every list sorted: rows of (rank(u), rank(x)) keys sorted as 64-bit
// integers, the row offsets from the degrees in rank order.
int ensure_rank_csr(gpm_graph* g) {
  if (g->rk_off) return GPM_OK;
  const uint32_t n = g->n;
  const uint64_t m = g->m;
  std::vector<uint32_t> order(n), rank(n), rk_off(n + 1, 0u);
  std::iota(order.begin(), order.end(), 0u);
  auto deg = [&](uint32_t v) { return g->h_off[v + 1] - g->h_off[v]; };
  std::sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    return deg(a) < deg(b) || (deg(a) == deg(b) && a < b);
  });
  for (uint32_t i = 0; i < n; ++i) {
    rank[order[i]] = i;
    rk_off[i + 1] = rk_off[i] + deg(order[i]);
  }
  uint32_t* d_rank = nullptr;
  uint64_t* keys = nullptr;
  void* temp = nullptr;
  size_t temp_bytes = 0;
  unsigned bits = 32;
  while (bits < 64 && (1ull << (bits - 32)) < (uint64_t)std::max(n, 1u)) ++bits;
  int st = GPM_OK;
  auto cleanup = [&]() {
    (void)hipFree(d_rank);
    (void)hipFree(keys);
    (void)hipFree(temp);
  };
  auto fail_all = [&](int code) {  // leaves no half-built graph on the handle
    cleanup();
    (void)hipFree(g->rk_off);
    (void)hipFree(g->rk_adj);
    g->rk_off = g->rk_adj = nullptr;
    return code;
  };
  if (hipMalloc(&g->rk_off, (size_t)(n + 1) * 4) != hipSuccess ||
      hipMalloc(&g->rk_adj, std::max<uint64_t>(m, 1) * 4) != hipSuccess ||
      hipMalloc(&d_rank, (size_t)std::max(n, 1u) * 4) != hipSuccess ||
      hipMalloc(&keys, std::max<uint64_t>(m, 1) * 16) != hipSuccess)
    return fail_all(
        fail(GPM_ENOMEM, "rank-relabelled graph (%llu entries)", (unsigned long long)m));
  if ((st = h2d(g, g->rk_off, rk_off.data(), (size_t)(n + 1) * 4)) != GPM_OK ||
      (st = h2d(g, d_rank, rank.data(), (size_t)n * 4)) != GPM_OK)
    return fail_all(st);
  if (m) {
    uint64_t* sorted = keys + m;
    hipLaunchKernelGGL(rank_keys_kernel, dim3(grid_of(g, (uint64_t)n * kWave)),
                       dim3(kBlock), 0, g->stream, g->off, g->adj, d_rank, n, keys);
    if (rocprim::radix_sort_keys(nullptr, temp_bytes, keys, sorted, m, 0u, bits, g->stream) !=
            hipSuccess ||
        hipMalloc(&temp, std::max<size_t>(temp_bytes, 1)) != hipSuccess ||
        rocprim::radix_sort_keys(temp, temp_bytes, keys, sorted, m, 0u, bits, g->stream) !=
            hipSuccess)
      return fail_all(fail(GPM_EHIP, "sorting the rank-relabelled graph"));
    hipLaunchKernelGGL(low_words_kernel, dim3(grid_of(g, m)), dim3(256), 0, g->stream,
                       sorted, m, g->rk_adj);
  }
  if (hipStreamSynchronize(g->stream) != hipSuccess)
    return fail_all(fail(GPM_EHIP, "building the rank-relabelled graph"));
  cleanup();
  g->motif.h_off.swap(rk_off);
  return GPM_OK;
}

// Degree of the vertex of rank v.
uint32_t rk_degree(const gpm_graph* g, uint32_t v) {
  return g->motif.h_off[v + 1] - g->motif.h_off[v];
}

// The tasks of the motif counters (g->motif), built once per handle from every
// vertex's lower neighbours and wedge total.
int ensure_motif_tasks(gpm_graph* g) {
  if (g->motif.built) return GPM_OK;
  const uint32_t n = g->n;
  int st = ensure_scratch(g, (size_t)n * 8 + 64);
  if (st != GPM_OK) return st;
  unsigned long long* d_wedges = static_cast<unsigned long long*>(g->scratch);
  if (!g->motif.below && hipMalloc(&g->motif.below, (size_t)std::max(n, 1u) * 4) != hipSuccess) {
    g->motif.below = nullptr;
    (void)hipGetLastError();
    return fail(GPM_ENOMEM, "lower-neighbour counts (%u)", n);
  }
  uint32_t* d_below = g->motif.below;
  std::vector<unsigned long long> wedges(n + 1, 0ull);  // and the mirrored entries
  std::vector<uint32_t> below(n);
  if (n) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_of(g, 2ull * n + 2)), dim3(256), 0, g->stream,
                       reinterpret_cast<unsigned int*>(d_wedges), 2ull * n + 2);
    hipLaunchKernelGGL(lower_counts_kernel, dim3(grid_of(g, n)), dim3(kBlock), 0, g->stream,
                       g->rk_off, g->rk_adj, n, d_below);
    hipLaunchKernelGGL(wedge_totals_kernel, dim3(std::min(grid_of(g, g->m), 8u * device_cus(g))),
                       dim3(kBlock), 0, g->stream, g->rk_off, g->rk_adj, n, g->m, d_wedges,
                       d_wedges + n);
    GPM_HIP(hipGetLastError());
    GPM_HIP(hipMemcpyAsync(wedges.data(), d_wedges, ((size_t)n + 1) * 8, hipMemcpyDeviceToHost,
                           g->stream));
    GPM_HIP(hipMemcpyAsync(below.data(), d_below, (size_t)n * 4, hipMemcpyDeviceToHost,
                           g->stream));
    GPM_HIP(hipStreamSynchronize(g->stream));
  }
  g->mirrored = 2 * wedges[n] == g->m ? 1 : 0;
  std::vector<uint32_t> roots;
  std::vector<CycleTask> heavy, light;
  for (uint32_t u = n; u-- > 0;) {
    if (wedges[u] >= kCycHeavy)
      roots.push_back(u);
    else if (wedges[u] >= 2)
      light.push_back({u, below[u], 0u, u, 0u});
  }
  std::stable_sort(roots.begin(), roots.end(),
                   [&](uint32_t a, uint32_t b) { return wedges[a] > wedges[b]; });
  bool hbm = false;
  for (const uint32_t u : roots) {
    const uint32_t band = g->mirrored == 1 && below[u] < 65536u ? 2 * kCycWords : kCycWords;
    uint32_t hi = u;
    auto task_to = [&](uint32_t lo) {
      heavy.push_back({u, below[u], lo, hi, hi - lo > band ? hi - band : lo});
      hi = lo;
    };
    const uint32_t first = u > band ? u - band : 0u;
    if (wedges[u] >= kCycBand1 && first) task_to(first);
    if (wedges[u] >= kCycBand2 && hi > band) task_to(hi - band);
    hbm |= hi > band;
    if (hi) task_to(0u);
  }
  // Triangle tasks, in decreasing degree (rank).
  std::vector<TriangleTask> tri;
  for (uint32_t v = g->mirrored == 1 ? n : 0u; v-- > 0;) {
    const uint32_t deg = rk_degree(g, v), high = deg - below[v];
    if (deg <= kTriPairs) break;  // so have all vertices of lower rank
    if (!high) continue;
    // Higher neighbours only where v's pairs are not searched.
    const uint32_t end = high > kTriPairs ? deg : below[v];
    for (uint32_t c = 0; c < end; c += kTriLists) tri.push_back({v, c, std::min(end, c + kTriLists)});
  }
  auto put = [&](const auto& list, void** d) -> int {
    (void)hipFree(*d);  // of an attempt that did not get to the end
    *d = nullptr;
    if (list.empty()) return GPM_OK;
    if (hipMalloc(d, list.size() * sizeof(list[0])) != hipSuccess) {
      *d = nullptr;
      (void)hipGetLastError();
      return fail(GPM_ENOMEM, "motif tasks (%zu)", list.size());
    }
    return h2d(g, *d, list.data(), list.size() * sizeof(list[0]));
  };
  if ((st = put(heavy, &g->motif.heavy)) != GPM_OK || (st = put(light, &g->motif.light)) != GPM_OK ||
      (st = put(tri, &g->motif.triangles)) != GPM_OK)
    return st;
  g->motif.n_heavy = (uint32_t)heavy.size();
  g->motif.n_light = (uint32_t)light.size();
  g->motif.n_triangles = (uint32_t)tri.size();
  g->motif.hbm = hbm;
  g->motif.built = true;
  return GPM_OK;
}

}  // namespace

namespace gpm {

int motif4_by_identities(gpm_graph* g, uint64_t out[6]) {
  int st;
  if ((st = ensure_rank_csr(g)) != GPM_OK) return st;
  if (!g->dag && (st = gpm_graph_orient(g, &g->dag)) != GPM_OK) return st;
  if ((st = ensure_motif_tasks(g)) != GPM_OK) return st;
  const int cus = device_cus(g);
  const auto& tk = g->motif;
  // Scratch: where some root's ranks pass its LDS bands, n 4-cycle counters per
  // block, within 8 GiB (fewer blocks when that much is not free).
  const uint64_t stride = tk.hbm ? g->n : 0;
  unsigned blocks_c = (unsigned)std::min<uint64_t>(cus, std::max(tk.n_heavy, 1u));
  while (blocks_c > 16 && (uint64_t)blocks_c * stride * 4 > (8ull << 30)) blocks_c /= 2;
  // The per-edge triangle counts (one uint32 per adjacency entry) use the same
  // scratch before the 4-cycle counters do.
  const uint64_t tri_bytes = std::max<uint64_t>(g->m, 1) * 4;
  while (true) {
    const uint64_t want = std::max((uint64_t)blocks_c * stride * 4, tri_bytes) + 256;
    if ((st = ensure_scratch(g, want)) == GPM_OK) break;
    if (st != GPM_ENOMEM || blocks_c <= 16) return st;
    clear_error();
    blocks_c /= 2;
  }
  const uint64_t cyc_bytes = (uint64_t)blocks_c * stride * 4;
  uint32_t* tri = static_cast<uint32_t*>(g->scratch);
  uint32_t* ccnt = static_cast<uint32_t*>(g->scratch);
  // Kernels that end in a sum over all blocks: at most 8 blocks per CU.
  auto sum_grid = [&](uint64_t threads) {
    return (unsigned)std::min<uint64_t>(grid_of(g, threads), (uint64_t)cus * 8);
  };
  if ((st = timing_begin(g)) != GPM_OK) return st;
  if ((st = zero_counters(g, 16)) != GPM_OK) return st;
  unsigned int* queue = reinterpret_cast<unsigned int*>(g->counters + 8);
  if (g->m) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_of(g, g->m)), dim3(256), 0, g->stream, tri, g->m);
    if (g->mirrored != 1)
      hipLaunchKernelGGL(entry_triangles_kernel, dim3(grid_of(g, g->m * kWave)), dim3(kBlock), 0,
                         g->stream, g->rk_off, g->rk_adj, tk.below, g->n, g->m, tri);
    if (tk.n_triangles)
      hipLaunchKernelGGL(stream_triangles_kernel,
                         dim3((unsigned)std::min<uint64_t>(tk.n_triangles, (uint64_t)cus * 8)),
                         dim3(kBlock), 0, g->stream, g->rk_off, g->rk_adj, tk.below, g->n,
                         static_cast<const TriangleTask*>(tk.triangles), tk.n_triangles, tri);
    if (g->mirrored == 1)
      hipLaunchKernelGGL(pair_triangles_kernel, dim3(grid_of(g, (uint64_t)g->n * kTriPairs)),
                         dim3(kBlock), 0, g->stream, g->rk_off, g->rk_adj, tk.below, g->n, tri);
    hipLaunchKernelGGL(edge_stats_kernel, dim3(sum_grid((uint64_t)g->n * kWave)), dim3(kBlock), 0,
                       g->stream, g->rk_off, g->rk_adj, tk.below, tri, g->n, g->counters);
    GPM_HIP(hipGetLastError());
  }
  timing_mark(g, "motif_edge_sums");
  hipLaunchKernelGGL(star_sum_kernel, dim3(sum_grid(g->n)), dim3(kBlock), 0, g->stream, g->off,
                     g->n, g->counters);
  GPM_HIP(hipGetLastError());
  timing_mark(g, "motif_star_sum");
  // The 4-cycle counters start at zero (the triangle counts lived here).
  if (cyc_bytes)
    hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_of(g, cyc_bytes / 4)), dim3(256), 0, g->stream,
                       ccnt, cyc_bytes / 4);
  if (tk.n_heavy)
    hipLaunchKernelGGL(g->mirrored == 1 ? cycles_kernel<true> : cycles_kernel<false>,
                       dim3(blocks_c), dim3(kCycBlock), 0, g->stream, g->rk_off, g->rk_adj, g->n,
                       static_cast<const CycleTask*>(tk.heavy), tk.n_heavy, queue, ccnt,
                       g->counters + 5);
  if (tk.n_light)
    hipLaunchKernelGGL(light_cycles_kernel,
                       dim3((unsigned)std::min<uint64_t>(tk.n_light, (uint64_t)cus * 5)),
                       dim3(kLightBlock), 0, g->stream, g->rk_off, g->rk_adj,
                       static_cast<const CycleTask*>(tk.light), tk.n_light, g->counters + 5);
  GPM_HIP(hipGetLastError());
  timing_mark(g, "motif_cycles");
  unsigned long long h[6];
  if ((st = timing_end(g, h, g->counters, sizeof(h))) != GPM_OK) return st;
  double ms_main = g->last_ms;
  uint64_t k4 = 0;
  if ((st = gpm_clique(g->dag, 4, nullptr, &k4)) != GPM_OK) return st;
  g->last_ms = ms_main + g->dag->last_ms;
  const uint64_t T = h[0] / 6;
  const uint64_t n_star = h[1];
  const uint64_t n_paw = h[2] / 2;
  const uint64_t n_dia = h[3] / 2;
  const uint64_t n_path = h[4] / 2 - 3 * T;
  const uint64_t n_cyc = h[5];
  const uint64_t i_k4 = k4;
  const uint64_t i_dia = n_dia - 6 * i_k4;
  const uint64_t i_cyc = n_cyc - i_dia - 3 * i_k4;
  const uint64_t i_paw = n_paw - 4 * i_dia - 12 * i_k4;
  const uint64_t i_path = n_path - 2 * i_paw - 4 * i_cyc - 6 * i_dia - 12 * i_k4;
  const uint64_t i_star = n_star - i_paw - 2 * i_dia - 4 * i_k4;
  out[0] = i_star;
  out[1] = i_path;
  out[2] = i_paw;
  out[3] = i_cyc;
  out[4] = i_dia;
  out[5] = i_k4;
  return GPM_OK;
}

}  // namespace gpm
