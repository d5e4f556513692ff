// k-clique counting (3 <= k <= 5) on a degree-oriented DAG (replaces
// src/CFSolver.cuh).
//
// The reference runs one 32-lane warp per oriented edge (v0, v1) and
// materialises W1 = N+(v0) & N+(v1), W2 = W1 & N+(v2), ... in per-warp global
// scratch (CFSolver.cuh:15-97).  Here every root vertex v0 instead builds the
// DAG induced on its out-list S = N+(v0) once, as adjacency bitmaps over the
// positions of S ("rows": bit j of row i says S[j] is in N+(S[i])), and then
// counts (k-1)-cliques of that local DAG with AND + popcount:
//     k=3: sum_i |row_i|
//     k=4: sum_i sum_{j in row_i} |row_i & row_j|
//     k=5: sum_i sum_{j in row_i} sum_{l in row_i & row_j} |row_i & row_j & row_l|
// Row i equals the reference's W1 for the edge (v0, S[i]); row_i & row_j is its
// W2.  Rows are built by streaming the lists N+(S[i]) past a bitmap (block
// tiers) of S in LDS, or, for lists much longer than S and in the wave tier, by
// binary-searching each S[j] in N+(S[i]).  In the block tiers the k = 5
// sum is a masked product of 0/1 matrices on the matrix cores (count5_row).
//
// The kernels read the DAG relabelled in a topological order (gpm_graph's
// toff/tadj, built once per handle), so S = N+(v0) is sorted topologically
// and every row is upper triangular: row i only holds positions > i.  For
// k=5 the product for l then starts at l's 128-position chunk.  Counts do not
// depend on ids.
//
// Three tiers by |S| (tiers.hpp): one wave per root with rows in registers
// (|S| <= 64, one 64-bit word per row, lane i owns row i); one 512-thread
// block per root with rows in LDS (|S| <= 1024, in two tiers); one block per
// root with rows in a per-block HBM region (larger |S|).
//
// MODE selects what is accumulated: kCount (the clique count), kBytes (the
// algorithmic bytes of the reference's edge-rooted plan, see gpm.h), kWork
// (per-root plan entries, the cost-model training target).
#include <algorithm>
#include <vector>

#include "fp4_bits.hpp"
#include "graph_dev.hpp"
#include "tiers.hpp"

using namespace gpm;

namespace {

constexpr uint32_t kBlockCap = 512;
// Threads per block of the block tiers.  Rows are shared by the whole block,
// so wider blocks raise the waves per SIMD that hide latency without more LDS.
// Three blocks of the LDS tier fit a CU, and one of the wide tier.
constexpr int kLdsBlock = 512;
constexpr int kWideBlock = 512;
constexpr int kHbmBlock = 1024;
// Consecutive list entries one thread streams in the row build of the HBM
// tier.
constexpr uint32_t kSeg = 8;
// Row build of the LDS tiers: the ids of [n - kIdBits, n) have one bit each in
// LDS.  The relabelled DAG gives the most linked vertices the highest ids, so
// on R-MAT scale 20 nine in ten list entries fall into the top 32768.
constexpr uint32_t kIdBits = 32768;
constexpr uint32_t kIdWords = kIdBits / 32;
// 64-entry windows of a list one wave has in flight in that build.
constexpr uint32_t kListWindows = 4;
enum { kCount = 0, kBytes = 1, kWork = 2, kAll = 3 };
// kAll (with K = 5): the 3-, 4- and 5-clique counts of every root from one
// build of its rows; out[0..2] receive them.

// A list N+(S[i]) much longer than S is not streamed: each S[t] is looked up
// in it by binary search instead (d searches of log2(len) steps against len
// streamed entries).  In the block tiers, whose bitmap makes a streamed entry
// cheap, that are lists longer than 16d (R-MAT scale 20: the 3-clique count of
// the LDS tier took 3.5 ms with 4d, 3.0 ms with 16d).
__device__ __forceinline__ bool use_probe(uint32_t len, uint32_t d) {
  return len > max(64u, 16u * d);
}
// Threads per block of the wave tier: a root per wave, and one addition to the count
// per block.
constexpr int kTierBlock = 512;
constexpr int kTierWaves = kTierBlock / kWave;

__device__ __forceinline__ uint32_t ctz64(uint64_t x) { return (uint32_t)__builtin_ctzll(x); }

// Position of the k-th (0-based) set bit of x; x must have more than k bits.
__device__ __forceinline__ uint32_t select_bit(uint64_t x, uint32_t k) {
  uint32_t pos = 0;
#pragma unroll
  for (uint32_t half = 32; half >= 1; half >>= 1) {
    const uint64_t lo_mask = (half == 64) ? ~0ull : ((1ull << half) - 1);
    const uint32_t c = (uint32_t)__popcll(x & lo_mask);
    if (k >= c) {
      k -= c;
      x >>= half;
      pos += half;
    }
  }
  return pos;
}

// ------------------------------------------------------------ wave tier
// Rows by searches alone, bound by their scattered loads (about 7 a pair): lists are
// some 80 to 170 entries on R-MAT graphs, so even at |S| = 64 streaming them past a
// hash table, or through LDS with the searches there, was no faster.  4-cliques of
// R-MAT n = 100 k, 1.1 M samples: 200 us with a hash table and an addition to the
// count per wave, 84 us with searches and one per block; 5-cliques of scale 18 488 ->
// 350 us, 3- to 5-cliques of scale 20 1455 -> 1060 us.
// Pair first + lane of the pairs (i, t), i < t < d, in the order of i, t: row i gets
// bit t where S[t] is in S[i]'s list.
__device__ __forceinline__ void pair_search(const uint32_t* __restrict__ adj, const uint32_t* beg,
                                            const uint32_t* lens, const uint32_t* svals, uint32_t d,
                                            uint32_t first, unsigned long long* rows) {
  const uint32_t pairs = d * (d - 1) / 2, f = first + lane_id();
  if (f >= pairs) return;
  // Counted from the last pair, row d - 2 - k begins at k (k + 1) / 2: exact in FP32
  // for at most 64 rows.
  const uint32_t back = pairs - 1 - f;
  const uint32_t k = (uint32_t)((sqrtf((float)(8 * back + 1)) - 1.f) * 0.5f);
  const uint32_t i = d - 2 - k, t = d - 1 - (back - k * (k + 1) / 2);
  if (sorted_contains(adj + beg[i], lens[i], svals[t])) atomicOr(&rows[i], 1ull << t);
}

// Wave w takes the chunks of `chunk` roots w, w + waves, ... of the tier's
// list (ordered by degree or predicted cost, so the interleave evens the
// waves' loads out).  No task queue: a queue fetch is an atomic on one
// address, and those serialise (about 10 ns each), which bounded this tier
// at ~1 M roots per fused pass.
template <int K, int MODE>
__global__ __launch_bounds__(kTierBlock) void clique_wave_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    const uint32_t* __restrict__ roots, uint32_t n_roots, uint32_t chunk,
    unsigned long long* __restrict__ out, unsigned long long* __restrict__ work) {
  __shared__ unsigned long long s_rows[kTierWaves][kWave];
  __shared__ uint32_t s_pre[kTierWaves][kWave];
  __shared__ uint32_t s_beg[kTierWaves][kWave];
  __shared__ uint32_t s_len[kTierWaves][kWave];
  __shared__ uint32_t s_sv[kTierWaves][kWave];
  const uint32_t lane = lane_id();
  const uint32_t w = threadIdx.x / kWave;
  unsigned long long* rows = s_rows[w];
  uint32_t* pre = s_pre[w];
  uint32_t* beg = s_beg[w];
  uint32_t* lens = s_len[w];
  uint32_t* svals = s_sv[w];
  uint64_t acc = 0, acc3 = 0, acc4 = 0;
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / kWave;
  for (uint64_t base = wave * chunk; base < n_roots; base += nwaves * chunk) {
    const uint32_t stop = (uint32_t)min<uint64_t>(base + chunk, n_roots);
    for (uint32_t r = (uint32_t)base; r < stop; ++r) {
      const uint32_t u = uniform(roots[r]);
      const uint32_t sb = uniform(off[u]), d = uniform(off[u + 1]) - sb;  // d <= 64 by tiering
      const bool act = lane < d;
      const uint32_t s = act ? adj[sb + lane] : kEmpty;
      uint32_t b = 0, len = 0;
      if (act) {
        b = off[s];
        len = off[s + 1] - b;
      }
      rows[lane] = 0ull;
      lens[lane] = len;
      beg[lane] = b;
      svals[lane] = s;
      __builtin_amdgcn_wave_barrier();
      for (uint32_t f = 0; f < d * (d - 1) / 2; f += kWave)  // d >= 2 by tiering
        pair_search(adj, beg, lens, svals, d, f, rows);
      __builtin_amdgcn_wave_barrier();
      const uint64_t row = act ? rows[lane] : 0ull;
      uint64_t c = 0;
      if (MODE == kAll) acc3 += __popcll(row);
      if (MODE == kCount || MODE == kAll) {
        if (K == 3) {
          c = __popcll(row);
        } else {
          // The (i, j in row_i) pairs are dealt out evenly over the lanes:
          // pair p belongs to the row whose prefix range holds p, and j is
          // the (p - start)-th set bit of that row.
          const uint32_t pincl = wave_incl_scan((uint32_t)__popcll(row));
          pre[lane] = pincl;
          const uint32_t npairs = wave_bcast(pincl, kWave - 1);
          __builtin_amdgcn_wave_barrier();
          for (uint32_t t = 0; t < npairs; t += kWave) {
            const uint32_t p = t + lane;
            if (p < npairs) {
              const uint32_t i = upper_index(pre, kWave, p);
              const uint32_t excl = i ? pre[i - 1] : 0u;
              const uint64_t ri = rows[i];
              const uint32_t j = select_bit(ri, p - excl);
              const uint64_t mij = ri & rows[j];
              if (MODE == kAll) acc4 += __popcll(mij);
              if (K == 4) {
                c += __popcll(mij);
              } else {
                uint64_t mm = mij;
                while (mm) {
                  const uint32_t l = ctz64(mm);
                  mm &= mm - 1;
                  c += __popcll(mij & rows[l]);
                }
              }
            }
          }
        }
      } else if (act) {
        // Edge (u, S[lane]) of the reference plan.
        const uint64_t w1 = __popcll(row);
        c = (uint64_t)d + len + (K >= 4 ? w1 : 0);
        if (K >= 4) {
          uint64_t bits = row;
          while (bits) {
            const uint32_t j = ctz64(bits);
            bits &= bits - 1;
            if (K == 4) {
              c += w1 + lens[j];
            } else {
              const uint64_t w2m = row & rows[j];
              const uint64_t w2 = __popcll(w2m);
              c += w1 + lens[j] + w2;
              uint64_t mm = w2m;
              while (mm) {
                const uint32_t l = ctz64(mm);
                mm &= mm - 1;
                c += w2 + lens[l];
              }
            }
          }
        }
        c *= 4;  // bytes
      }
      if (MODE == kWork) {
        const uint64_t tot = wave_sum_u64(c);
        if (lane == 0) work[u] = tot / 4;
      } else {
        acc += c;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (MODE == kAll) {
    block_add(out, acc3);
    block_add(out + 1, acc4);
    block_add(out + 2, acc);
  } else if (MODE != kWork) {
    block_add(out, acc);
  }
}

// ------------------------------------------------------ block tiers

__device__ __forceinline__ uint32_t block_incl_scan(uint32_t v, uint32_t* s_wsum) {
  const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
  const uint32_t incl = wave_incl_scan(v);
  if (lane == kWave - 1) s_wsum[w] = incl;
  __syncthreads();
  uint32_t add = 0;
  for (uint32_t i = 0; i < w; ++i) add += s_wsum[i];
  __syncthreads();
  return incl + add;
}

// Per-root counting (or accounting) over W-word rows; thread-owned rows.
// K=4/5 counting with the (i, j in row_i) pairs dealt out evenly over the
// block: rows are taken BS at a time, a block scan of their popcounts
// gives each pair an owner row, and j is found by popcount over the words.
//
// For rows in HBM.
template <int K, int BS, bool ALL>
__device__ __forceinline__ uint64_t count_pairs(const unsigned long long* rows, uint32_t d,
                                                uint32_t W, uint32_t RS, uint32_t part,
                                                uint32_t n_parts, uint32_t* s_pre,
                                                uint32_t* s_wsum, uint64_t& c3, uint64_t& c4) {
  uint64_t c = 0;
  // This task counts rows part, part + n_parts, ...: nr of them.
  const uint32_t nr = d > part ? (d - part + n_parts - 1) / n_parts : 0u;
  for (uint32_t c0 = 0; c0 < nr; c0 += BS) {
    const uint32_t t0 = c0 + threadIdx.x;
    uint32_t pc = 0;
    if (t0 < nr) {
      const unsigned long long* r0 = rows + (size_t)(part + t0 * n_parts) * RS;
      for (uint32_t w = 0; w < W; ++w) pc += (uint32_t)__popcll(r0[w]);
    }
    if (ALL) c3 += pc;
    const uint32_t incl = block_incl_scan(pc, s_wsum);
    s_pre[threadIdx.x] = incl;
    __syncthreads();
    const uint32_t total = uniform(s_pre[BS - 1]);
    for (uint32_t p = threadIdx.x; p < total; p += BS) {
      const uint32_t jj = upper_index(s_pre, BS, p);
      uint32_t kth = p - (jj ? s_pre[jj - 1] : 0u);
      const unsigned long long* ri = rows + (size_t)(part + (c0 + jj) * n_parts) * RS;
      uint32_t w = 0;
      while (true) {
        const uint32_t pw = (uint32_t)__popcll(ri[w]);
        if (kth < pw) break;
        kth -= pw;
        ++w;
      }
      const uint32_t j = w * 64 + select_bit(ri[w], kth);
      const unsigned long long* rj = rows + (size_t)j * RS;
      if (K == 4) {
        for (uint32_t x = 0; x < W; ++x) c += __popcll(ri[x] & rj[x]);
      } else {
        for (uint32_t x = 0; x < W; ++x) {
          uint64_t mm = ri[x] & rj[x];
          if (ALL) c4 += __popcll(mm);
          while (mm) {
            const uint32_t l = x * 64 + ctz64(mm);
            mm &= mm - 1;
            const unsigned long long* rl = rows + (size_t)l * RS;
            for (uint32_t y = x; y < W; ++y) c += __popcll(ri[y] & rj[y] & rl[y]);
          }
        }
      }
    }
    __syncthreads();
  }
  return c;
}

template <int K, int MODE, int BS>
__device__ __forceinline__ uint64_t count_rows(const unsigned long long* rows, uint32_t d,
                                               uint32_t W, uint32_t RS, uint32_t part,
                                               uint32_t n_parts, const uint32_t* lens) {
  uint64_t c = 0;
  for (uint32_t i = part + threadIdx.x * n_parts; i < d; i += BS * n_parts) {
    const unsigned long long* ri = rows + (size_t)i * RS;
    if (MODE == kCount) {
      for (uint32_t w = 0; w < W; ++w) c += __popcll(ri[w]);  // K == 3 only
    } else {
      uint64_t w1 = 0;
      for (uint32_t w = 0; w < W; ++w) w1 += __popcll(ri[w]);
      uint64_t e = (uint64_t)d + lens[i] + (K >= 4 ? w1 : 0);
      if (K >= 4) {
        for (uint32_t w = 0; w < W; ++w) {
          uint64_t bits = ri[w];
          while (bits) {
            const uint32_t j = w * 64 + ctz64(bits);
            bits &= bits - 1;
            if (K == 4) {
              e += w1 + lens[j];
            } else {
              const unsigned long long* rj = rows + (size_t)j * RS;
              uint64_t w2 = 0;
              for (uint32_t x = 0; x < W; ++x) w2 += __popcll(ri[x] & rj[x]);
              e += w1 + lens[j] + w2;
              for (uint32_t x = 0; x < W; ++x) {
                uint64_t mm = ri[x] & rj[x];
                while (mm) {
                  const uint32_t l = x * 64 + ctz64(mm);
                  mm &= mm - 1;
                  e += w2 + lens[l];
                }
              }
            }
          }
        }
      }
      c += 4 * e;
    }
  }
  return c;
}

// Rows of one root in LDS: bit idx of row i is set when S[idx] is in N+(S[i]).
// One wave per list, 64 consecutive entries per load; an entry x >= id_base is
// looked up in the bitmap of S (one LDS word: in S or not), and its position in
// S is the word's prefix plus the set bits below x.  Entries below id_base only
// matter when S has some there (*s_low of them, at its front): those are
// binary-searched.  Lists much longer than S are left to the probing pass
// (*s_any_probe).  A bitmap word answers an entry in a fixed few instructions,
// where an open-addressed table of S made the 64 lanes wait for the longest
// probe sequence among them: the 3-clique count of the LDS tier on R-MAT scale
// 20, nearly all row build, fell from 7.2 to 3.0 ms (2.3e9 entries).
template <int BS>
__device__ __forceinline__ void build_rows(const uint32_t* __restrict__ adj,
                                           unsigned long long* rows, uint32_t RS, uint32_t d,
                                           const uint32_t* lens, const uint32_t* begs,
                                           const uint32_t* sids, uint32_t* bits, uint16_t* pre,
                                           uint32_t id_base, uint32_t* s_wsum, uint32_t* s_low,
                                           int* s_any_probe) {
  constexpr uint32_t kPer = kIdWords / BS;  // consecutive bitmap words per thread
  static_assert(kPer * BS == kIdWords, "whole words per thread");
  const uint32_t lane = lane_id();
  uint32_t low = 0;
  for (uint32_t i = threadIdx.x; i < d; i += BS) {
    const uint32_t t = sids[i] - id_base;
    if (sids[i] < id_base)
      ++low;
    else
      atomicOr(&bits[t >> 5], 1u << (t & 31));
  }
  if (low) atomicAdd(s_low, low);
  __syncthreads();
  const uint32_t nlow = uniform(*s_low);
  {
    uint32_t c[kPer], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) sum += c[k] = (uint32_t)__popc(bits[kPer * threadIdx.x + k]);
    uint32_t at = nlow + block_incl_scan(sum, s_wsum) - sum;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      pre[kPer * threadIdx.x + k] = (uint16_t)at;
      at += c[k];
    }
  }
  __syncthreads();
  // The next kListWindows windows of a wave's lists are loaded before the last
  // ones are looked up, so a wave always has a batch of loads in flight.
  uint32_t* rows32 = reinterpret_cast<uint32_t*>(rows);
  struct Batch {
    uint32_t row, len, t0;  // entries [t0, t0 + kListWindows * kWave) of list `row`
    const uint32_t* list;
    uint32_t x[kListWindows];
  };
  // Moves to the wave's list i or the next one that is streamed.
  auto open = [&](Batch& b, uint32_t i) {
    b.t0 = 0;
    for (; i < d; i += BS / kWave) {
      b.len = uniform(lens[i]);
      if (!use_probe(b.len, d) && b.len) break;
      if (b.len && lane == 0) *s_any_probe = 1;
    }
    b.row = i;
    b.list = adj + (i < d ? uniform(begs[i]) : 0u);
  };
  auto load = [&](Batch& b) {
#pragma unroll
    for (uint32_t q = 0; q < kListWindows; ++q) {
      const uint32_t p = b.t0 + q * kWave + lane;
      b.x[q] = p < b.len ? b.list[p] : kEmpty;  // kEmpty: past every id and bitmap word
    }
  };
  Batch cur;
  open(cur, uniform(threadIdx.x / kWave));
  if (cur.row < d) load(cur);
  while (cur.row < d) {
    Batch next = cur;
    next.t0 += kListWindows * kWave;
    if (next.t0 >= next.len) open(next, cur.row + BS / kWave);
    if (next.row < d) load(next);
    uint32_t* row = rows32 + 2 * cur.row * RS;
#pragma unroll
    for (uint32_t q = 0; q < kListWindows; ++q) {
      if (cur.t0 + q * kWave >= cur.len) break;
      const uint32_t t = cur.x[q] - id_base;
      if (t < kIdBits) {
        const uint32_t w = bits[t >> 5], below = (1u << (t & 31)) - 1u;
        if ((w >> (t & 31)) & 1u) {
          const uint32_t idx = pre[t >> 5] + (uint32_t)__popc(w & below);
          atomicOr(&row[idx >> 5], 1u << (idx & 31));
        }
      } else if (nlow && cur.x[q] < id_base) {
        const uint32_t p = upper_index(sids, nlow, cur.x[q]);
        if (p > 0 && sids[p - 1] == cur.x[q]) atomicOr(&row[(p - 1) >> 5], 1u << ((p - 1) & 31));
      }
    }
    cur = next;
  }
  __syncthreads();
}

// Column blocks lb, lb + 1, ... whose first position lies in chunk C0 (of 128
// positions), against the row blocks in a; adds to sum.  Rows l hold positions
// > l only, so the sizes start at chunk C0, and the adjacency of a column block
// sits in the chunks of its positions.  Then the same for the chunks after C0.
template <int NC, int J, int C0>
__device__ __forceinline__ void count5_columns(const uint32_t* rows32, uint32_t RS32,
                                               const intx4 (&a)[J][NC], const uint16_t* list,
                                               uint32_t nt, uint32_t lb, floatx4& sum) {
  const uint32_t lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  for (; lb < nt; ++lb) {
    const uint32_t l = list[16 * lb + r16];
    if (C0 + 1 < NC && uniform(l) >= 128 * (C0 + 1)) break;
    const uint32_t last = __builtin_amdgcn_readlane(l, 15) / 128;
    const uint32_t* rl = rows32 + __umul24(l, RS32) + g;
    const uint32_t lw = (l >> 5) - g;  // word of l's own bit, from this lane's first
    const uint32_t lbit = 1u << (l & 31);
    floatx4 both[J], adj[J];
    const intx4 b0 = fp4_in_place(rl[4 * C0]);
    const intx4 e0 = fp4_in_place(lw == 4 * C0 ? lbit : 0u);
#pragma unroll
    for (int q = 0; q < J; ++q) {
      both[q] = mfma_fp4(a[q][C0], b0, zero);
      adj[q] = mfma_fp4(a[q][C0], e0, zero);
    }
#pragma unroll
    for (int c = C0 + 1; c < NC; ++c) {
      const intx4 b = fp4_in_place(rl[4 * c]);
#pragma unroll
      for (int q = 0; q < J; ++q) both[q] = mfma_fp4(a[q][c], b, both[q]);
      if ((uint32_t)c <= last) {
        const intx4 e = fp4_in_place(lw == 4 * c ? lbit : 0u);
#pragma unroll
        for (int q = 0; q < J; ++q) adj[q] = mfma_fp4(a[q][c], e, adj[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < J; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] = __builtin_fmaf(both[q][r], adj[q][r], sum[r]);
  }
  if constexpr (C0 + 1 < NC) count5_columns<NC, J, C0 + 1>(rows32, RS32, a, list, nt, lb, sum);
}

// Row blocks jg .. jg + J - 1 (16 positions of N_i each) of the k = 5 count of
// row i, see count5_row.
template <int NC, int J, bool ALL>
__device__ __forceinline__ float count5_blocks(const uint32_t* rows32, uint32_t RS32,
                                               const uint32_t (&ri)[NC], const uint16_t* list,
                                               uint32_t nt, uint32_t jg, uint32_t& c4) {
  const uint32_t lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  intx4 a[J][NC];
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const uint32_t* rj = rows32 + __umul24(list[16 * (jg + q) + r16], RS32) + g;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const uint32_t w = rj[4 * c] & ri[c];
      if (ALL) c4 += (uint32_t)__popc(w);
      a[q][c] = fp4_reciprocal(w);
    }
  }
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
  count5_columns<NC, J, 0>(rows32, RS32, a, list, nt, jg, sum);
  return (sum[0] + sum[1]) + (sum[2] + sum[3]);
}

// One row i of the k = 5 count, by one wave: with N_i the set bits of row i,
//     sum over j, l in N_i, l in row j, of |row_i & row_j & row_l|.
// The sizes are a product of 0/1 matrices (rows j masked by row i, times rows
// l), which the matrix cores evaluate in FP4 with FP32 sums, 16 x 16 pairs and
// 128 positions per instruction; the rows of N_i are gathered from LDS and
// expanded in registers.  The pairs that are adjacent are picked by a second
// product, of the same rows j with the unit vectors of l, which leaves the 0/1
// adjacency of the pair in the register and lane of its size: one fused
// multiply-add then sums.  Every value is a whole number below 2^24 (a lane
// sums at most 1024^2 / 64 pairs of at most 1024), so FP32 is exact.
// The pairs within a hub's out-list are dense (30 - 45 % of all pairs on R-MAT
// scale 20), so a dense product does less work than AND + popcount over the
// set bits one by one, which ran at 95 % of the VALU issue rate with 54 % of the
// lanes in use.  On R-MAT scale 20 the k = 5 launch of the LDS tier went from
// 19.7 to 9.6 ms (with the row build above) and the wide tier's from 7.2 to
// 2.9 ms.  VALU issue still bounds it: expanding and gathering take about 20
// instructions per 16 x 16 pairs.  The kernel must not spill inside the count:
// matrix instructions read every lane's register, whatever the active lanes.
// The list of N_i is filled up with d, the index of a row of zeros.
template <int NC, bool ALL>
__device__ __forceinline__ uint32_t count5_row(const uint32_t* rows32, uint32_t RS32, uint32_t d,
                                               uint32_t W, uint32_t i, uint16_t* list,
                                               uint32_t& c3, uint32_t& c4) {
  const uint32_t lane = lane_id(), g = lane >> 4;
  const uint32_t* row = rows32 + i * RS32;
  uint32_t ni = 0;
  for (uint32_t w = 0; w < W; ++w) {
    const uint64_t word = (uint64_t)uniform(row[2 * w + 1]) << 32 | uniform(row[2 * w]);
    const bool in = (word >> lane) & 1ull;
    if (in) list[ni + lanes_below(word)] = (uint16_t)(64 * w + lane);
    if (ALL) c3 += in ? 1u : 0u;
    ni += (uint32_t)__popcll(word);
  }
  list[ni + lane] = (uint16_t)d;
  __builtin_amdgcn_wave_barrier();
  if (ni < 2) return 0;  // no pair j, l
  uint32_t ri[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) ri[c] = 4 * c + g < 2 * W ? row[4 * c + g] : 0u;
  float s = 0.f;
  const uint32_t nt = (ni + 15) / 16;
  // One row block at a time keeps the registers of the 8-word tier low enough for three
  // resident blocks, which also hide the row build's loads better (two of four or two
  // row blocks at a time: 9.9 ms a fused launch on R-MAT scale 20, three of one 8.9);
  // the wide tier's single block per CU gains from two (2.9 ms, 3.15 with one).
  constexpr uint32_t J = NC <= 4 ? 1 : 2;
  if (J == 1 || nt == 1) {
    for (uint32_t jg = 0; jg < nt; ++jg)
      s += count5_blocks<NC, 1, ALL>(rows32, RS32, ri, list, nt, jg, c4);
  } else {
    for (uint32_t jg = 0; jg < nt; jg += J)
      s += count5_blocks<NC, J, ALL>(rows32, RS32, ri, list, nt, jg, c4);
  }
  __builtin_amdgcn_wave_barrier();
  return (uint32_t)s;
}

// The k = 5 count of the rows part, part + n_parts, ... of a root: the block's
// waves take them in turn (the rows' costs fall slowly with their index, so
// the waves end together).  Rows are MAXW words at most; words past W are
// masked out by row i's.  A lane's sums over one root fit 32 bits (at most
// C(1024, 4) 4-cliques over the block's lanes).
template <int NC, bool ALL, int BS>
__device__ __forceinline__ uint32_t count5_rows(const unsigned long long* rows, uint32_t d,
                                                uint32_t W, uint32_t RS, uint32_t part,
                                                uint32_t n_parts, uint16_t* list, uint32_t& c3,
                                                uint32_t& c4) {
  uint32_t c = 0;
  for (uint32_t i = part + uniform(threadIdx.x / kWave) * n_parts; i < d; i += BS / kWave * n_parts)
    c += count5_row<NC, ALL>(reinterpret_cast<const uint32_t*>(rows), 2 * RS, d, W, i, list, c3, c4);
  return c;
}

// The k = 4 count of a root, sum over j, l in row j, of |row_j & row_l|: the same
// product as a row's k = 5 count (count5_row), of all rows unmasked.  The blocks
// part, part + n_parts, ... of 16 rows go to the waves there and back, since their
// costs fall with the index (two or four blocks at a time left waves without one).
// list: 0 .. d - 1, then d.  Of a 4-clique launch on R-MAT scale 20 it leaves the row
// build: LDS tier 5.1 -> 3.2 ms, of which 3.0 are the build, and wide tier 0.99 -> 0.32,
// against AND + popcount over the set bits as for rows in HBM.
template <int NC, int BS>
__device__ __forceinline__ uint32_t count4_rows(const unsigned long long* rows, uint32_t d,
                                                uint32_t W, uint32_t RS, uint32_t part,
                                                uint32_t n_parts, const uint16_t* list) {
  constexpr uint32_t kWaves = BS / kWave;
  const uint32_t g = lane_id() >> 4, w = uniform(threadIdx.x / kWave);
  uint32_t all[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) all[c] = 4 * c + g < 2 * W ? ~0u : 0u;
  const uint32_t nt = (d + 15) / 16;
  uint32_t c = 0, unused = 0;
  for (uint32_t k = 0; part + k * kWaves * n_parts < nt; ++k) {
    const uint32_t jg = part + (k * kWaves + (k & 1 ? kWaves - 1 - w : w)) * n_parts;
    if (jg < nt)
      c += (uint32_t)count5_blocks<NC, 1, false>(reinterpret_cast<const uint32_t*>(rows), 2 * RS,
                                                 all, list, nt, jg, unused);
  }
  return c;
}

// Block per root.  LDS_ROWS: rows, S, lens, begins and the bitmap of S live in
// dynamic LDS (|S| <= cap, W <= MAXW words per row).  Otherwise rows live in this block's
// HBM region `grows` (cap*W words) and membership in S is a binary search.
// Waves per SIMD the registers have to leave room for: as many as the LDS of
// three resident blocks (8-word rows) needs.
constexpr int block_waves(int k, int mode, bool lds_rows, int maxw) {
  return k >= 4 && (mode == kCount || mode == kAll) && lds_rows && maxw == 8 ? 6 : 1;
}

// into = GPM_ROWS(128-position chunks of this root's rows), among the tier's counts.
#define GPM_BY_CHUNKS(into)                                                 \
  if (MAXW == 8) {                                                          \
    switch ((W + 1) / 2) {                                                  \
      case 0: case 1: into = GPM_ROWS(1); break;                            \
      case 2: into = GPM_ROWS(2); break;                                    \
      case 3: into = GPM_ROWS(3); break;                                    \
      default: into = GPM_ROWS(4); break;                                   \
    }                                                                       \
  } else {                                                                  \
    switch ((W + 1) / 2) {                                                  \
      case 0: case 1: case 2: case 3: case 4: case 5: into = GPM_ROWS(5); break; \
      case 6: into = GPM_ROWS(6); break;                                    \
      case 7: into = GPM_ROWS(7); break;                                    \
      default: into = GPM_ROWS(8); break;                                   \
    }                                                                       \
  }

template <int K, int MODE, bool LDS_ROWS, int MAXW, int BS>
__global__ __launch_bounds__(BS, block_waves(K, MODE, LDS_ROWS, MAXW)) void clique_block_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
    uint32_t n, const uint32_t* __restrict__ roots, const uint32_t* __restrict__ parts,
    uint32_t n_roots, uint32_t cap, unsigned int* __restrict__ queue,
    unsigned long long* __restrict__ grows, uint32_t* __restrict__ gmeta,
    unsigned long long* __restrict__ out, unsigned long long* __restrict__ work) {
  extern __shared__ unsigned long long s_dyn[];
  __shared__ uint32_t s_pre[BS];
  __shared__ uint32_t s_wsum[(BS / kWave)];
  __shared__ uint32_t s_root;
  __shared__ uint32_t s_np;
  __shared__ int s_any_probe;
  __shared__ uint32_t s_low;   // entries of S below id_base
  __shared__ unsigned long long s_red[(BS / kWave)];
  __shared__ unsigned long long s_tot[BS / kWave][3];  // k = 5: counts for k = 5, 3, 4
  const uint32_t Wcap = (cap + 63) / 64;
  // LDS rows of the 8-word tier are padded to an odd stride (in 8-byte words):
  // the rows read together sit at data-dependent indices, and an even stride
  // maps them onto few banks.
  constexpr bool kPad = LDS_ROWS && MAXW == 8;
  const uint32_t RScap = kPad ? (Wcap | 1u) : Wcap;
  unsigned long long* rows;
  uint32_t *lens, *begs;
  uint32_t* sids = nullptr;   // S itself
  uint32_t* bits = nullptr;   // kIdWords words: the ids of S from id_base on
  uint16_t* pre = nullptr;    // position in S of the first id of each word
  uint16_t* lists = nullptr;  // cap + 64 entries per wave (k = 5), over lens .. pre
  if (LDS_ROWS) {
    rows = s_dyn;
    lens = reinterpret_cast<uint32_t*>(rows + (size_t)(cap + 1) * RScap);
    begs = lens + cap;
    sids = begs + cap;
    bits = sids + cap;
    pre = reinterpret_cast<uint16_t*>(bits + kIdWords);
    lists = reinterpret_cast<uint16_t*>(lens) + (threadIdx.x / kWave) * (cap + kWave);
  } else {
    rows = grows + (size_t)blockIdx.x * cap * Wcap;
    lens = gmeta + (size_t)blockIdx.x * 2 * cap;
    begs = lens + cap;
  }
  const uint32_t id_base = n > kIdBits ? n - kIdBits : 0u;
  constexpr bool kCount5 = LDS_ROWS && K == 5 && (MODE == kCount || MODE == kAll);
  constexpr bool kCount4 = LDS_ROWS && K == 4 && MODE == kCount;
  uint64_t acc = 0, acc3 = 0, acc4 = 0;
  if (kCount5 && threadIdx.x < BS / kWave * 3) (&s_tot[0][0])[threadIdx.x] = 0ull;
  while (true) {
    if (threadIdx.x == 0) s_root = atomicAdd(queue, 1u);
    __syncthreads();
    const uint32_t r = uniform(s_root);
    __syncthreads();
    if (r >= n_roots) break;
    const uint32_t u = uniform(roots[r]);
    const uint32_t pp = parts ? uniform(parts[r]) : (1u << 16);
    const uint32_t part = pp & 0xFFFFu, n_parts = pp >> 16;
    const uint32_t sb = uniform(off[u]), d = uniform(off[u + 1]) - sb;
    const uint32_t* S = adj + sb;
    const uint32_t W = (d + 63) / 64;
    const uint32_t RS = kPad ? (W | 1u) : W;
    if (threadIdx.x == 0) {
      s_any_probe = 0;
      s_low = 0;
    }
    for (uint32_t i = threadIdx.x; i < d; i += BS) {
      const uint32_t v = S[i];
      const uint32_t b = off[v];
      const uint32_t len = off[v + 1] - b;
      lens[i] = len;
      begs[i] = b;
      if (LDS_ROWS) sids[i] = v;
    }
    // LDS rows: row d stays empty.
    for (uint32_t i = threadIdx.x; i < (LDS_ROWS ? d + 1 : d) * RS; i += BS) rows[i] = 0ull;
    if (LDS_ROWS)
      for (uint32_t i = threadIdx.x; i < kIdWords; i += BS) bits[i] = 0u;
    __syncthreads();
    // HBM rows: drop stale L1 lines of the previous root before reading.
    if (!LDS_ROWS) __threadfence();
    if constexpr (LDS_ROWS) {
      build_rows<BS>(adj, rows, RS, d, lens, begs, sids, bits, pre, id_base, s_wsum, &s_low,
                     &s_any_probe);
    } else
    // Flattened walk over the lists that are streamed.
    for (uint32_t c0 = 0; c0 < d; c0 += BS) {
      const uint32_t i = c0 + threadIdx.x;
      uint32_t wl = 0;
      if (i < d) {
        const uint32_t len = lens[i];
        if (use_probe(len, d))
          s_any_probe = 1;
        else
          wl = len;
      }
      const uint32_t incl = block_incl_scan(wl, s_wsum);
      s_pre[threadIdx.x] = incl;
      __syncthreads();
      const uint32_t total = uniform(s_pre[BS - 1]);
      // Each thread takes kSeg consecutive entries: one owner search for the
      // first, then the owner row advances along the prefix sums.
      for (uint32_t f0 = threadIdx.x * kSeg; f0 < total; f0 += BS * kSeg) {
        uint32_t j = upper_index(s_pre, BS, f0);
        uint32_t excl = j ? s_pre[j - 1] : 0u;
        uint32_t end = s_pre[j];
#pragma unroll
        for (uint32_t k = 0; k < kSeg; ++k) {
          const uint32_t f = f0 + k;
          if (f >= total) break;
          while (f >= end) {  // next non-empty row; ends since f < total
            excl = end;
            end = s_pre[++j];
          }
          const uint32_t row_i = c0 + j;
          const uint32_t x = adj[begs[row_i] + (f - excl)];
          const uint32_t p = upper_index(S, d, x);
          const int idx = (p > 0 && S[p - 1] == x) ? (int)(p - 1) : -1;
          // The rows are this block's slice of HBM scratch.
          if (idx >= 0) wg_atomic_or(&rows[(size_t)row_i * RS + (idx >> 6)], 1ull << (idx & 63));
        }
      }
      __syncthreads();
    }
    // Probed lists: the ballot of "S[t] in N+(S[i])" over 64 consecutive t
    // is row word t/64.
    if (uniform((uint32_t)s_any_probe)) {
      // Probed rows of each BS-row chunk are listed in s_pre, then the
      // (probed row, element of S) pairs are dealt out over the block.
      for (uint32_t c0 = 0; c0 < d; c0 += BS) {
        const uint32_t i = c0 + threadIdx.x;
        const uint32_t flag = (i < d && use_probe(lens[i], d)) ? 1u : 0u;
        const uint32_t incl = block_incl_scan(flag, s_wsum);
        if (flag) s_pre[incl - 1] = i;
        if (threadIdx.x == BS - 1) s_np = incl;
        __syncthreads();
        const uint32_t np = uniform(s_np);
        for (uint32_t f = threadIdx.x; f < np * d; f += BS) {
          const uint32_t k = f / d, t = f - k * d;
          const uint32_t ri = s_pre[k];
          if (sorted_contains(adj + begs[ri], lens[ri], S[t]))
            wg_atomic_or(&rows[(size_t)ri * RS + (t >> 6)], 1ull << (t & 63));
        }
        __syncthreads();
      }
    }
    __syncthreads();
    if (!LDS_ROWS) __threadfence();
    uint64_t c = 0;
    if constexpr (kCount5) {
      constexpr bool ALL = MODE == kAll;
      uint32_t r3 = 0, r4 = 0, c = 0;
#define GPM_ROWS(NC) count5_rows<NC, ALL, BS>(rows, d, W, RS, part, n_parts, lists, r3, r4)
      GPM_BY_CHUNKS(c)
#undef GPM_ROWS
      // The totals stay in LDS: the count needs the registers.
      const uint64_t w5 = wave_sum_u64(c), w3 = ALL ? wave_sum_u64(r3) : 0,
                     w4 = ALL ? wave_sum_u64(r4) : 0;
      if (lane_id() == 0) {
        unsigned long long* t = s_tot[threadIdx.x / kWave];
        t[0] += w5;
        if (ALL) {
          t[1] += w3;
          t[2] += w4;
        }
      }
    } else if constexpr (kCount4) {
      uint16_t* list = reinterpret_cast<uint16_t*>(lens);
      for (uint32_t i = threadIdx.x; i < d + kWave; i += BS) list[i] = (uint16_t)min(i, d);
      __syncthreads();
#define GPM_ROWS(NC) count4_rows<NC, BS>(rows, d, W, RS, part, n_parts, list)
      GPM_BY_CHUNKS(c)
#undef GPM_ROWS
    } else if ((MODE == kCount || MODE == kAll) && K >= 4) {
      c = count_pairs<K, BS, MODE == kAll>(rows, d, W, RS, part, n_parts, s_pre, s_wsum, acc3, acc4);
    } else {
      c = count_rows<K, MODE, BS>(rows, d, W, RS, part, n_parts, lens);
    }
    if (MODE == kWork) {
      c = wave_sum_u64(c);
      if (lane_id() == 0) s_red[threadIdx.x / kWave] = c;
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < (BS / kWave); ++i) t += s_red[i];
        work[u] = t / 4;
      }
    } else {
      acc += c;
    }
    __syncthreads();
  }
  if (kCount5 && lane_id() == 0) {
    acc = s_tot[threadIdx.x / kWave][0];
    acc3 = s_tot[threadIdx.x / kWave][1];
    acc4 = s_tot[threadIdx.x / kWave][2];
  }
  if (MODE == kAll) {
    block_add(out, acc3);
    block_add(out + 1, acc4);
    block_add(out + 2, acc);
  } else if (MODE != kWork) {
    block_add(out, acc);
  }
}

__global__ void zero_u32_kernel(unsigned int* p, int count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = 0u;
}

// Dynamic LDS of a block of `waves` waves: rows and an empty row; then S with
// its list bounds and the bitmap of S with its prefixes, whose place the k = 5
// count's position lists take over.
size_t block_lds_bytes(uint32_t cap, uint32_t waves, bool pad) {
  const uint32_t W = (cap + 63) / 64;
  return (size_t)(cap + 1) * (pad ? (W | 1u) : W) * 8 +
         std::max<size_t>((size_t)cap * 12 + kIdWords * 6, (size_t)waves * (cap + kWave) * 2);
}

// Largest out-degree whose rows fit one block's LDS on this device (at most
// 1024 = 16 words per row); kBlockCap when the device allows only 64 KiB.
uint32_t lds_wide_cap() {
  static int cached = -1;
  if (cached < 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    size_t limit = 64 * 1024;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      limit = prop.sharedMemPerBlock;
    uint32_t cap = kBlockCap;
    for (uint32_t c = 1024; c > kBlockCap; c -= 64) {
      if (block_lds_bytes(c, kWideBlock / kWave, false) + 4096 <= limit) {
        cap = c;
        break;
      }
    }
    cached = (int)cap;
  }
  return (uint32_t)cached;
}

// Blocks of an LDS-rows tier of this cap resident per CU: limited by LDS
// (160 KiB per CU) and by 32 waves per CU.
int lds_blocks_per_cu(uint32_t cap, int block_threads, bool pad) {
  const size_t lds = block_lds_bytes(cap, block_threads / kWave, pad);
  const int by_waves = std::max(1, 32 / (block_threads / kWave));
  return std::min(by_waves, std::max<int>(1, (int)(160 * 1024 / (lds + 2048))));
}

// One LDS-rows tier: rows of up to MAXW words, cap = its largest out-degree.
template <int K, int MODE, int MAXW, int BS>
int launch_lds_tier(gpm_graph* g, hipStream_t stream, const uint32_t* roots,
                    const uint32_t* parts, uint32_t n_roots, uint32_t cap,
                    unsigned int* queue, unsigned long long* out, unsigned long long* work,
                    const char* name) {
  const int cus = device_cus(g);
  const size_t lds = block_lds_bytes(cap, BS / kWave, MAXW == 8);
  auto kern = clique_block_kernel<K, MODE, true, MAXW, BS>;
  if (lds > 48 * 1024)
    GPM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned blocks =
      (unsigned)std::min<uint64_t>(n_roots, (uint64_t)cus * lds_blocks_per_cu(cap, BS, MAXW == 8));
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(BS), lds, stream, g->toff, g->tadj, g->n,
                     roots, parts, n_roots, cap, queue, nullptr, nullptr, out, work);
  GPM_HIP(hipGetLastError());
  if ((MODE == kCount || MODE == kAll) && stream == g->stream) timing_mark(g, name);
  return GPM_OK;
}

template <int K, int MODE>
int launch_wave_tier(gpm_graph* g, hipStream_t stream, const RootTiers* t, unsigned int* q,
                     unsigned long long* out, unsigned long long* work) {
  const int cus = device_cus(g);
  const uint32_t chunk = t->wave_chunk;
  const uint64_t waves_wanted = (t->n_wave + chunk - 1) / chunk;
  const uint64_t waves = std::min<uint64_t>(waves_wanted, (uint64_t)cus * 32);
  const unsigned blocks =
      (unsigned)std::max<uint64_t>(1, (waves + kTierWaves - 1) / kTierWaves);
  hipLaunchKernelGGL((clique_wave_kernel<K, MODE>), dim3(blocks), dim3(kTierBlock), 0, stream,
                     g->toff, g->tadj, t->d_wave, t->n_wave, chunk, out, work);
  GPM_HIP(hipGetLastError());
  if ((MODE == kCount || MODE == kAll) && stream == g->stream) timing_mark(g, "clique_wave");
  return GPM_OK;
}

// Launches every non-empty tier on the handle's stream, one after another.
// (Running the rows-in-HBM and wave tiers on a second stream beside the LDS
// tiers was measured slower: 254 ms against 230 ms for the learned 5-clique
// count on R-MAT s22, from contention with the LDS tiers.)
template <int K, int MODE>
int launch_tiers(gpm_graph* g, const RootTiers* t, unsigned long long* out,
                 unsigned long long* work) {
  const int cus = device_cus(g);
  unsigned int* q = t->queues;
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, g->stream, q, 4);
  GPM_HIP(hipGetLastError());
  if (t->n_big) {
    const uint32_t cap = t->max_big_deg;
    const uint32_t W = (cap + 63) / 64;
    const unsigned blocks = (unsigned)std::min<uint64_t>(t->n_big, (uint64_t)cus);
    const size_t row_bytes = (size_t)blocks * cap * W * 8;
    const size_t meta_bytes = (size_t)blocks * 2 * cap * 4;
    int st = ensure_scratch(g, row_bytes + meta_bytes + 256);
    if (st != GPM_OK) return st;
    unsigned long long* grows = static_cast<unsigned long long*>(g->scratch);
    uint32_t* gmeta = reinterpret_cast<uint32_t*>(static_cast<char*>(g->scratch) + row_bytes);
    hipLaunchKernelGGL((clique_block_kernel<K, MODE, false, 0, kHbmBlock>), dim3(blocks),
                       dim3(kHbmBlock), 0, g->stream, g->toff, g->tadj, g->n, t->d_big,
                       t->d_big_parts, t->n_big, cap, q + 2, grows, gmeta, out, work);
    GPM_HIP(hipGetLastError());
    if (MODE == kCount || MODE == kAll) timing_mark(g, "clique_hbm_block");
  }
  if (t->n_block2) {
    int st = launch_lds_tier<K, MODE, 16, kWideBlock>(g, g->stream, t->d_block2, t->d_block2_parts,
                                                      t->n_block2, t->max_block2_deg, q + 3, out,
                                                      work, "clique_lds_block_wide");
    if (st != GPM_OK) return st;
  }
  if (t->n_block) {
    int st = launch_lds_tier<K, MODE, 8, kLdsBlock>(g, g->stream, t->d_block, t->d_block_parts,
                                                    t->n_block, t->max_block_deg, q + 1, out, work,
                                                    "clique_lds_block");
    if (st != GPM_OK) return st;
  }
  if (t->n_wave) {
    int st = launch_wave_tier<K, MODE>(g, g->stream, t, q, out, work);
    if (st != GPM_OK) return st;
  }
  return GPM_OK;
}

template <int MODE>
int launch_k(gpm_graph* g, int k, const RootTiers* t, unsigned long long* out,
             unsigned long long* work) {
  if constexpr (MODE == kAll) return launch_tiers<5, MODE>(g, t, out, work);
  else switch (k) {
    case 3: return launch_tiers<3, MODE>(g, t, out, work);
    case 4: return launch_tiers<4, MODE>(g, t, out, work);
    default: return launch_tiers<5, MODE>(g, t, out, work);
  }
}

TierRequest request_from(const gpm_sched* s, uint32_t min_deg) {
  TierRequest r;
  r.min_deg = min_deg;
  r.wave_cap = 64;
  r.block_cap = kBlockCap;
  r.block2_cap = lds_wide_cap();
  if (s) {
    r.root_begin = s->root_begin;
    r.root_end = s->root_end;
    r.policy = s->policy;
    r.cost = s->root_cost;
    r.chunk = s->chunk;
    r.root_list = s->root_list;
    r.n_root_list = s->root_list ? s->n_root_list : 0;
    if (s->wave_cap && s->wave_cap < 64) r.wave_cap = s->wave_cap;
  }
  return r;
}

}  // namespace

namespace gpm {
// Heavy-root threshold for the learned policy: wave roots whose predicted
// cost exceeds it are served by a whole block.
float learned_heavy_cost(const float* cost, uint32_t n);
}

namespace {

// Tier request of one k-clique call.  LEARNED uses the caller's predicted
// costs; DEGREE_SPLIT uses the same ordering, promotion and splitting with
// the plain degree estimate cost(v) = d+(v)^2 (the root's pair count), so
// the two differ only in where the cost comes from; DEGREE keeps the
// reference-style degree order without splitting.
int prepare_request(gpm_graph* g, const gpm_sched* sched, uint32_t min_deg, TierRequest* req,
                    std::vector<float>* deg_cost) {
  GPM_CHECK_ARG(!sched || sched->policy == GPM_SCHED_DEGREE ||
                    sched->policy == GPM_SCHED_LEARNED || sched->policy == GPM_SCHED_DEGREE_SPLIT,
                "unknown scheduling policy");
  GPM_CHECK_ARG(!sched || sched->policy != GPM_SCHED_LEARNED || sched->root_cost,
                "LEARNED policy needs root_cost");
  int st = ensure_topo(g);
  if (st != GPM_OK) return st;
  *req = request_from(sched, min_deg);
  req->rank = g->h_rank.data();
  if (req->policy == GPM_SCHED_DEGREE_SPLIT) {
    deg_cost->resize(g->n);
    for (uint32_t v = 0; v < g->n; ++v) {
      const float d = (float)(g->h_off[v + 1] - g->h_off[v]);
      (*deg_cost)[v] = d * d;
    }
    req->cost = deg_cost->data();
    req->policy = GPM_SCHED_LEARNED;
  }
  if (req->policy == GPM_SCHED_LEARNED) {
    req->heavy_cost = learned_heavy_cost(req->cost, g->n);
    const uint32_t cus = (uint32_t)device_cus(g);
    req->resident_block = cus * lds_blocks_per_cu(req->block_cap, kLdsBlock, true);
    req->resident_block2 = cus * lds_blocks_per_cu(req->block2_cap, kWideBlock, false);
    req->resident_big = cus;
  }
  return GPM_OK;
}

}  // namespace

extern "C" {

int gpm_clique(gpm_graph* g, int k, const gpm_sched* sched, uint64_t* out) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(g && out, "null pointer");
    GPM_CHECK_ARG(g->flags & GPM_GRAPH_ORIENTED, "k-clique counting needs an ORIENTED graph");
    GPM_CHECK_ARG(k >= 3 && k <= 5, "k must be 3, 4 or 5 (got %d)", k);
    TierRequest req;
    std::vector<float> deg_cost;
    int st = prepare_request(g, sched, (uint32_t)(k - 1), &req, &deg_cost);
    if (st != GPM_OK) return st;
    if (k == 4) req.min_part_rows = 16;  // count4_rows deals whole blocks of 16 rows
    const RootTiers* t = nullptr;
    if ((st = get_tiers(g, req, &t)) != GPM_OK) return st;
    if ((st = timing_begin(g)) != GPM_OK) return st;
    if ((st = zero_counters(g, 1)) != GPM_OK) return st;
    if ((st = launch_k<kCount>(g, k, t, g->counters, nullptr)) != GPM_OK) return st;
    unsigned long long h = 0;
    if ((st = timing_end(g, &h, g->counters, sizeof(h))) != GPM_OK) return st;
    *out = h;
    return GPM_OK;
  });
}

int gpm_clique_all(gpm_graph* g, const gpm_sched* sched, uint64_t out[3]) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(g && out, "null pointer");
    GPM_CHECK_ARG(g->flags & GPM_GRAPH_ORIENTED, "k-clique counting needs an ORIENTED graph");
    TierRequest req;
    std::vector<float> deg_cost;
    int st = prepare_request(g, sched, 2u, &req, &deg_cost);  // triangles need d+ >= 2
    if (st != GPM_OK) return st;
    const RootTiers* t = nullptr;
    if ((st = get_tiers(g, req, &t)) != GPM_OK) return st;
    if ((st = timing_begin(g)) != GPM_OK) return st;
    if ((st = zero_counters(g, 3)) != GPM_OK) return st;
    if ((st = launch_k<kAll>(g, 5, t, g->counters, nullptr)) != GPM_OK) return st;
    unsigned long long h[3] = {0, 0, 0};
    if ((st = timing_end(g, h, g->counters, sizeof(h))) != GPM_OK) return st;
    for (int i = 0; i < 3; ++i) out[i] = h[i];
    return GPM_OK;
  });
}

int gpm_clique_tier_caps(uint32_t* wave_cap, uint32_t* lds_cap, uint32_t* wide_cap) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(wave_cap && lds_cap && wide_cap, "null pointer");
    *wave_cap = 64;
    *lds_cap = kBlockCap;
    *wide_cap = lds_wide_cap();
    return GPM_OK;
  });
}

int gpm_clique_plan_bytes(gpm_graph* g, int k, uint64_t* bytes) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(g && bytes, "null pointer");
    GPM_CHECK_ARG(g->flags & GPM_GRAPH_ORIENTED, "needs an ORIENTED graph");
    GPM_CHECK_ARG(k >= 3 && k <= 5, "k must be 3, 4 or 5 (got %d)", k);
    if (!g->plan_bytes[k]) {
      int st = ensure_topo(g);
      if (st != GPM_OK) return st;
      TierRequest req = request_from(nullptr, 1);
      req.rank = g->h_rank.data();
      const RootTiers* t = nullptr;
      st = get_tiers(g, req, &t);
      if (st != GPM_OK) return st;
      if ((st = zero_counters(g, 1)) != GPM_OK) return st;
      if ((st = launch_k<kBytes>(g, k, t, g->counters, nullptr)) != GPM_OK) return st;
      unsigned long long h = 0;
      GPM_HIP(hipMemcpyAsync(&h, g->counters, sizeof(h), hipMemcpyDeviceToHost, g->stream));
      GPM_HIP(hipStreamSynchronize(g->stream));
      g->plan_bytes[k] = h + 4ull * (g->n + 1) + 8ull * g->m;
    }
    *bytes = g->plan_bytes[k];
    return GPM_OK;
  });
}

int gpm_clique_root_work(gpm_graph* g, int k, uint64_t* work) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(g && work, "null pointer");
    GPM_CHECK_ARG(g->flags & GPM_GRAPH_ORIENTED, "needs an ORIENTED graph");
    GPM_CHECK_ARG(k >= 3 && k <= 5, "k must be 3, 4 or 5 (got %d)", k);
    int st = ensure_topo(g);
    if (st != GPM_OK) return st;
    TierRequest req = request_from(nullptr, 1);
    req.rank = g->h_rank.data();
    const RootTiers* t = nullptr;
    st = get_tiers(g, req, &t);
    if (st != GPM_OK) return st;
    unsigned long long* d_work = nullptr;
    GPM_HIP(hipMalloc(&d_work, (size_t)std::max(g->n, 1u) * 8));
    if (hipMemsetAsync(d_work, 0, (size_t)std::max(g->n, 1u) * 8, g->stream) != hipSuccess) {
      (void)hipFree(d_work);
      return fail(GPM_EHIP, "clearing the work log failed");
    }
    st = launch_k<kWork>(g, k, t, g->counters, d_work);
    // The kernels log by topological id; report by vertex id.
    std::vector<uint64_t> by_rank(g->n);
    if (st == GPM_OK) {
      if (hipMemcpyAsync(by_rank.data(), d_work, (size_t)g->n * 8, hipMemcpyDeviceToHost,
                         g->stream) != hipSuccess ||
          hipStreamSynchronize(g->stream) != hipSuccess)
        st = fail(GPM_EHIP, "work log copy failed");
    }
    hipFree(d_work);
    if (st == GPM_OK)
      for (uint32_t v = 0; v < g->n; ++v) work[v] = by_rank[g->h_rank[v]];
    return st;
  });
}

}  // extern "C"
