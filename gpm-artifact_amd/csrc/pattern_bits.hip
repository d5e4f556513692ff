// Fixed patterns on the adjacency bit matrix (both formulations of
// gpm_pattern, see pattern.hip for what each counts).
//
// The nested set operations of the patterns walk sets of vertices and, for
// each, intersect or subtract its neighbours from another set.  As lists those
// are a binary search per entry; here sets and neighbourhoods are rows of bits,
// and the two inner loops of a pattern become one masked product per edge:
//     sum over a in R1, b in R2 with Q(a, b) of |C & X[a] & Y[b]|
// with X, Y one of the matrices below.  16 x 16 pairs (a, b) and 128 columns
// are one FP4 matrix instruction (fp4_bits.hpp).  Q is always "b is in X[a]" or
// its opposite, so it is the product of the same rows of a with the unit
// vectors of b, and lands in the lanes that hold the sizes.
//
//   D01 = N(v0) \ N(v1), D10 = N(v1) \ N(v0), I = N(v0) & N(v1)
//         R1   R2   C    X    direct: Y, Q       counting: Y, Q
//   P2    D10  D01  D01  !N   below, !N   in     above, !N   not in
//   P3    D01  D01  D01  below, !N  below, !N in  above, !N  not in
//   P5    I    D01  D10  !N   !N          in     the same
//   P6    I    I    D10  !N   !N          in     the same
//   P7    I    I    I    below, !N  below, !N in  above, !N  not in
//   P8    D10  I    I    !N   below, N    in     above, N    not in
// (the opposite: an a and b that are adjacent; where X and Y leave no column
// between them the size is 0 whatever Q says).  P1, P4 and the direct Motif4
// have one inner loop: |C & X[a]| summed over a.
//
// A row has n / 512 steps to multiply, whatever the lists' lengths, so this
// path is for graphs of at most kBitsMaxN vertices and not for sparse large
// ones (bits_pay).
#include <algorithm>
#include <cmath>

#include "fp4_bits.hpp"
#include "graph_dev.hpp"

using namespace gpm;

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr uint32_t kBitsMaxN = 16384;
static_assert(kPatternQueue + kQueueShards * kQueueStride <= kCounters, "the queue is in the counters");
// A segment: the 2048 ids whose bits are one word per lane.
constexpr uint32_t kSegWords = kWave, kSegIds = 32 * kSegWords;
// Columns of a step of a product.
constexpr uint32_t kStepIds = 512;
static_assert(kSegIds % kStepIds == 0, "rows are whole steps");
// Entries of a list: a segment's ids, filled up with the empty row's index.
constexpr uint32_t kListLen = kSegIds + kWave;
enum Matrix { kN, kNotN, kBelowNotN, kAboveNotN, kBelowN, kAboveN, kMatrices };

struct Bits {
  const uint32_t* base;  // kMatrices matrices of n + 1 rows of rw words; row n is empty
  uint32_t n, rw;
  __device__ const uint32_t* row(int matrix, uint32_t v) const {
    return base + ((size_t)matrix * (n + 1) + v) * rw;
  }
};

// Bits of word w below / above id v.
__device__ __forceinline__ uint32_t bits_below(uint32_t w, uint32_t v) {
  return w < v / 32 ? 0xFFFFFFFFu : w == v / 32 ? (1u << (v & 31)) - 1u : 0u;
}
__device__ __forceinline__ uint32_t bits_above(uint32_t w, uint32_t v) {
  return w > v / 32 ? 0xFFFFFFFFu : w == v / 32 ? ~((2u << (v & 31)) - 1u) : 0u;
}

// ------------------------------------------------------------- the matrices

// Sets the neighbour bits of every vertex (N zeroed before); one wave per v.
__global__ __launch_bounds__(kBlock) void neighbour_bits_kernel(const uint32_t* __restrict__ off,
                                                                const uint32_t* __restrict__ adj,
                                                                uint32_t n, uint32_t rw,
                                                                uint32_t* __restrict__ bits) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = gridDim.x * blockDim.x / kWave;
  for (uint32_t v = wave; v < n; v += nwaves)
    for (uint32_t i = off[v] + lane_id(); i < off[v + 1]; i += kWave)
      atomicOr(&bits[(size_t)v * rw + adj[i] / 32], 1u << (adj[i] & 31));
}

__global__ __launch_bounds__(kBlock) void zero_words_kernel(uint32_t* p, uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

// The other matrices from N; total[0] += the bits of N, total[1] += those whose mirror
// is set.
__global__ __launch_bounds__(kBlock) void derived_bits_kernel(uint32_t* __restrict__ base,
                                                              uint32_t n, uint32_t rw,
                                                              unsigned long long* __restrict__ total) {
  const uint64_t words = (uint64_t)(n + 1) * rw;
  uint64_t set = 0, mirrored = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t v = (uint32_t)(i / rw), w = (uint32_t)(i % rw);
    const uint32_t m = base[i];
    const uint32_t ids = v < n ? bits_below(w, n) : 0u;  // row n stays empty
    const uint32_t lo = ids & bits_below(w, v), hi = ids & bits_above(w, v);
    base[kNotN * words + i] = ~m & ids;
    base[kBelowNotN * words + i] = ~m & lo;
    base[kAboveNotN * words + i] = ~m & hi;
    base[kBelowN * words + i] = m & lo;
    base[kAboveN * words + i] = m & hi;
    set += (uint32_t)__popc(m);
    for (uint32_t b = m; b; b &= b - 1)
      mirrored += (base[(32 * w + (uint32_t)__builtin_ctz(b)) * (uint64_t)rw + v / 32] >> (v & 31)) & 1u;
  }
  block_add(&total[0], set);
  block_add(&total[1], mirrored);
}

// ---------------------------------------------------------------- the count

// The set bits of as many segments from *seg on (word(w): word w of the set) as fit the
// list, as ascending ids, filled up with `none` to a multiple of 64; returns how
// many there are and moves *seg on.  (A list per segment padded every segment's few ids
// to a block: Erdos-Renyi n = 16384, degree 46, 64 pairs of blocks an edge for the 9 that
// hold its ids, 374 ms for the direct P2, 28.5 now; lists 441.)
template <typename F>
__device__ __forceinline__ uint32_t list_bits(F&& set_word, uint32_t* seg, uint32_t segs,
                                              uint32_t none, uint16_t* list) {
  uint32_t total = 0;
  __builtin_amdgcn_wave_barrier();
  for (uint32_t s = uniform(*seg); s < segs; ++s) {
    uint32_t word = set_word(s * kSegWords + lane_id());
    const uint32_t incl = wave_incl_scan((uint32_t)__popc(word));
    const uint32_t here = uniform(wave_bcast(incl, kWave - 1));
    if (total + here > kSegIds) break;  // the next list's
    uint32_t at = total + incl - (uint32_t)__popc(word);
    const uint32_t id0 = s * kSegIds + 32 * lane_id();
    for (; word; word &= word - 1) list[at++] = (uint16_t)(id0 + __builtin_ctz(word));
    total += here;
    *seg = s + 1;
  }
  list[total + lane_id()] = (uint16_t)none;
  __builtin_amdgcn_wave_barrier();
  return total;
}

struct Product {
  const uint32_t *x, *y;   // matrices of a's and b's rows
  const uint32_t *ca, *cb; // column sets of X[a] (with R2's ids for Q) and of Y[b], in LDS
  uint32_t rw, steps;      // words of a row; steps of kStepIds columns that hold ids
  bool in;                 // Q: b in X[a], or not
};

// Blocks ja .. ja + J - 1 of R1 (list a) against blocks lb .. lb + L - 1 of R2.
// A step takes 512 columns: a lane loads four words of a row together (64 bytes of
// every row, where a word each left the wave 16 bytes of 16 lines), and matrix
// instruction k of the step multiplies word k of every lane, the same columns on both
// sides.  The sizes of all J x L tiles accumulate over the steps; the adjacency of
// one block of b at a time then masks its column of tiles.  A lane's sum stays
// below 2^24: 4 J L sizes of at most kBitsMaxN.
template <int J, int L>
__device__ __forceinline__ uint32_t product_tiles(const Product& p, const uint16_t* a,
                                                  const uint16_t* b, uint32_t ja, uint32_t lb) {
  static_assert(4ull * J * L * kBitsMaxN < (1ull << 24), "sums must be exact");
  const uint32_t lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  uint32_t ra[J], rb[L], ib[L];
#pragma unroll
  for (int q = 0; q < J; ++q) ra[q] = a[16 * (ja + q) + r16] * p.rw + 4 * g;
#pragma unroll
  for (int q = 0; q < L; ++q) {
    ib[q] = b[16 * (lb + q) + r16];
    rb[q] = ib[q] * p.rw + 4 * g;
  }
  floatx4 both[J][L];
#pragma unroll
  for (int q = 0; q < J; ++q)
#pragma unroll
    for (int t = 0; t < L; ++t) both[q][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto four = [](const uint32_t* w) { return *reinterpret_cast<const uintx4*>(w); };
  for (uint32_t c = 0; c < p.steps; ++c) {
    const uintx4 ca = four(p.ca + 16 * c + 4 * g), cb = four(p.cb + 16 * c + 4 * g);
    if (wave_ballot((cb.x | cb.y | cb.z | cb.w) != 0u) == 0ull) continue;
    uintx4 wa[J], wb[L];
#pragma unroll
    for (int q = 0; q < J; ++q) wa[q] = four(p.x + ra[q] + 16 * c);
#pragma unroll
    for (int t = 0; t < L; ++t) wb[t] = four(p.y + rb[t] + 16 * c);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      intx4 fb[L];
#pragma unroll
      for (int t = 0; t < L; ++t) fb[t] = fp4_in_place(wb[t][k] & cb[k]);
#pragma unroll
      for (int q = 0; q < J; ++q) {
        const intx4 fa = fp4_reciprocal(wa[q][k] & ca[k]);
#pragma unroll
        for (int t = 0; t < L; ++t) both[q][t] = mfma_fp4(fa, fb[t], both[q][t]);
      }
    }
  }
  float sum = 0.f;
#pragma unroll
  for (int t = 0; t < L; ++t) {
    floatx4 adj[J];
#pragma unroll
    for (int q = 0; q < J; ++q) adj[q] = floatx4{0.f, 0.f, 0.f, 0.f};
    // b's ascend, the empty row (index n) last: it has no column.
    const uint32_t first = uniform(ib[t]) / kStepIds;
    const uint32_t last = min(__builtin_amdgcn_readlane(ib[t], 15) / kStepIds, p.steps - 1);
    const uint32_t word = ib[t] / 32 - 4 * g, bit = 1u << (ib[t] & 31);
    for (uint32_t c = first; c <= last; ++c) {
      // Ids of several segments may leave steps out.
      if (p.steps > kSegIds / kStepIds && wave_ballot(ib[t] / kStepIds == c) == 0ull) continue;
      const uintx4 ca = four(p.ca + 16 * c + 4 * g);
      uintx4 wa[J];
#pragma unroll
      for (int q = 0; q < J; ++q) wa[q] = four(p.x + ra[q] + 16 * c);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t w = word == 16 * c + k ? bit : 0u;
        if (wave_ballot(w != 0u) == 0ull) continue;
        const intx4 e = fp4_in_place(w);
#pragma unroll
        for (int q = 0; q < J; ++q) adj[q] = mfma_fp4(fp4_reciprocal(wa[q][k] & ca[k]), e, adj[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < J; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sum = __builtin_fmaf(both[q][t][r], p.in ? adj[q][r] : 1.f - adj[q][r], sum);
  }
  return (uint32_t)sum;
}

// The pairs of two short lists one by one, each lane some of the columns: where a row has
// many steps, a tile of mostly empty rows takes longer.  Erdos-Renyi n = 16384, degree
// 80, P6 (0.4 common neighbours an edge): 6.8 ms in tiles, 4.5 so.
constexpr uint32_t kFewPairs = 4;
__device__ __forceinline__ uint64_t few_pairs(const Product& p, const uint16_t* a, uint32_t na,
                                              const uint16_t* b, uint32_t nb) {
  uint32_t sum = 0;
  for (uint32_t i = 0; i < na; ++i) {
    const uint32_t* x = p.x + uniform(a[i]) * p.rw;
    for (uint32_t j = 0; j < nb; ++j) {
      const uint32_t ib = uniform(b[j]);
      const uint32_t* y = p.y + ib * p.rw;
      const bool in = ((x[ib / 32] & p.ca[ib / 32]) >> (ib & 31)) & 1u;
      uint32_t c = 0;
      for (uint32_t w = lane_id(); w < 16 * p.steps; w += kWave)
        c += (uint32_t)__popc(x[w] & p.ca[w] & y[w] & p.cb[w]);
      if (in == p.in) sum += c;
    }
  }
  return sum;
}

// Every pair of the lists a (na entries) and b (nb); triangular: only pairs with
// b's block up to a's count (lists of one set, X or Y leave nothing beyond).
__device__ __forceinline__ uint64_t product(const Product& p, const uint16_t* a, uint32_t na,
                                            const uint16_t* b, uint32_t nb, bool triangular) {
  const uint32_t ta = (na + 15) / 16, tb = (nb + 15) / 16;
  uint64_t sum = 0;
  uint32_t ja = 0;
  while (ja < ta) {
    const uint32_t left = ta - ja, step = left >= 3 ? 4 : left;
    const uint32_t end = triangular ? min(tb, ja + step) : tb;
    for (uint32_t lb = 0; lb < end; lb += 4) {
      if (step == 4)
        sum += end - lb == 1 ? product_tiles<4, 1>(p, a, b, ja, lb) : product_tiles<4, 4>(p, a, b, ja, lb);
      else if (step == 2)
        sum += end - lb == 1 ? product_tiles<2, 1>(p, a, b, ja, lb) : product_tiles<2, 4>(p, a, b, ja, lb);
      else
        sum += end - lb == 1 ? product_tiles<1, 1>(p, a, b, ja, lb) : product_tiles<1, 4>(p, a, b, ja, lb);
    }
    ja += step;
  }
  return sum;
}

// sum over the ids v of the list of |C & X[v]|, this lane's share; the set in
// LDS, four rows at a time.
__device__ __forceinline__ uint64_t sum_rows(const uint32_t* x, const uint32_t* set, uint32_t rw,
                                             uint32_t words, const uint16_t* list, uint32_t n) {
  uint64_t sum = 0;
  for (uint32_t t = 0; t < n; t += 4) {
    // The list is filled up with the empty row.
    const uint32_t* r0 = x + uniform(list[t]) * (size_t)rw;
    const uint32_t* r1 = x + uniform(list[t + 1]) * (size_t)rw;
    const uint32_t* r2 = x + uniform(list[t + 2]) * (size_t)rw;
    const uint32_t* r3 = x + uniform(list[t + 3]) * (size_t)rw;
    uint32_t c = 0;
    for (uint32_t w = lane_id(); w < words; w += kWave) {
      const uint32_t s = set[w];
      c += (uint32_t)__popc(r0[w] & s) + (uint32_t)__popc(r1[w] & s) +
           (uint32_t)__popc(r2[w] & s) + (uint32_t)__popc(r3[w] & s);
    }
    sum += c;
  }
  return sum;
}

// sum over the ids v of the list of |S & X[v]| |T & Y[v]| (one lane's share):
// the two sizes are summed over the wave in the halves of one word.
__device__ __forceinline__ uint64_t sum_products(const uint32_t* x, const uint32_t* s,
                                                 const uint32_t* y, const uint32_t* t, uint32_t rw,
                                                 uint32_t words, const uint16_t* list, uint32_t n) {
  static_assert(kBitsMaxN < (1u << 16), "two sizes in a word");
  uint64_t sum = 0;
  for (uint32_t k = 0; k < n; k += 4) {
    uint32_t c[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const size_t r = uniform(list[k + q]) * (size_t)rw;
      c[q] = 0;
      for (uint32_t w = lane_id(); w < words; w += kWave)
        c[q] += (uint32_t)__popc(x[r + w] & s[w]) | (uint32_t)__popc(y[r + w] & t[w]) << 16;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) c[q] = wave_sum_u32(c[q]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (lane_id() == (uint32_t)q) sum += (uint64_t)(c[q] & 0xFFFFu) * (c[q] >> 16);
  }
  return sum;
}

// One wave per directed edge, in chunks from a queue.  LDS per wave: two lists
// and two sets of rw words.  ONE: the graph has one segment.  SUMS: the
// frequency sums too (the counting P2, P3, P7, P8), which spilled scalars slow down, so
// several segments have an instance without them.  PRODUCTS: P2, P3, P5 - P8 (16 tiles of sizes and
// their operands: 226 registers, 2 waves per SIMD; bounds that make it spill are
// not safe, as matrix instructions read every lane's register); otherwise P1,
// P4 and Motif4.  R-MAT, 16 edges a vertex, all of P1 - P8 and Motif4: n = 512
// direct 362 ms on lists, 1.0 ms here; n = 2048 counting 982 ms, 8.0 ms, a third
// of it P3 (3.2 M blocks of 16 x 16 pairs, 4 steps each): latency of the row loads
// bounds it, at two waves per SIMD (four with half the tiles: 9.3 ms).  The chunks come from kQueueShards
// counters, and a block adds its sums up: additions to one address take about
// 10 ns each, and with one counter and a sum per wave they were most of the n = 512
// launches (P1 - P8 and Motif4: 1.71 ms so, 1.26 now).
template <bool PRODUCTS, bool ONE, bool SUMS>
__global__ __launch_bounds__(kBlock, PRODUCTS ? 2 : 4) void pattern_bits_kernel(
    const uint32_t* __restrict__ adj, const uint32_t* __restrict__ src, uint64_t m, Bits g,
    int pid, bool counting, uint32_t chunk, unsigned long long* __restrict__ queue,
    unsigned long long* __restrict__ out) {
  extern __shared__ __align__(16) uint32_t s_words[];
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  const uint32_t per_wave = 2 * g.rw + kListLen;  // words: two sets, two lists of halves
  uint32_t* s0 = s_words + wave * per_wave;
  uint32_t* s1 = s0 + g.rw;
  uint16_t* l0 = reinterpret_cast<uint16_t*>(s1 + g.rw);
  uint16_t* l1 = l0 + kListLen;
  const uint32_t segs = ONE ? 1u : g.rw / kSegWords, words = (g.n + 31) / 32, steps = (g.n + kStepIds - 1) / kStepIds;
  const uint32_t none = g.n;
  uint64_t c[6] = {0, 0, 0, 0, 0, 0};
  const uint32_t n_chunks = (uint32_t)((m + chunk - 1) / chunk);
  uint32_t shard = blockIdx.x % kQueueShards, drained = 0;
  while (true) {
    // Each counter deals out every kQueueShards-th chunk; other blocks' are read before
    // they are added to, since most are drained by then.
    const uint32_t mine = n_chunks > shard ? (n_chunks - shard - 1) / kQueueShards + 1 : 0u;
    unsigned long long* counter = queue + shard * kQueueStride;
    uint32_t t = 0;
    if (lane == 0)
      t = drained && __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= mine
              ? mine
              : (uint32_t)atomicAdd(counter, 1ull);
    t = uniform(wave_bcast(t, 0));
    if (t >= mine) {
      shard = (shard + 1) % kQueueShards;
      if (++drained == kQueueShards) break;
      continue;
    }
    const uint64_t base = ((uint64_t)t * kQueueShards + shard) * chunk;
    const uint64_t stop = min(m, base + chunk);
    for (uint64_t e = base; e < stop; ++e) {
      const uint32_t v0 = uniform(src[e]), v1 = uniform(adj[e]);
      if (v0 == v1 || (pid == 4 && v1 >= v0)) continue;
      const uint32_t *n0 = g.row(kN, v0), *n1 = g.row(kN, v1);
      // Word w of the sets of the edge.
      auto d01 = [&](uint32_t w) { return n0[w] & ~n1[w]; };
      auto d10 = [&](uint32_t w) { return n1[w] & ~n0[w]; };
      auto both = [&](uint32_t w) { return n0[w] & n1[w]; };
      auto fill = [&](uint32_t* set, auto f) {
        __builtin_amdgcn_wave_barrier();
        for (uint32_t w = lane; w < g.rw; w += kWave) set[w] = f(w);
        __builtin_amdgcn_wave_barrier();
      };
      // sum over a in R of |set & X[a]|
      auto sums = [&](auto r, int x, const uint32_t* set) {
        uint64_t t = 0;
        for (uint32_t k = 0; k < segs;) {
          const uint32_t na = list_bits(r, &k, segs, none, l0);
          t += sum_rows(g.row(x, 0), set, g.rw, words, l0, na);
        }
        return t;
      };
      if (!PRODUCTS && pid == 1) {
        auto r = [&](uint32_t w) { return d01(w) & bits_below(w, v1); };
        fill(s0, r);
        c[0] += sums(r, kBelowNotN, s0);
      } else if (!PRODUCTS && pid == 4) {
        fill(s0, d10);
        const uint64_t t = sums(d01, kNotN, s0);
        (counting ? c[1] : c[0]) += t;
      } else if (!PRODUCTS) {
        auto star = [&](uint32_t w) { return d01(w) & bits_below(w, v1); };
        fill(s0, star);
        c[0] += sums(star, kBelowNotN, s0);
        if (v1 > v0) continue;
        fill(s0, both);
        fill(s1, [&](uint32_t w) { return ~n0[w] & ~n1[w]; });
        c[4] += sums(both, kBelowNotN, s0);
        c[2] += sums(both, kN, s1);
        auto top = [&](uint32_t w) { return both(w) & bits_below(w, v1); };
        fill(s0, top);
        c[5] += sums(top, kBelowN, s0);
        fill(s0, d10);
        c[1] += sums(d01, kNotN, s0);
        fill(s0, [&](uint32_t w) { return d10(w) & bits_below(w, v0); });
        c[3] += sums([&](uint32_t w) { return d01(w) & bits_below(w, v1); }, kN, s0);
      } else {
        const bool wedge = pid == 3 || pid == 7, pairs = pid == 5 || pid == 6;
        const bool i1 = pairs || pid == 7, i2 = pid >= 6;
        auto r1 = [&](uint32_t w) { return i1 ? both(w) : wedge ? d01(w) : d10(w); };
        auto r2 = [&](uint32_t w) { return i2 ? both(w) : d01(w); };
        // Edges without a common neighbour, or whose ends share all of them,
        // often have nothing to count: R1 and R2 need an entry each, R2 two in P2 and P8
        // (b and one of its columns) and three in P3 and P7 (and an a).
        const uint32_t least = wedge ? 3u : pairs ? 1u : 2u;
        uint32_t any1 = 0, in2 = 0;
        for (uint32_t w = lane; w < g.rw; w += kWave) {
          any1 |= r1(w);
          in2 += (uint32_t)__popc(r2(w));
        }
        if (wave_ballot(any1 != 0u) == 0ull) continue;
        const uint32_t lanes = (uint32_t)__popcll(wave_ballot(in2 != 0u));
        if (lanes < least && (lanes == 0u || uniform(wave_sum_u32(in2)) < least)) continue;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t w = lane; w < g.rw; w += kWave) {
          const uint32_t r = r2(w), d = pairs ? d10(w) : 0u;
          s0[w] = r | d;
          if (pairs) s1[w] = d;
        }
        __builtin_amdgcn_wave_barrier();
        // R2, and R1 where it is the same set, off the words in LDS.
        auto set2 = [&](uint32_t w) { return pairs ? s0[w] & ~s1[w] : s0[w]; };
        auto set1 = [&](uint32_t w) { return wedge || pid == 6 ? set2(w) : r1(w); };
        Product p;
        p.x = g.row(wedge ? kBelowNotN : kNotN, 0);
        p.y = g.row(pairs ? kNotN
                    : pid == 8 ? (counting ? kAboveN : kBelowN)
                               : (counting ? kAboveNotN : kBelowNotN), 0);
        p.ca = s0;
        p.cb = pairs ? s1 : s0;
        p.rw = g.rw;
        p.steps = steps;
        p.in = pairs || !counting;
        uint64_t t = 0;
        for (uint32_t k = 0; k < segs;) {
          const uint32_t first = k, na = list_bits(set1, &k, segs, none, l0);
          if (!na) continue;
          // One set's lists are cut at the same segments.
          for (uint32_t k2 = 0; k2 < (wedge ? k : segs);) {
            const bool same = wedge && k2 == first;
            const uint32_t nb = list_bits(set2, &k2, segs, none, l1);
            if (!ONE && !SUMS && na * nb <= kFewPairs)
              t += few_pairs(p, l0, na, l1, nb);
            else if (nb)
              t += product(p, l0, na, l1, nb, same);
          }
        }
        if (!counting) {
          c[0] += t;
        } else if (pairs) {
          c[1] += t;
        } else if (SUMS) {
          c[2] += t;
          // Frequency times count per v in R2 (s0): P2, P8: non-neighbours in
          // D10 times the entries of R2 below v; P3, P7: non-neighbours in R2
          // below times above.
          if (!wedge) fill(s1, d10);
          const uint32_t* x = g.row(wedge ? kAboveNotN : kNotN, 0);
          const uint32_t* y = g.row(pid == 8 ? kBelowN : kBelowNotN, 0);
          for (uint32_t k = 0; k < segs;) {
            const uint32_t nb = list_bits(set2, &k, segs, none, l1);
            c[1] += sum_products(x, wedge ? s0 : s1, y, s0, g.rw, words, l1, nb);
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < (PRODUCTS ? 3 : 6); ++i) block_add(&out[i], c[i]);
}

unsigned grid_of(const gpm_graph* g, uint64_t threads) {
  return (unsigned)std::max<uint64_t>(
      1, std::min<uint64_t>((threads + kBlock - 1) / kBlock, (uint64_t)device_cus(g) * 16));
}

// Whether the matrix path is the faster one for the pattern.  Up to one segment it is
// everywhere (a half of the lists' time on sparse graphs, a hundredth on dense or skewed
// ones).  Beyond, an edge costs it n / 2048 segments of set work and a block pair n / 512
// steps, and lists the pairs of its sets, so the lists get longer with the graph: dw =
// sum d^2 / sum d >= 16 sqrt(n / 2048).  On skewed lists the hubs' edges, one wave's
// work each, bound the list kernels: matrix / list ms on R-MAT n = 16384, 31762
// entries, P2 1.8 / 480, counting 3.7 / 20; counting P3 5.3 / 43.  On lists of
// about one length the patterns that are cheap on lists cross later, measured on
// Erdos-Renyi graphs:
//   counting P3 (its sums read whole rows):  n = 8192: dw = 32 8.9 / 6.5, 65 34 / 41;
//                                            n = 16384: 81 215 / 168, 129 569 / 661
//   counting P2:  n = 16384: dw = 47 71 / 58, 81 264 / 373;  n = 8192: 32 9.6 / 12.5
//   P1:           n = 16384: dw = 47 6.3 / 5.5, 81 16 / 20;  Motif4: 47 17 / 13, 57 23 / 21
// Vertices of few common neighbours leave the matrices up to 1.3 times the lists' time in
// P5 - P7 (n = 16384, dw = 101, P6 7.1 / 5.5); where there are some they take a fifth
// (groups of 200 in n = 16000: P6 19 / 86), which the degrees do not tell.
bool bits_pay(gpm_graph* g, int pid, bool counting) {
  if (g->n > kBitsMaxN || !g->m) return false;
  if (g->n <= kSegIds) return true;
  const double segs = (double)g->n / kSegIds, dw = mean_met_degree(g);
  if (dw < 16.0 * std::sqrt(segs)) return false;
  if (segs <= 2.0) return true;
  if (pid == GPM_P1) return dw >= 8.0 * segs || g->met_skew >= 1.5;
  if (pid == GPM_MOTIF4) return dw >= 7.0 * segs || g->met_skew >= 1.5;
  if (counting && pid == GPM_P2) return dw >= 8.0 * segs || g->met_skew >= 2.5;
  if (counting && pid == GPM_P3) return dw >= 14.0 * segs || g->met_skew >= 2.5;
  return true;
}

// Builds g->nbits if missing; *ok is false where the lists hold an entry twice
// (a bit cannot) or the matrices do not fit.
int ensure_bits(gpm_graph* g, bool* ok) {
  *ok = g->nbits != nullptr;
  if (g->nbits || g->nbits_off) return GPM_OK;
  const uint32_t rw = (g->n + kSegIds - 1) / kSegIds * kSegWords;
  const uint64_t words = (uint64_t)(g->n + 1) * rw;
  uint32_t* bits = nullptr;
  if (hipMalloc(&bits, kMatrices * words * 4) != hipSuccess) {
    (void)hipGetLastError();
    g->nbits_off = true;
    return GPM_OK;
  }
  unsigned long long set[2] = {0, 0};
  int st = zero_counters(g, 2);
  if (st == GPM_OK) {
    hipLaunchKernelGGL(zero_words_kernel, dim3(grid_of(g, words)), dim3(kBlock), 0, g->stream, bits,
                       words);
    hipLaunchKernelGGL(neighbour_bits_kernel, dim3(grid_of(g, (uint64_t)g->n * kWave)), dim3(kBlock),
                       0, g->stream, g->off, g->adj, g->n, rw, bits);
    hipLaunchKernelGGL(derived_bits_kernel, dim3(grid_of(g, words)), dim3(kBlock), 0, g->stream,
                       bits, g->n, rw, g->counters);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(set, g->counters, sizeof(set), hipMemcpyDeviceToHost, g->stream) !=
            hipSuccess ||
        hipStreamSynchronize(g->stream) != hipSuccess)
      st = fail(GPM_EHIP, "adjacency bit matrices");
  }
  if (st != GPM_OK || set[0] != g->m) {
    (void)hipStreamSynchronize(g->stream);
    (void)hipFree(bits);
    g->nbits_off = st == GPM_OK;
    return st;
  }
  g->nbits = bits;
  g->nbits_mirrored = set[1] == set[0];
  *ok = true;
  return GPM_OK;
}

}  // namespace

namespace gpm {

int prepare_pattern_bits(gpm_graph* g, int pid, bool counting, bool* ok) {
  *ok = false;
  if (!bits_pay(g, pid, counting)) return GPM_OK;
  const bool pairs = counting && (pid == GPM_P4 || pid == GPM_P5 || pid == GPM_P6);
  const int st = ensure_bits(g, ok);
  // The lists take a pair's adjacency from the end of the shorter list, the matrices from
  // one side: the same only where every edge is in both its lists.
  if (pairs && !g->nbits_mirrored) *ok = false;
  return st != GPM_OK || !*ok ? st : ensure_src(g);
}

int launch_pattern_bits(gpm_graph* g, int pid, bool counting, unsigned long long* queue,
                        unsigned long long* out) {
  Bits b;
  b.base = g->nbits;
  b.n = g->n;
  b.rw = (g->n + kSegIds - 1) / kSegIds * kSegWords;
  const size_t lds = (size_t)kWaves * (2 * b.rw + kListLen) * 4;
  const unsigned per_cu = (unsigned)std::min<size_t>(3, 160 * 1024 / (lds + 1024));
  const uint32_t chunk = 2;
  const unsigned blocks = (unsigned)std::min<uint64_t>(
      (g->m + (uint64_t)chunk * kWaves - 1) / (chunk * kWaves), (uint64_t)device_cus(g) * per_cu);
  const bool products = pid != GPM_P1 && pid != GPM_P4 && pid != GPM_MOTIF4;
  const bool one = g->n <= kSegIds, sums = counting && pid != GPM_P5 && pid != GPM_P6;
  auto kern = !products ? (one ? pattern_bits_kernel<false, true, false>
                               : pattern_bits_kernel<false, false, false>)
              : one  ? pattern_bits_kernel<true, true, true>
              : sums ? pattern_bits_kernel<true, false, true>
                     : pattern_bits_kernel<true, false, false>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kBlock), lds, g->stream, g->adj, g->src, g->m, b,
                     pid, counting, chunk, queue, out);
  GPM_HIP(hipGetLastError());
  timing_mark(g, counting ? "pattern_counting" : "pattern_direct");
  return GPM_OK;
}

}  // namespace gpm
