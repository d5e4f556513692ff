// Batched sorted-set operations (gpm_setops): one wave per list pair, with
// the membership test picked by `variant` -- the primitives of
// src/graph/search.cuh, set_intersection.cuh and set_difference.cuh, each
// rewritten for wave64:
//
//   GPM_SETV_BINARY     each lane binary-searches its entry of A in B
//                       (search.cuh:20-35).
//   GPM_SETV_TWO_PHASE  64 pivots B[k*|B|/64] are staged in LDS; a lane
//                       bisects the pivots in LDS, then searches one 1/64
//                       slice of B in HBM (binary_search_2phase,
//                       search.cuh:54-87; 64 pivots instead of 32, and no
//                       read of B[0] when B is empty).
//   GPM_SETV_MERGE      merge path: the merged order of A and B is cut into
//                       64 equal diagonal segments, one per lane; each lane
//                       finds its cut by a binary search on the diagonal and
//                       merges its segment sequentially (no per-entry search).
//   GPM_SETV_HASH       B goes into an open-addressed LDS table of the wave
//                       (|B| <= kHashCap, else binary search), lanes probe it.
//   GPM_SETV_BITMAP     B goes into an LDS bitmap over [B[0], B[|B|-1]]
//                       (span <= kBitmapBits, else binary search).
//
// Operations (A is iterated, B probed; A \ B never swaps the operands,
// set_difference.cuh:98-234; A & B iterates A as given):
//   ISECT_COUNT / ISECT  |{x in A & B : x < ub}| / the list
//   DIFF_COUNT / DIFF    |{x in A \ B : x < ub}| / the list
//   FUSE                 one pass giving A \ B, A & B and B \ A, with the
//                        matched entries of B marked as they are found
//                        (fuse_set, set_difference.cuh:236-325); returns
//                        the three sizes.
// Materialised lists are sorted and written at the pair's offset into the
// caller's buffers.
#include <algorithm>
#include <vector>

#include "device_common.hpp"
#include "setops.hpp"

using namespace gpm;

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr uint32_t kHashCap = 512;              // B entries an LDS table takes
constexpr uint32_t kHashSlots = 2 * kHashCap;   // load factor <= 1/2
constexpr uint32_t kBitmapBits = 32 * 1024;     // span of ids an LDS bitmap covers
constexpr uint32_t kNoMatch = 0xFFFFFFFFu;

struct WaveLds {
  uint32_t pivots[kWave];
  uint32_t keys[kHashSlots];
  uint32_t vals[kHashSlots];
};  // the bitmap reuses keys+vals (2 * kHashSlots words = kBitmapBits bits)
static_assert(2 * kHashSlots * 32 >= kBitmapBits, "bitmap does not fit the LDS area");

// Position of key in sorted b[lo, hi), or kNoMatch.
__device__ __forceinline__ uint32_t search_range(const uint32_t* __restrict__ b, uint32_t lo,
                                                 uint32_t hi, uint32_t key) {
  uint32_t n = hi - lo;
  if (n == 0) return kNoMatch;
  uint32_t at = lo;
  while (n > 1) {
    const uint32_t half = n >> 1;
    at = b[at + half] <= key ? at + half : at;
    n -= half;
  }
  return b[at] == key ? at : kNoMatch;
}

// Probe state of one wave for one pair: the variant actually used (table
// variants fall back to binary search when B does not fit) and its LDS.
struct Probe {
  int variant;
  const uint32_t* b;
  uint32_t nb;
  uint32_t base;  // bitmap: id of bit 0
  WaveLds* lds;
};

__device__ Probe make_probe(int variant, const uint32_t* b, uint32_t nb, WaveLds* lds) {
  const uint32_t lane = lane_id();
  Probe p{variant, b, nb, 0, lds};
  if (variant == GPM_SETV_HASH && nb > kHashCap) p.variant = GPM_SETV_BINARY;
  if (variant == GPM_SETV_BITMAP && (nb == 0 || b[nb - 1] - b[0] >= kBitmapBits))
    p.variant = nb == 0 ? GPM_SETV_HASH : GPM_SETV_BINARY;  // empty B: an empty table
  if (p.variant == GPM_SETV_TWO_PHASE) {
    if (nb) lds->pivots[lane] = b[(uint32_t)(((uint64_t)lane * nb) / kWave)];
  } else if (p.variant == GPM_SETV_HASH) {
    for (uint32_t i = lane; i < kHashSlots; i += kWave) lds->keys[i] = kEmpty;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t i = lane; i < nb; i += kWave) lds_hash_insert(lds->keys, lds->vals, kHashSlots - 1, b[i], i);
  } else if (p.variant == GPM_SETV_BITMAP) {
    uint32_t* bits = lds->keys;
    p.base = b[0];
    for (uint32_t i = lane; i < 2 * kHashSlots; i += kWave) bits[i] = 0u;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t i = lane; i < nb; i += kWave) {
      const uint32_t o = b[i] - p.base;
      atomicOr(&bits[o >> 5], 1u << (o & 31));
    }
  }
  __builtin_amdgcn_wave_barrier();
  return p;
}

// Position of x in B, or kNoMatch (bitmap: 0 for a hit, positions unknown).
__device__ __forceinline__ uint32_t probe(const Probe& p, uint32_t x) {
  switch (p.variant) {
    case GPM_SETV_TWO_PHASE: {
      if (p.nb == 0) return kNoMatch;
      const uint32_t* piv = p.lds->pivots;
      uint32_t k = 0;  // last pivot <= x (pivot 0 is B[0])
#pragma unroll
      for (uint32_t step = kWave / 2; step > 0; step >>= 1)
        k = piv[k + step] <= x ? k + step : k;
      if (piv[0] > x) return kNoMatch;
      const uint32_t lo = (uint32_t)(((uint64_t)k * p.nb) / kWave);
      const uint32_t hi = (uint32_t)(((uint64_t)(k + 1) * p.nb) / kWave);
      return search_range(p.b, lo, max(hi, lo + 1u), x);
    }
    case GPM_SETV_HASH: {
      const int v = lds_hash_find(p.lds->keys, p.lds->vals, kHashSlots - 1, x);
      return v < 0 ? kNoMatch : (uint32_t)v;
    }
    case GPM_SETV_BITMAP: {
      if (x < p.base || x - p.base >= kBitmapBits) return kNoMatch;
      const uint32_t o = x - p.base;
      return (p.lds->keys[o >> 5] >> (o & 31)) & 1u ? 0u : kNoMatch;
    }
    default:
      return search_range(p.b, 0, p.nb, x);
  }
}

// Merge-path cut of diagonal d between sorted A (na) and B (nb): the number
// of A entries among the first d entries of the merged order (A before B on
// ties, so a match A[i] == B[j] is consumed A first).
__device__ __forceinline__ uint32_t merge_cut(const uint32_t* a, uint32_t na, const uint32_t* b,
                                              uint32_t nb, uint32_t d) {
  uint32_t lo = d > nb ? d - nb : 0, hi = min(d, na);
  while (lo < hi) {
    const uint32_t i = (lo + hi) >> 1;  // i A entries, d - i B entries taken?
    if (a[i] <= b[d - i - 1])
      lo = i + 1;
    else
      hi = i;
  }
  return lo;
}

// Merge-path pass: every lane walks its diagonal segment and calls
// f(i, match) for each A entry i it consumes, match = position in B or
// kNoMatch.  An A entry equal to the next unconsumed B entry is a match
// (that B entry may lie past the segment).
template <typename F>
__device__ __forceinline__ void merge_walk(const uint32_t* a, uint32_t na, const uint32_t* b,
                                           uint32_t nb, F&& f) {
  const uint32_t lane = lane_id();
  const uint64_t total = (uint64_t)na + nb;
  const uint32_t d0 = (uint32_t)(total * lane / kWave), d1 = (uint32_t)(total * (lane + 1) / kWave);
  uint32_t i = merge_cut(a, na, b, nb, d0), j = d0 - i;
  for (uint32_t d = d0; d < d1; ++d) {
    if (i < na && (j >= nb || a[i] <= b[j])) {
      f(i, (j < nb && a[i] == b[j]) ? j : kNoMatch);
      ++i;
    } else {
      ++j;
    }
  }
}

__global__ __launch_bounds__(kBlock) void setops_kernel(
    int op, int variant, uint32_t n_pairs, const uint64_t* __restrict__ a_off,
    const uint32_t* __restrict__ a_all, const uint64_t* __restrict__ b_off,
    const uint32_t* __restrict__ b_all, const uint32_t* __restrict__ ubs,
    unsigned long long* __restrict__ counts, uint32_t* __restrict__ out_a,
    uint32_t* __restrict__ out_ab, uint32_t* __restrict__ out_b) {
  __shared__ WaveLds s_lds[kWavesPerBlock];
  WaveLds* lds = &s_lds[threadIdx.x / kWave];
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = gridDim.x * blockDim.x / kWave;
  const bool keep_in = op == GPM_SETOP_ISECT_COUNT || op == GPM_SETOP_ISECT;
  const bool write = op == GPM_SETOP_ISECT || op == GPM_SETOP_DIFF;
  for (uint32_t pr = wave; pr < n_pairs; pr += nwaves) {
    const uint64_t ab = a_off[pr], bb = b_off[pr];
    const uint32_t* A = a_all + ab;
    const uint32_t* B = b_all + bb;
    uint32_t na = uniform((uint32_t)(a_off[pr + 1] - ab));
    const uint32_t nb = uniform((uint32_t)(b_off[pr + 1] - bb));
    if (op == GPM_SETOP_FUSE) {
      // Marks of matched B entries live in out_b until B \ A is compacted.
      for (uint32_t i = lane; i < nb; i += kWave) out_b[bb + i] = 0u;
      __builtin_amdgcn_wave_barrier();
      uint32_t c_dif = 0, c_int = 0;
      if (variant == GPM_SETV_MERGE) {
        // Per-lane sizes first (merge order is A order), then the writes.
        uint32_t kd = 0, ki = 0;
        merge_walk(A, na, B, nb, [&](uint32_t, uint32_t m) { (m == kNoMatch ? kd : ki) += 1; });
        const uint32_t ed = wave_incl_scan(kd) - kd, ei = wave_incl_scan(ki) - ki;
        c_dif = uniform(wave_bcast(ed + kd, kWave - 1));
        c_int = uniform(wave_bcast(ei + ki, kWave - 1));
        uint32_t wd = ed, wi = ei;
        merge_walk(A, na, B, nb, [&](uint32_t i, uint32_t m) {
          if (m == kNoMatch) {
            out_a[ab + wd++] = A[i];
          } else {
            out_ab[ab + wi++] = A[i];
            out_b[bb + m] = 1u;
          }
        });
      } else {
        const Probe p = make_probe(variant == GPM_SETV_BITMAP ? GPM_SETV_BINARY : variant, B, nb, lds);
        for (uint32_t base = 0; base < na; base += kWave) {
          const uint32_t i = base + lane;
          const bool valid = i < na;
          const uint32_t x = valid ? A[i] : 0u;
          const uint32_t m = valid ? probe(p, x) : kNoMatch;
          const uint64_t dm = wave_ballot(valid && m == kNoMatch), im = wave_ballot(valid && m != kNoMatch);
          if (valid && m == kNoMatch) out_a[ab + c_dif + lanes_below(dm)] = x;
          if (valid && m != kNoMatch) {
            out_ab[ab + c_int + lanes_below(im)] = x;
            out_b[bb + m] = 1u;
          }
          c_dif += (uint32_t)__popcll(dm);
          c_int += (uint32_t)__popcll(im);
        }
        __builtin_amdgcn_wave_barrier();
      }
      __threadfence_block();
      // B \ A: the unmarked entries of B, compacted in place (writes never
      // pass the reads of the same window).
      uint32_t c_ba = 0;
      for (uint32_t base = 0; base < nb; base += kWave) {
        const uint32_t i = base + lane;
        const bool valid = i < nb;
        const bool keep = valid && out_b[bb + i] == 0u;
        const uint32_t x = keep ? B[i] : 0u;
        const uint64_t km = wave_ballot(keep);
        __builtin_amdgcn_wave_barrier();
        if (keep) out_b[bb + c_ba + lanes_below(km)] = x;
        c_ba += (uint32_t)__popcll(km);
        __threadfence_block();
      }
      if (lane == 0) {
        counts[3 * (uint64_t)pr] = c_dif;
        counts[3 * (uint64_t)pr + 1] = c_int;
        counts[3 * (uint64_t)pr + 2] = c_ba;
      }
      continue;
    }
    // Upper bound: only x < ub of A take part (the walk stops there).
    const uint32_t ub = ubs ? ubs[pr] : kNoBound;
    if (ub != kNoBound) na = uniform(upper_index(A, na, ub - 1u) * (ub > 0u));
    uint32_t cnt = 0;
    if (variant == GPM_SETV_MERGE) {
      uint32_t k = 0;
      merge_walk(A, na, B, nb, [&](uint32_t, uint32_t m) { k += (m != kNoMatch) == keep_in; });
      const uint32_t excl = wave_incl_scan(k) - k;
      cnt = uniform(wave_bcast(excl + k, kWave - 1));
      if (write) {
        uint32_t w = excl;
        merge_walk(A, na, B, nb, [&](uint32_t i, uint32_t m) {
          if ((m != kNoMatch) == keep_in) out_a[ab + w++] = A[i];
        });
      }
    } else {
      const Probe p = make_probe(variant, B, nb, lds);
      for (uint32_t base = 0; base < na; base += kWave) {
        const uint32_t i = base + lane;
        const bool valid = i < na;
        const uint32_t x = valid ? A[i] : 0u;
        const bool keep = valid && ((probe(p, x) != kNoMatch) == keep_in);
        const uint64_t km = wave_ballot(keep);
        if (write && keep) out_a[ab + cnt + lanes_below(km)] = x;
        cnt += (uint32_t)__popcll(km);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) counts[pr] = cnt;
  }
}

// First entry of x that is not above the one before it within its list (off[0 ..
// n_lists]: where the lists begin and end), to *first (preset to the largest value)
// per array; blockIdx.y is the array.  Bound by the one read of the entries.  4096
// pairs (25 MB): the call took 3.7 - 4.0 ms with this on the host, 2.6 with it here and
// short results packed.
struct Lists {
  const uint32_t* x[2];
  const uint64_t* off[2];
  uint64_t count[2];
};

__global__ __launch_bounds__(kBlock) void order_kernel(Lists lists, uint32_t n_lists,
                                                       unsigned long long* __restrict__ first) {
  const uint32_t* __restrict__ x = lists.x[blockIdx.y];
  const uint64_t* __restrict__ off = lists.off[blockIdx.y];
  unsigned long long bad = ~0ull;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x + 1; i < lists.count[blockIdx.y];
       i += (uint64_t)gridDim.x * kBlock) {
    if (x[i - 1] < x[i]) continue;
    uint32_t lo = 0, hi = n_lists + 1;  // a list may begin here
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (off[mid] < i)
        lo = mid + 1;
      else
        hi = mid;
    }
    if (lo > n_lists || off[lo] != i) bad = min(bad, (unsigned long long)i);
  }
  for (int o = kWave / 2; o; o >>= 1) bad = min(bad, (unsigned long long)__shfl_xor(bad, o, kWave));
  if (lane_id() == 0 && bad != ~0ull) atomicMin(first + blockIdx.y, bad);
}

// The first cnt[stride p] entries of every pair's part of an output, end to end.
__global__ __launch_bounds__(kBlock) void pack_kernel(const uint32_t* __restrict__ src,
                                                      const uint64_t* __restrict__ off,
                                                      const unsigned long long* __restrict__ cnt,
                                                      uint32_t stride, uint32_t n_pairs,
                                                      const uint64_t* __restrict__ at,
                                                      uint32_t* __restrict__ dst) {
  const uint32_t nw = gridDim.x * kWavesPerBlock;
  for (uint64_t p = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; p < n_pairs; p += nw)
    for (uint64_t i = lane_id(); i < cnt[p * stride]; i += kWave) dst[at[p] + i] = src[off[p] + i];
}

int run_setops(int op, int variant, uint32_t n_pairs, const uint64_t* a_off, const uint32_t* a,
               const uint64_t* b_off, const uint32_t* b, const uint32_t* ub, uint64_t* counts,
               uint32_t* out_a, uint32_t* out_ab, uint32_t* out_b, void** workspace) {
  GPM_CHECK_ARG(op >= GPM_SETOP_ISECT_COUNT && op <= GPM_SETOP_FUSE, "unknown set op %d", op);
  GPM_CHECK_ARG(variant >= GPM_SETV_BINARY && variant <= GPM_SETV_BITMAP, "unknown variant %d",
                variant);
  GPM_CHECK_ARG(a_off && b_off && counts, "null pointer");
  if (n_pairs == 0) return GPM_OK;
  const uint64_t na = a_off[n_pairs], nb = b_off[n_pairs];
  GPM_CHECK_ARG((a || na == 0) && (b || nb == 0), "null list data");
  for (uint32_t i = 0; i < n_pairs; ++i) {
    GPM_CHECK_ARG(a_off[i] <= a_off[i + 1] && b_off[i] <= b_off[i + 1], "offsets decrease at %u", i);
    GPM_CHECK_ARG(a_off[i + 1] - a_off[i] < (1ull << 32) && b_off[i + 1] - b_off[i] < (1ull << 32),
                  "list %u longer than 2^32 - 1", i);
  }
  const bool write = op == GPM_SETOP_ISECT || op == GPM_SETOP_DIFF || op == GPM_SETOP_FUSE;
  GPM_CHECK_ARG(!write || out_a || na == 0, "null output");
  GPM_CHECK_ARG(op != GPM_SETOP_FUSE || ((out_ab || na == 0) && (out_b || nb == 0)),
                "FUSE needs out_ab and out_b");
  const bool fuse = op == GPM_SETOP_FUSE;
  const bool bounded = ub && !fuse;
  const size_t ncnt = (size_t)n_pairs * (fuse ? 3 : 1);
  // One workspace; 64-bit arrays first.
  size_t bytes = 0;
  auto place = [&](size_t b) {
    const size_t at = bytes;
    bytes += (b + 255) & ~(size_t)255;
    return at;
  };
  const size_t off_bytes = ((size_t)n_pairs + 1) * 8;
  const size_t first_at = place(16), cnt_at = place(ncnt * 8), aoff_at = place(off_bytes),
               boff_at = place(off_bytes), at_at = place(write ? off_bytes : 0),
               a_at = place(na * 4), b_at = place(nb * 4), ub_at = place(bounded ? n_pairs * 4ull : 0),
               oa_at = place(write ? na * 4 : 0), oab_at = place(fuse ? na * 4 : 0),
               ob_at = place(fuse ? nb * 4 : 0);
  if (hipMalloc(workspace, bytes) != hipSuccess) {
    *workspace = nullptr;
    return fail(GPM_ENOMEM, "device workspace of %zu bytes", bytes);
  }
  char* w = static_cast<char*>(*workspace);
  auto* d_first = reinterpret_cast<unsigned long long*>(w + first_at);
  auto* d_cnt = reinterpret_cast<unsigned long long*>(w + cnt_at);
  auto* d_aoff = reinterpret_cast<uint64_t*>(w + aoff_at);
  auto* d_boff = reinterpret_cast<uint64_t*>(w + boff_at);
  auto* d_at = reinterpret_cast<uint64_t*>(w + at_at);
  auto* d_a = reinterpret_cast<uint32_t*>(w + a_at);
  auto* d_b = reinterpret_cast<uint32_t*>(w + b_at);
  uint32_t* d_ub = bounded ? reinterpret_cast<uint32_t*>(w + ub_at) : nullptr;
  uint32_t* d_oa = write && na ? reinterpret_cast<uint32_t*>(w + oa_at) : nullptr;
  uint32_t* d_oab = fuse && na ? reinterpret_cast<uint32_t*>(w + oab_at) : nullptr;
  uint32_t* d_ob = fuse && nb ? reinterpret_cast<uint32_t*>(w + ob_at) : nullptr;
  const unsigned long long none[2] = {~0ull, ~0ull};
  GPM_HIP(hipMemcpy(d_first, none, sizeof(none), hipMemcpyHostToDevice));
  GPM_HIP(hipMemcpy(d_aoff, a_off, off_bytes, hipMemcpyHostToDevice));
  GPM_HIP(hipMemcpy(d_boff, b_off, off_bytes, hipMemcpyHostToDevice));
  if (na) GPM_HIP(hipMemcpy(d_a, a, na * 4, hipMemcpyHostToDevice));
  if (nb) GPM_HIP(hipMemcpy(d_b, b, nb * 4, hipMemcpyHostToDevice));
  if (d_ub) GPM_HIP(hipMemcpy(d_ub, ub, n_pairs * 4ull, hipMemcpyHostToDevice));
  int dev = 0, cus = 256;
  GPM_HIP(hipGetDevice(&dev));
  GPM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const unsigned entry_blocks = (unsigned)std::max<uint64_t>(
      1, std::min<uint64_t>((std::max(na, nb) + kBlock - 1) / kBlock, (uint64_t)cus * 8));
  hipLaunchKernelGGL(order_kernel, dim3(entry_blocks, 2), dim3(kBlock), 0, 0,
                     Lists{{d_a, d_b}, {d_aoff, d_boff}, {na, nb}}, n_pairs, d_first);
  GPM_HIP(hipGetLastError());
  // The searches below rely on the order, so it is known before they start.
  unsigned long long first[2];
  GPM_HIP(hipMemcpy(first, d_first, sizeof(first), hipMemcpyDeviceToHost));
  GPM_CHECK_ARG(first[0] == ~0ull, "list A is not strictly increasing at entry %llu", first[0]);
  GPM_CHECK_ARG(first[1] == ~0ull, "list B is not strictly increasing at entry %llu", first[1]);
  const unsigned blocks = (unsigned)std::max<uint64_t>(
      1, std::min<uint64_t>(((uint64_t)n_pairs + kWavesPerBlock - 1) / kWavesPerBlock,
                            (uint64_t)cus * 8));
  hipLaunchKernelGGL(setops_kernel, dim3(blocks), dim3(kBlock), 0, 0, op, variant, n_pairs, d_aoff,
                     d_a, d_boff, d_b, d_ub, d_cnt, d_oa, d_oab, d_ob);
  GPM_HIP(hipGetLastError());
  static_assert(sizeof(unsigned long long) == sizeof(uint64_t), "counts are copied as they are");
  GPM_HIP(hipMemcpy(counts, d_cnt, ncnt * 8, hipMemcpyDeviceToHost));
  // An output's lists lie where the iterated list's do, so short results are far
  // apart: below a quarter of the room they are packed on the device (over A, which is
  // done with) and put in place on the host, instead of 11 MB copied for a few KB.
  std::vector<uint64_t> at;
  std::vector<uint32_t> packed;
  auto take = [&](const uint32_t* d, const uint64_t* d_off, const uint64_t* off, uint64_t room,
                  uint32_t which, uint32_t* out) -> int {
    if (!d) return GPM_OK;
    const uint32_t stride = fuse ? 3 : 1;
    at.assign((size_t)n_pairs + 1, 0);
    for (uint32_t p = 0; p < n_pairs; ++p) at[p + 1] = at[p] + counts[(size_t)p * stride + which];
    const uint64_t total = at[n_pairs];
    if (total > room / 4 || total > na) {
      GPM_HIP(hipMemcpy(out, d, room * 4, hipMemcpyDeviceToHost));
      return GPM_OK;
    }
    if (!total) return GPM_OK;
    GPM_HIP(hipMemcpy(d_at, at.data(), off_bytes, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(pack_kernel, dim3(blocks), dim3(kBlock), 0, 0, d, d_off, d_cnt + which, stride,
                       n_pairs, d_at, d_a);
    GPM_HIP(hipGetLastError());
    packed.resize(total);
    GPM_HIP(hipMemcpy(packed.data(), d_a, total * 4, hipMemcpyDeviceToHost));
    for (uint32_t p = 0; p < n_pairs; ++p)
      std::copy(packed.begin() + at[p], packed.begin() + at[p + 1], out + off[p]);
    return GPM_OK;
  };
  int st;
  if ((st = take(d_oa, d_aoff, a_off, na, 0, out_a)) != GPM_OK) return st;
  if ((st = take(d_oab, d_aoff, a_off, na, 1, out_ab)) != GPM_OK) return st;
  return take(d_ob, d_boff, b_off, nb, 2, out_b);
}

}  // namespace

extern "C" int gpm_setops(int op, int variant, uint32_t n_pairs, const uint64_t* a_off,
                          const uint32_t* a, const uint64_t* b_off, const uint32_t* b,
                          const uint32_t* ub, uint64_t* counts, uint32_t* out_a,
                          uint32_t* out_ab, uint32_t* out_b) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    struct Workspace {
      void* p = nullptr;
      ~Workspace() { (void)hipFree(p); }
    } workspace;
    return run_setops(op, variant, n_pairs, a_off, a, b_off, b, ub, counts, out_a, out_ab, out_b,
                      &workspace.p);
  });
}
