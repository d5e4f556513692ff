// Graph preparation on the device: CSR build from an edge list (symmetrise,
// drop self loops, sort, dedup) and the degree relabel, replacing the host
// passes of Graph::Init (src/graph/graph.h:254-340, with the symmetrise /
// dedup the configurations' inputs need) and Graph::SortCSRGraph
// (graph.h:206-252).  Orientation already runs on the device
// (gpm_graph_orient).
//
// CSR build: every kept edge becomes one or two records (u, v); sorted mode
// (GPM_CSR_SORT or GPM_CSR_DEDUP) radix-sorts 64-bit keys u << 32 | v, so
// lists come out sorted, and DEDUP keeps the first of equal keys; input-order
// mode radix-sorts the records by u alone (LSD radix sort is stable), so
// every list keeps the order of the edge list, the reverse record of an edge
// right after the forward one -- the order Graph::Init and
// gpm_csr_from_edges produce.  Dropped self loops get the source key n and
// sort past every real record.  Offsets come from the sorted sources in one
// pass (entry i starts the lists of vertices src[i-1]+1 .. src[i]).
#include <algorithm>
#include <numeric>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_select.hpp>

#include "graph_dev.hpp"

using namespace gpm;

namespace {

constexpr int kBlock = 256;

unsigned grid_for_items(uint64_t items, int cus) {
  return (unsigned)std::max<uint64_t>(
      1, std::min<uint64_t>((items + kBlock - 1) / kBlock, (uint64_t)cus * 32));
}

int bits_for(uint64_t max_value) {
  int b = 1;
  while (b < 64 && (max_value >> b)) ++b;
  return b;
}

__global__ void zero_words_kernel(uint32_t* a, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) a[i] = 0u;
}

// What a pass over the edges found: checks[0] endpoints outside the graph,
// checks[2..3] self loops (64 bits; one addition per block, since additions to one
// address take about 10 ns each).
__device__ __forceinline__ void add_checks(bool bad, uint32_t loops, uint32_t* checks) {
  __shared__ uint32_t s_loops;
  if (threadIdx.x == 0) s_loops = 0u;
  __syncthreads();
  if (wave_ballot(bad) && lane_id() == 0) checks[0] = 1u;
  loops = wave_sum_u32(loops);
  if (lane_id() == 0 && loops) atomicAdd(&s_loops, loops);
  __syncthreads();
  if (threadIdx.x == 0 && s_loops)
    atomicAdd(reinterpret_cast<unsigned long long*>(checks + 2), (unsigned long long)s_loops);
}

// Records of edge i: (u, v) and, when symmetrising, (v, u) right after it.
__global__ void emit_keys_kernel(const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst,
                                 uint64_t n_edges, uint32_t n, bool sym, bool drop_self,
                                 unsigned long long* __restrict__ keys,
                                 uint32_t* __restrict__ checks) {
  const uint32_t per = sym ? 2u : 1u;
  bool bad = false;
  uint32_t loops = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_edges;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t u = src[i], v = dst[i];
    const bool drop = drop_self && u == v;
    const unsigned long long sentinel = (unsigned long long)n << 32;
    keys[per * i] = drop ? sentinel : ((unsigned long long)u << 32 | v);
    if (sym) keys[per * i + 1] = drop ? sentinel : ((unsigned long long)v << 32 | u);
    bad |= u >= n || v >= n;
    loops += u == v;
  }
  add_checks(bad, loops, checks);
}

// Input-order mode: source keys (n for dropped records) and target values.
__global__ void emit_pairs_kernel(const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst,
                                  uint64_t n_edges, uint32_t n, bool sym, bool drop_self,
                                  uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                  uint32_t* __restrict__ checks) {
  const uint32_t per = sym ? 2u : 1u;
  bool bad = false;
  uint32_t loops = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_edges;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t u = src[i], v = dst[i];
    const bool drop = drop_self && u == v;
    keys[per * i] = drop ? n : u;
    vals[per * i] = v;
    if (sym) {
      keys[per * i + 1] = drop ? n : v;
      vals[per * i + 1] = u;
    }
    bad |= u >= n || v >= n;
    loops += u == v;
  }
  add_checks(bad, loops, checks);
}

__global__ void split_keys_kernel(const unsigned long long* __restrict__ keys, uint64_t m,
                                  uint32_t* __restrict__ hi, uint32_t* __restrict__ lo) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const unsigned long long k = keys[i];
    hi[i] = (uint32_t)(k >> 32);
    lo[i] = (uint32_t)k;
  }
}

// off[v] = first record with source >= v, for v in [0, n]; src holds the
// sorted sources of the m kept records.
__global__ void offsets_kernel(const uint32_t* __restrict__ src, uint64_t m, uint32_t n,
                               uint32_t* __restrict__ off) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i <= m;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t first = i == 0 ? 0 : (uint64_t)src[i - 1] + 1;  // vertices starting here
    const uint64_t last = i == m ? n : src[i];
    for (uint64_t v = first; v <= last; ++v) off[v] = (uint32_t)i;
  }
}

// Degree relabel: sort keys (max_deg - deg(v)) with values v, then
// new_id[order[r]] = r.
__global__ void degree_keys_kernel(const uint32_t* __restrict__ off, uint32_t n, uint32_t max_deg,
                                   uint32_t* __restrict__ keys, uint32_t* __restrict__ ids) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    keys[v] = max_deg - (off[v + 1] - off[v]);
    ids[v] = v;
  }
}

__global__ void scatter_rank_kernel(const uint32_t* __restrict__ order, uint32_t n,
                                    uint32_t* __restrict__ new_id) {
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x)
    new_id[order[r]] = r;
}

// Degree order of a range: sort keys max_deg - deg(v) and values rank[v] (or v).
__global__ void order_keys_kernel(const uint32_t* __restrict__ off, uint32_t first, uint32_t count,
                                  uint32_t max_deg, const uint32_t* __restrict__ rank,
                                  uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
    const uint32_t v = first + i;
    keys[i] = max_deg - (off[v + 1] - off[v]);
    vals[i] = rank ? rank[v] : v;
  }
}

// Keys new_id[u] << 32 | new_id[x] for every entry (u, x); one wave per u.
__global__ void relabel_keys_kernel(const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                    const uint32_t* __restrict__ new_id, uint32_t n,
                                    unsigned long long* __restrict__ keys) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = gridDim.x * blockDim.x / kWave;
  for (uint32_t u = wave; u < n; u += nwaves) {
    const unsigned long long hi = (unsigned long long)new_id[u] << 32;
    for (uint32_t i = off[u] + lane_id(); i < off[u + 1]; i += kWave) keys[i] = hi | new_id[adj[i]];
  }
}

// Orientation of a symmetric CSR, by entries: every list has a hub's length or a
// leaf's, so a wave or block per list leaves the hubs for last.  Pass 1 decides each
// entry (u, v) -- kept when (deg, id) of v is above u's (graph.h:128-129) -- and writes one bit per
// entry and a count per 64; after a scan of the counts, pass 2 compacts the
// entries and a pass over the vertices reads the new offsets off the bits.  Pass 1 is
// bound by the gathers of off[v]; the other two stream.  R-MAT scale 17 ef 16 (3.7 M
// entries): the two passes of a wave per list took 336 + 380 us, the three take
// 37 + 9 + 4 us.
constexpr uint32_t kOrientEntries = 2048;  // per block and step of pass 1
constexpr uint32_t kOrientOffsets = 1024;  // offsets kept in LDS, where that covers them

__global__ __launch_bounds__(kBlock) void orient_bits_kernel(
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj, uint32_t n, uint64_t m,
    unsigned long long* __restrict__ bits, uint32_t* __restrict__ count) {
  __shared__ uint32_t s_off[kOrientOffsets + 2];
  for (uint64_t base = (uint64_t)blockIdx.x * kOrientEntries; base < m;
       base += (uint64_t)gridDim.x * kOrientEntries) {
    // Owners of the step's first and last entry: the last vertices whose offset is
    // not past them.
    const uint32_t last_entry = (uint32_t)(min(base + kOrientEntries, m) - 1);
    const uint32_t first = upper_index(off, n + 1, (uint32_t)base) - 1;
    const uint32_t last = upper_index(off, n + 1, last_entry) - 1;
    const uint32_t span = last - first + 1;
    const bool local = span <= kOrientOffsets;
    __syncthreads();  // the last step's readers are done
    if (local)
      for (uint32_t i = threadIdx.x; i <= span; i += kBlock) s_off[i] = off[first + i];
    __syncthreads();
    for (uint32_t i0 = 0; i0 < kOrientEntries; i0 += kBlock) {
      const uint64_t i = base + i0 + threadIdx.x;
      bool keep = false;
      if (i < m) {
        uint32_t u, du;
        if (local) {
          const uint32_t k = upper_index(s_off, span, (uint32_t)i) - 1;
          u = first + k;
          du = s_off[k + 1] - s_off[k];
        } else {
          u = first + upper_index(off + first, span, (uint32_t)i) - 1;
          du = off[u + 1] - off[u];
        }
        const uint32_t v = adj[i], dv = off[v + 1] - off[v];
        keep = dv > du || (dv == du && v > u);
      }
      const uint64_t mask = wave_ballot(keep);
      if (lane_id() == 0 && i < m) {
        bits[i / kWave] = mask;
        count[i / kWave] = (uint32_t)__popcll(mask);
      }
    }
  }
}

// adj[i] of every set bit, packed; before[w]: set bits below word w.
__global__ __launch_bounds__(kBlock) void orient_pack_kernel(
    const uint32_t* __restrict__ adj, uint64_t m, const unsigned long long* __restrict__ bits,
    const uint32_t* __restrict__ before, uint32_t* __restrict__ new_adj) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t mask = bits[i / kWave];
    if ((mask >> (i % kWave)) & 1u) new_adj[before[i / kWave] + lanes_below(mask)] = adj[i];
  }
}

// New offset of every vertex (and of the end): the set bits below its old one.
__global__ __launch_bounds__(kBlock) void orient_offsets_kernel(
    const uint32_t* __restrict__ off, uint32_t n, uint64_t m,
    const unsigned long long* __restrict__ bits, const uint32_t* __restrict__ before,
    uint32_t* __restrict__ new_off) {
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= n;
       v += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t o = off[v], w = o / kWave;
    new_off[v] = before[w] + (o % kWave ? (uint32_t)__popcll(bits[w] << (kWave - o % kWave)) : 0u);
  }
}

// Topological relabel of a DAG (topo_relabel_device).  deg[v] = out-degree
// plus in-degree: the out-degrees first, then the
__global__ void out_degree_kernel(const uint32_t* __restrict__ off, uint32_t n,
                                  uint32_t* __restrict__ deg, uint32_t* __restrict__ ids) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    deg[v] = off[v + 1] - off[v];
    ids[v] = v;
  }
}

// in-degrees off the sorted targets: x's run [b, e) adds e - b.  (An increment per
// entry serialises on the hubs: 1.44 ms on R-MAT scale 19 ef 16; at scale 20, twice
// the entries, this takes 30 us behind three sort passes of about 60.)
__global__ void in_degree_kernel(const uint32_t* __restrict__ targets, uint64_t m,
                                 uint32_t* __restrict__ deg) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t x = targets[i];
    if (i == 0 || targets[i - 1] != x) atomicSub(&deg[x], (uint32_t)i);
    if (i + 1 == m || targets[i + 1] != x) atomicAdd(&deg[x], (uint32_t)i + 1u);
  }
}

// Keys rank(u) << bits | rank(x) of every entry, one wave per u;
// *descent is set when some edge does not go up in rank.
__global__ void topo_keys_kernel(const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                 const uint32_t* __restrict__ rank, uint32_t n, uint32_t bits,
                                 unsigned long long* __restrict__ keys,
                                 unsigned int* __restrict__ descent) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = gridDim.x * blockDim.x / kWave;
  bool down = false;
  for (uint32_t u = wave; u < n; u += nwaves) {
    const uint32_t ru = rank[u];
    for (uint32_t i = off[u] + lane_id(); i < off[u + 1]; i += kWave) {
      const uint32_t rx = rank[adj[i]];
      down |= rx <= ru;
      keys[i] = (unsigned long long)ru << bits | rx;
    }
  }
  if (down) *descent = 1u;
}

// Out-degrees in rank order (entry n = 0, so the scan ends with m).
__global__ void ranked_degree_kernel(const uint32_t* __restrict__ off,
                                     const uint32_t* __restrict__ order, uint32_t n,
                                     uint32_t* __restrict__ out) {
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r <= n; r += gridDim.x * blockDim.x)
    out[r] = r < n ? off[order[r] + 1] - off[order[r]] : 0u;
}

__global__ void key_targets_kernel(const unsigned long long* __restrict__ keys, uint64_t m,
                                   uint32_t bits, uint32_t* __restrict__ out) {
  const uint32_t mask = bits >= 32 ? 0xFFFFFFFFu : (1u << bits) - 1u;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
       i += (uint64_t)gridDim.x * blockDim.x)
    out[i] = (uint32_t)keys[i] & mask;
}

// Device buffers of one preparation call, freed on every exit path unless
// handed to the new graph.
struct Bufs {
  std::vector<void*> owned;
  template <typename T>
  int alloc(T** p, uint64_t count) {
    *p = nullptr;
    if (hipMalloc(p, std::max<uint64_t>(count, 1) * sizeof(T)) != hipSuccess) {
      *p = nullptr;
      return fail(GPM_ENOMEM, "device buffer of %llu bytes",
                  (unsigned long long)(count * sizeof(T)));
    }
    owned.push_back(*p);
    return GPM_OK;
  }
  void release(void* p) { owned.erase(std::remove(owned.begin(), owned.end(), p), owned.end()); }
  ~Bufs() {
    for (void* p : owned) (void)hipFree(p);
  }
};

uint64_t aligned(uint64_t bytes) { return (bytes + 255) & ~255ull; }

// Sorted 64-bit keys (u << 32 | v, the m_kept first valid) -> CSR in new
// buffers *d_off, *d_adj (owned by `b` until released).  d_src: room for m sources,
// apart from the keys.
int keys_to_csr(Bufs& b, const unsigned long long* keys, uint64_t m, uint32_t n, int cus,
                hipStream_t stream, uint32_t* d_src, uint32_t** d_off, uint32_t** d_adj) {
  int st;
  if ((st = b.alloc(d_adj, m)) != GPM_OK || (st = b.alloc(d_off, (uint64_t)n + 1)) != GPM_OK)
    return st;
  if (m)
    hipLaunchKernelGGL(split_keys_kernel, dim3(grid_for_items(m, cus)), dim3(kBlock), 0, stream,
                       keys, m, d_src, *d_adj);
  hipLaunchKernelGGL(offsets_kernel, dim3(grid_for_items(m + 1, cus)), dim3(kBlock), 0, stream,
                     d_src, m, n, *d_off);
  GPM_HIP(hipGetLastError());
  return GPM_OK;
}

int build(uint32_t n, const uint32_t* src, const uint32_t* dst, uint64_t n_edges, uint32_t csr_flags,
          const uint32_t* labels, uint32_t n_labels, uint32_t graph_flags, gpm_graph** out) {
  GPM_CHECK_ARG(out, "null pointer");
  GPM_CHECK_ARG(n_edges == 0 || (src && dst), "null edge arrays");
  GPM_CHECK_ARG(n < 0xFFFFFFFFu, "n must be < 2^32 - 1");
  GPM_CHECK_ARG(!labels || (n_labels >= 1 && n_labels <= 4096), "n_labels must be in [1, 4096]");
  if (labels)
    for (uint32_t v = 0; v < n; ++v)
      if (labels[v] >= n_labels) return fail(GPM_EINVAL, "label of %u >= n_labels", v);
  const bool sym = csr_flags & GPM_CSR_SYMMETRIZE;
  const bool dedup = csr_flags & GPM_CSR_DEDUP;
  const bool drop_self = csr_flags & GPM_CSR_DROP_SELF;
  const bool sorted = (csr_flags & GPM_CSR_SORT) || dedup;
  const uint64_t records = n_edges * (sym ? 2 : 1);
  GPM_CHECK_ARG(records < (1ull << 32), "too many adjacency records (%llu)",
                (unsigned long long)records);
  int dev = 0, cus = 256;
  GPM_HIP(hipGetDevice(&dev));
  GPM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  hipStream_t stream = nullptr;
  GPM_HIP(stream_take(&stream));
  struct StreamGuard {
    hipStream_t* s;
    ~StreamGuard() { stream_give(*s); }
  } guard{&stream};
  Bufs b;
  int st;
  // One workspace: the records as emitted (later the unique keys), the sorted
  // records, whose room first holds the edges, temporary storage, the checks and
  // the number of unique keys.
  const int vbits = bits_for(n);  // source keys go up to n (the drop sentinel)
  const unsigned end_bit = 32u + (unsigned)vbits;
  size_t sort_bytes = 0, unique_bytes = 0;
  unsigned long long *keys = nullptr, *sorted_keys = nullptr, *d_count = nullptr;
  uint32_t *keys32 = nullptr, *vals = nullptr, *skeys = nullptr;
  uint32_t *d_off = nullptr, *d_adj = nullptr;
  if (records && sorted) {
    GPM_HIP(rocprim::radix_sort_keys(nullptr, sort_bytes, keys, sorted_keys, records, 0u, end_bit,
                                     stream));
    if (dedup)
      GPM_HIP(rocprim::unique(nullptr, unique_bytes, sorted_keys, keys, d_count, records,
                              rocprim::equal_to<unsigned long long>(), stream));
  } else if (records) {
    GPM_HIP(rocprim::radix_sort_pairs(nullptr, sort_bytes, keys32, skeys, vals, d_adj, records, 0u,
                                      (unsigned)vbits, stream));
  }
  const uint64_t edge_at = aligned(std::max(sort_bytes, unique_bytes));
  const uint64_t key_at = edge_at + aligned(std::max(n_edges, records) * 8);
  const uint64_t small_at = key_at + aligned(records * 8);
  char* temp = nullptr;
  if ((st = b.alloc(&temp, small_at + 24)) != GPM_OK) return st;
  uint32_t* d_src = reinterpret_cast<uint32_t*>(temp + edge_at);
  uint32_t* d_dst = d_src + n_edges;
  uint32_t* checks = reinterpret_cast<uint32_t*>(temp + small_at);
  d_count = reinterpret_cast<unsigned long long*>(checks + 4);
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, stream, checks, 6u);
  if (n_edges) {
    GPM_HIP(hipMemcpyAsync(d_src, src, n_edges * 4, hipMemcpyHostToDevice, stream));
    GPM_HIP(hipMemcpyAsync(d_dst, dst, n_edges * 4, hipMemcpyHostToDevice, stream));
  }
  const unsigned emit_grid = std::min(grid_for_items(n_edges, cus), (unsigned)cus * 8);
  if (sorted) {
    keys = reinterpret_cast<unsigned long long*>(temp + key_at);
    sorted_keys = reinterpret_cast<unsigned long long*>(d_src);
    if (records) {
      hipLaunchKernelGGL(emit_keys_kernel, dim3(emit_grid), dim3(kBlock), 0,
                         stream, d_src, d_dst, n_edges, n, sym, drop_self, keys, checks);
      GPM_HIP(hipGetLastError());
      GPM_HIP(rocprim::radix_sort_keys(temp, sort_bytes, keys, sorted_keys, records, 0u, end_bit,
                                       stream));
      if (dedup)  // unique keys into `keys`, which the sort is done with
        GPM_HIP(rocprim::unique(temp, unique_bytes, sorted_keys, keys, d_count, records,
                                rocprim::equal_to<unsigned long long>(), stream));
    }
  } else {
    keys32 = reinterpret_cast<uint32_t*>(temp + key_at);
    vals = keys32 + records;
    skeys = d_src;
    if ((st = b.alloc(&d_adj, records)) != GPM_OK) return st;
    if (records) {
      hipLaunchKernelGGL(emit_pairs_kernel, dim3(emit_grid), dim3(kBlock), 0,
                         stream, d_src, d_dst, n_edges, n, sym, drop_self, keys32, vals, checks);
      GPM_HIP(hipGetLastError());
      GPM_HIP(rocprim::radix_sort_pairs(temp, sort_bytes, keys32, skeys, vals, d_adj, records, 0u,
                                        (unsigned)vbits, stream));
    }
  }
  // The edges are checked where they are read; nothing below indexes by a vertex
  // before this.
  uint32_t found[6];
  GPM_HIP(hipMemcpyAsync(found, checks, sizeof(found), hipMemcpyDeviceToHost, stream));
  GPM_HIP(hipStreamSynchronize(stream));
  if (found[0]) return fail(GPM_EINVAL, "edge endpoint >= n (%u)", n);
  // Dropped self loops became sentinel records that sort past the real ones; dedup
  // keeps one of them.
  const uint64_t self_loops = (uint64_t)found[3] << 32 | found[2];
  const uint64_t dropped = drop_self ? self_loops * (sym ? 2 : 1) : 0;
  const uint64_t unique = (uint64_t)found[5] << 32 | found[4];
  const uint64_t m = dedup ? unique - (dropped ? 1 : 0) : records - dropped;
  if (sorted) {
    // The keys are in `keys` after dedup, else where the sort put them; the other
    // buffer holds the sources.
    if ((st = keys_to_csr(b, dedup ? keys : sorted_keys, m, n, cus, stream,
                          reinterpret_cast<uint32_t*>(dedup ? sorted_keys : keys), &d_off, &d_adj)) !=
        GPM_OK)
      return st;
  } else {
    if ((st = b.alloc(&d_off, (uint64_t)n + 1)) != GPM_OK) return st;
    hipLaunchKernelGGL(offsets_kernel, dim3(grid_for_items(m + 1, cus)), dim3(kBlock), 0, stream,
                       skeys, m, n, d_off);
    GPM_HIP(hipGetLastError());
  }
  std::vector<uint32_t> h_off((size_t)n + 1);
  GPM_HIP(hipMemcpyAsync(h_off.data(), d_off, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost, stream));
  std::vector<uint32_t> h_adj;
  if (labels) {
    h_adj.resize(std::max<uint64_t>(m, 1));
    if (m) GPM_HIP(hipMemcpyAsync(h_adj.data(), d_adj, m * 4, hipMemcpyDeviceToHost, stream));
  }
  GPM_HIP(hipStreamSynchronize(stream));
  b.release(d_off);
  b.release(d_adj);
  hipStream_t s = stream;
  stream = nullptr;  // the handle owns it now
  st = adopt_device_csr(n, m, d_off, d_adj, std::move(h_off), h_adj.data(), labels, n_labels,
                        graph_flags, s, out);
  if (st == GPM_OK && sym && dedup && drop_self) (*out)->mirrored = 1;
  return st;
}

int relabel(gpm_graph* g, gpm_graph** out, uint32_t** perm) {
  GPM_CHECK_ARG(g && out && perm, "null pointer");
  const uint32_t n = g->n;
  const uint64_t m = g->m;
  int cus = device_cus(g);
  hipStream_t stream = nullptr;
  GPM_HIP(stream_take(&stream));
  struct StreamGuard {
    hipStream_t* s;
    ~StreamGuard() { stream_give(*s); }
  } guard{&stream};
  // The source graph's pending work must be done before this stream reads it.
  GPM_HIP(hipStreamSynchronize(g->stream));
  Bufs b;
  int st;
  uint32_t *dkeys = nullptr, *ids = nullptr, *skeys = nullptr, *order = nullptr, *new_id = nullptr;
  if ((st = b.alloc(&dkeys, n)) != GPM_OK || (st = b.alloc(&ids, n)) != GPM_OK ||
      (st = b.alloc(&skeys, n)) != GPM_OK || (st = b.alloc(&order, n)) != GPM_OK ||
      (st = b.alloc(&new_id, n)) != GPM_OK)
    return st;
  void* temp = nullptr;
  size_t temp_bytes = 0;
  if (n) {
    hipLaunchKernelGGL(degree_keys_kernel, dim3(grid_for_items(n, cus)), dim3(kBlock), 0, stream,
                       g->off, n, g->max_deg, dkeys, ids);
    GPM_HIP(hipGetLastError());
    const unsigned end_bit = (unsigned)bits_for(g->max_deg);
    GPM_HIP(rocprim::radix_sort_pairs(nullptr, temp_bytes, dkeys, skeys, ids, order, n, 0u,
                                      end_bit, stream));
    if ((st = b.alloc(reinterpret_cast<char**>(&temp), temp_bytes)) != GPM_OK) return st;
    GPM_HIP(rocprim::radix_sort_pairs(temp, temp_bytes, dkeys, skeys, ids, order, n, 0u, end_bit,
                                      stream));
    hipLaunchKernelGGL(scatter_rank_kernel, dim3(grid_for_items(n, cus)), dim3(kBlock), 0, stream,
                       order, n, new_id);
    GPM_HIP(hipGetLastError());
  }
  unsigned long long *keys = nullptr, *sorted_keys = nullptr;
  if ((st = b.alloc(&keys, m)) != GPM_OK || (st = b.alloc(&sorted_keys, m)) != GPM_OK) return st;
  if (m) {
    const unsigned blocks = grid_for_items((uint64_t)n * kWave, cus);
    hipLaunchKernelGGL(relabel_keys_kernel, dim3(blocks), dim3(kBlock), 0, stream, g->off, g->adj,
                       new_id, n, keys);
    GPM_HIP(hipGetLastError());
    const unsigned end_bit = 32u + (unsigned)bits_for(n);
    size_t tb = 0;
    GPM_HIP(rocprim::radix_sort_keys(nullptr, tb, keys, sorted_keys, m, 0u, end_bit, stream));
    void* t2 = nullptr;
    if ((st = b.alloc(reinterpret_cast<char**>(&t2), tb)) != GPM_OK) return st;
    GPM_HIP(rocprim::radix_sort_keys(t2, tb, keys, sorted_keys, m, 0u, end_bit, stream));
  }
  uint32_t *d_off = nullptr, *d_adj = nullptr;
  if ((st = keys_to_csr(b, sorted_keys, m, n, cus, stream, reinterpret_cast<uint32_t*>(keys), &d_off,
                        &d_adj)) != GPM_OK)
    return st;
  std::vector<uint32_t> h_off((size_t)n + 1), h_new(std::max(n, 1u));
  GPM_HIP(hipMemcpyAsync(h_off.data(), d_off, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost, stream));
  if (n) GPM_HIP(hipMemcpyAsync(h_new.data(), new_id, (size_t)n * 4, hipMemcpyDeviceToHost, stream));
  std::vector<uint32_t> h_adj;
  std::vector<uint32_t> nlab;
  if (g->labels) {
    h_adj.resize(std::max<uint64_t>(m, 1));
    if (m) GPM_HIP(hipMemcpyAsync(h_adj.data(), d_adj, m * 4, hipMemcpyDeviceToHost, stream));
    nlab.resize(n);
    for (uint32_t v = 0; v < n; ++v) nlab[h_new[v]] = g->h_labels[v];
  }
  GPM_HIP(hipStreamSynchronize(stream));
  uint32_t* p = xmalloc<uint32_t>(std::max(n, 1u));
  if (!p) return fail(GPM_ENOMEM, "host allocation failed");
  std::copy(h_new.begin(), h_new.begin() + n, p);
  b.release(d_off);
  b.release(d_adj);
  hipStream_t s = stream;
  stream = nullptr;
  st = adopt_device_csr(n, m, d_off, d_adj, std::move(h_off), h_adj.data(),
                        g->labels ? nlab.data() : nullptr, g->n_labels, g->flags, s, out);
  if (st != GPM_OK) {
    std::free(p);
    return st;
  }
  (*out)->mirrored = g->mirrored;
  *perm = p;
  return GPM_OK;
}

}  // namespace

namespace gpm {

int orient_device(gpm_graph* sym, uint32_t** d_off, uint32_t** d_adj, std::vector<uint32_t>* h_off) {
  const uint32_t n = sym->n;
  const uint64_t m = sym->m;
  const uint64_t words = (m + kWave - 1) / kWave;
  const int cus = device_cus(sym);
  struct Drain {  // the buffers below are freed only once the stream is done with them
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  };
  Bufs b;
  Drain drain{sym->stream};
  int st;
  // One workspace: bits, counts and their scan (one word more each, so that the
  // scan ends with the total), temporary storage.
  size_t scan = 0;
  GPM_HIP(rocprim::exclusive_scan(nullptr, scan, (uint32_t*)nullptr, (uint32_t*)nullptr, 0u,
                                  (size_t)words + 1, rocprim::plus<uint32_t>(), sym->stream));
  const uint64_t flags_at = aligned(scan), count_at = flags_at + aligned(words * 8);
  const uint64_t before_at = count_at + aligned((words + 1) * 4);
  char* temp = nullptr;
  if ((st = b.alloc(&temp, before_at + (words + 1) * 4)) != GPM_OK ||
      (st = b.alloc(d_off, (uint64_t)n + 1)) != GPM_OK)
    return st;
  auto* bits = reinterpret_cast<unsigned long long*>(temp + flags_at);
  auto* count = reinterpret_cast<uint32_t*>(temp + count_at);
  auto* before = reinterpret_cast<uint32_t*>(temp + before_at);
  const dim3 block(kBlock);
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(1), 0, sym->stream, count + words, 1u);
  if (m)
    hipLaunchKernelGGL(orient_bits_kernel,
                       dim3((unsigned)std::min<uint64_t>((m + kOrientEntries - 1) / kOrientEntries,
                                                         (uint64_t)cus * 32)),
                       block, 0, sym->stream, sym->off, sym->adj, n, m, bits, count);
  GPM_HIP(hipGetLastError());
  GPM_HIP(rocprim::exclusive_scan(temp, scan, count, before, 0u, (size_t)words + 1,
                                  rocprim::plus<uint32_t>(), sym->stream));
  hipLaunchKernelGGL(orient_offsets_kernel, dim3(grid_for_items((uint64_t)n + 1, cus)), block, 0,
                     sym->stream, sym->off, n, m, bits, before, *d_off);
  GPM_HIP(hipGetLastError());
  h_off->resize((size_t)n + 1);
  GPM_HIP(hipMemcpyAsync(h_off->data(), *d_off, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost,
                         sym->stream));
  GPM_HIP(hipStreamSynchronize(sym->stream));
  if ((st = b.alloc(d_adj, h_off->back())) != GPM_OK) return st;
  if (m)
    hipLaunchKernelGGL(orient_pack_kernel, dim3(grid_for_items(m, cus)), block, 0, sym->stream,
                       sym->adj, m, bits, before, *d_adj);
  GPM_HIP(hipGetLastError());
  GPM_HIP(hipStreamSynchronize(sym->stream));
  b.release(*d_off);
  b.release(*d_adj);
  return GPM_OK;
}

int degree_order_device(gpm_graph* g, uint32_t first, uint32_t count, const uint32_t* rank,
                        uint32_t* out) {
  if (!count) return GPM_OK;
  struct Drain {  // the buffers below are freed only once the stream is done with them
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  };
  Bufs b;
  Drain drain{g->stream};
  const unsigned bits = (unsigned)bits_for(g->max_deg);
  size_t sort = 0;
  uint32_t* none = nullptr;
  GPM_HIP(rocprim::radix_sort_pairs(nullptr, sort, none, none, none, none, count, 0u, bits,
                                    g->stream));
  const uint64_t part = aligned((uint64_t)count * 4), rank_at = aligned(sort) + 3 * part;
  char* temp = nullptr;
  int st;
  if ((st = b.alloc(&temp, rank_at + (rank ? (uint64_t)g->n * 4 : 0))) != GPM_OK) return st;
  uint32_t* keys = reinterpret_cast<uint32_t*>(temp + aligned(sort));
  uint32_t* sorted = reinterpret_cast<uint32_t*>(temp + aligned(sort) + part);
  uint32_t* vals = reinterpret_cast<uint32_t*>(temp + aligned(sort) + 2 * part);
  uint32_t* d_rank = rank ? reinterpret_cast<uint32_t*>(temp + rank_at) : nullptr;
  if (rank && (st = h2d(g, d_rank, rank, (size_t)g->n * 4)) != GPM_OK) return st;
  hipLaunchKernelGGL(order_keys_kernel, dim3(grid_for_items(count, device_cus(g))), dim3(kBlock), 0,
                     g->stream, g->off, first, count, g->max_deg, d_rank, keys, vals);
  GPM_HIP(hipGetLastError());
  GPM_HIP(rocprim::radix_sort_pairs(temp, sort, keys, sorted, vals, out, count, 0u, bits, g->stream));
  return GPM_OK;
}

int topo_relabel_device(gpm_graph* g, uint32_t** toff, uint32_t** tadj, std::vector<uint32_t>* rank,
                        bool* ordered) {
  const uint32_t n = g->n;
  const uint64_t m = g->m;
  const int cus = device_cus(g);
  *ordered = false;
  if (!n || !m) return GPM_OK;
  struct Drain {  // the buffers below are freed only once the stream is done with them
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  };
  Bufs b;
  Drain drain{g->stream};
  int st;
  const unsigned bits = (unsigned)bits_for(std::max(n, 1u) - 1u);
  uint32_t *deg = nullptr, *ids = nullptr, *sdeg = nullptr, *order = nullptr, *new_id = nullptr;
  unsigned int* descent = nullptr;
  unsigned long long *keys = nullptr, *sorted = nullptr;
  if ((st = b.alloc(&deg, n)) != GPM_OK || (st = b.alloc(&ids, n)) != GPM_OK ||
      (st = b.alloc(&sdeg, (uint64_t)n + 1)) != GPM_OK || (st = b.alloc(&order, n)) != GPM_OK ||
      (st = b.alloc(&new_id, n)) != GPM_OK || (st = b.alloc(&descent, 1)) != GPM_OK ||
      (st = b.alloc(&keys, m)) != GPM_OK || (st = b.alloc(&sorted, m)) != GPM_OK ||
      (st = b.alloc(toff, (uint64_t)n + 1)) != GPM_OK || (st = b.alloc(tadj, m)) != GPM_OK)
    return st;
  const dim3 block(kBlock);
  const dim3 per_vertex(grid_for_items((uint64_t)n + 1, cus));
  size_t sort_ids = 0, sort_keys = 0, sort_targets = 0, scan = 0;
  uint32_t* targets = reinterpret_cast<uint32_t*>(sorted);  // until the keys are sorted
  GPM_HIP(rocprim::radix_sort_pairs(nullptr, sort_ids, deg, sdeg, ids, order, n, 0u, 32u,
                                    g->stream));
  GPM_HIP(rocprim::radix_sort_keys(nullptr, sort_keys, keys, sorted, m, 0u, 2 * bits, g->stream));
  GPM_HIP(rocprim::radix_sort_keys(nullptr, sort_targets, g->adj, targets, m, 0u, bits, g->stream));
  GPM_HIP(rocprim::exclusive_scan(nullptr, scan, sdeg, *toff, 0u, (size_t)n + 1,
                                  rocprim::plus<uint32_t>(), g->stream));
  char* temp = nullptr;
  if ((st = b.alloc(&temp, std::max(std::max(sort_ids, sort_keys), std::max(sort_targets, scan)))) != GPM_OK) return st;
  hipLaunchKernelGGL(out_degree_kernel, per_vertex, block, 0, g->stream, g->off, n, deg, ids);
  GPM_HIP(rocprim::radix_sort_keys(temp, sort_targets, g->adj, targets, m, 0u, bits, g->stream));
  hipLaunchKernelGGL(in_degree_kernel, dim3(grid_for_items(m, cus)), block, 0, g->stream, targets,
                     m, deg);
  GPM_HIP(hipGetLastError());
  GPM_HIP(rocprim::radix_sort_pairs(temp, sort_ids, deg, sdeg, ids, order, n, 0u, 32u, g->stream));
  hipLaunchKernelGGL(scatter_rank_kernel, per_vertex, block, 0, g->stream, order, n, new_id);
  hipLaunchKernelGGL(ranked_degree_kernel, per_vertex, block, 0, g->stream, g->off, order, n, sdeg);
  GPM_HIP(hipGetLastError());
  GPM_HIP(rocprim::exclusive_scan(temp, scan, sdeg, *toff, 0u, (size_t)n + 1,
                                  rocprim::plus<uint32_t>(), g->stream));
  const unsigned int zero = 0;
  if ((st = h2d(g, descent, &zero, sizeof(zero))) != GPM_OK) return st;
  hipLaunchKernelGGL(topo_keys_kernel, dim3(grid_for_items((uint64_t)n * kWave, cus)), block, 0,
                     g->stream, g->off, g->adj, new_id, n, bits, keys, descent);
  GPM_HIP(hipGetLastError());
  GPM_HIP(rocprim::radix_sort_keys(temp, sort_keys, keys, sorted, m, 0u, 2 * bits, g->stream));
  hipLaunchKernelGGL(key_targets_kernel, dim3(grid_for_items(m, cus)), block, 0, g->stream, sorted,
                     m, bits, *tadj);
  GPM_HIP(hipGetLastError());
  unsigned int down = 0;
  rank->resize(n);
  GPM_HIP(hipMemcpyAsync(&down, descent, sizeof(down), hipMemcpyDeviceToHost, g->stream));
  GPM_HIP(hipMemcpyAsync(rank->data(), new_id, (size_t)n * 4, hipMemcpyDeviceToHost, g->stream));
  GPM_HIP(hipStreamSynchronize(g->stream));
  if (down) return GPM_OK;
  *ordered = true;
  b.release(*toff);
  b.release(*tadj);
  return GPM_OK;
}

}  // namespace gpm

extern "C" {

int gpm_graph_build(uint32_t n, const uint32_t* src, const uint32_t* dst, uint64_t n_edges,
                    uint32_t csr_flags, const uint32_t* labels, uint32_t n_labels,
                    uint32_t graph_flags, gpm_graph** out) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    return build(n, src, dst, n_edges, csr_flags, labels, n_labels, graph_flags, out);
  });
}

int gpm_graph_relabel_by_degree(gpm_graph* g, gpm_graph** out, uint32_t** perm) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    return relabel(g, out, perm);
  });
}

int gpm_graph_copy_csr(const gpm_graph* g, uint32_t* offsets, uint32_t* adj) {
  return ::gpm::guarded([&]() -> int {
    clear_error();
    GPM_CHECK_ARG(g && offsets && (adj || g->m == 0), "null pointer");
    GPM_HIP(hipMemcpyAsync(offsets, g->off, ((size_t)g->n + 1) * 4, hipMemcpyDeviceToHost,
                           g->stream));
    if (g->m) GPM_HIP(hipMemcpyAsync(adj, g->adj, g->m * 4, hipMemcpyDeviceToHost, g->stream));
    GPM_HIP(hipStreamSynchronize(g->stream));
    return GPM_OK;
  });
}

}  // extern "C"
