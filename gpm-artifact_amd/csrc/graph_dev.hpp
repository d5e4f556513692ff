// Device graph handle of libgpm.  Holds the CSR resident in HBM, the
// graph's HIP stream and timing events, a host copy of the offsets (for
// scheduling decisions) and reusable scratch.
#pragma once

#include <hip/hip_runtime.h>

#include <deque>
#include <vector>

#include "device_common.hpp"
#include "tiers.hpp"

constexpr uint32_t kSigLabels = 8;

// A handle's counters: 64 for sums and queues, then the bit matrix patterns' queue,
// whose counters have a cache line each.
constexpr uint32_t kQueueShards = 8, kQueueStride = 16, kPatternQueue = 64;
constexpr uint32_t kCounters = kPatternQueue + kQueueShards * kQueueStride;

struct gpm_graph {
  int device = 0;
  uint32_t n = 0;
  uint64_t m = 0;
  uint32_t max_deg = 0;
  uint32_t flags = 0;
  uint32_t n_labels = 0;
  // CSR (uint32 offsets and ids), resident on the device.
  uint32_t* off = nullptr;
  uint32_t* adj = nullptr;
  // COO source of every adjacency entry, built on first use.
  uint32_t* src = nullptr;
  // Labels and the label-partitioned index: ladj holds every list sorted by
  // (label, id); loff[v * (L + 1) + l] is where label l starts in v's list.
  uint32_t* labels = nullptr;
  uint32_t* ladj = nullptr;
  uint32_t* loff = nullptr;
  // Label alphabets of at most kSigLabels labels: sig[v] = degree << 32 |
  // per label l, min(15, neighbours of label l) in bits 4l..4l+3 -- the
  // matcher's degree and neighbour-label filter in one load.
  unsigned long long* sig = nullptr;
  // Position of every vertex in lverts within its label, and of every ladj entry's
  // vertex, built on first use by the matcher.
  uint32_t* lpos = nullptr;
  uint32_t* lloc = nullptr;
  // Vertices grouped by label: lverts[h_lvoff[l] .. h_lvoff[l+1]) have label l.
  uint32_t* lverts = nullptr;
  std::vector<uint32_t> h_lvoff;
  // Adjacency entries per (label of source, label of target), L x L; empty
  // when L > 1024.  Feeds the matcher's cost estimates.
  std::vector<double> h_lpair;
  std::vector<uint32_t> h_off;
  double met_degree = -1.0, met_skew = 1.0;  // see mean_met_degree
  // 1: every edge is once in both its lists and there are no loops, 0: not so (an
  // unsymmetrised edge file), -1: not known yet.
  int mirrored = -1;
  std::vector<uint32_t> h_labels;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double last_ms = 0.0;
  // Per-kernel marks of the last call: an event after each launch.
  static constexpr int kMaxMarks = 8;
  hipEvent_t mark_ev[kMaxMarks] = {};
  const char* mark_name[kMaxMarks] = {};
  double mark_ms[kMaxMarks] = {};
  int n_marks = 0;
  // Scratch: one growable device buffer plus a block of kCounters counters.
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  unsigned long long* counters = nullptr;
  // Root tiers built for earlier calls, keyed by the request that made them.
  // A deque keeps pointers to cached tiers valid while entries are added.
  std::deque<std::pair<gpm::TierKey, gpm::RootTiers>> tier_cache;
  // Cached algorithmic-byte totals per k (0 = not computed yet).
  uint64_t plan_bytes[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  // Symmetric graphs: the graph relabelled by degree rank (position in
  // (degree, id) order) with sorted lists (rk_off/rk_adj), and the
  // degree-oriented DAG, both built on first use by the motif counters.
  uint32_t* rk_off = nullptr;
  uint32_t* rk_adj = nullptr;
  gpm_graph* dag = nullptr;
  // Motif counters (motif_count.hip), built on first use: host offsets and
  // lower-neighbour counts of rk_off / rk_adj, and the task lists of the 4-cycle
  // kernels (hbm: some heavy task counts in HBM) and the triangle kernel.
  struct {
    std::vector<uint32_t> h_off;
    uint32_t* below = nullptr;
    void *heavy = nullptr, *light = nullptr, *triangles = nullptr;
    uint32_t n_heavy = 0, n_light = 0, n_triangles = 0;
    bool hbm = false, built = false;
  } motif;
  // Last prepared matching batch (match.hip), replayed on identical calls.
  void* match_cache = nullptr;
  // Instantiated hipGraph of repeated edge-parallel triangle counts, and the
  // per-block partial sums of the edge kernel (tc.hip).
  hipGraphExec_t tc_exec = nullptr;
  hipGraph_t tc_graph = nullptr;
  unsigned long long* tc_partial = nullptr;
  // ORIENTED graphs: the same DAG relabelled in a topological order
  // (toff/tadj, every edge from a lower to a higher id; h_rank[v] = new id
  // of v), built on first use by the k-clique kernels: by total degree where
  // that order is topological (then the most linked vertices have the highest
  // ids), else in the order of Kahn's algorithm.
  uint32_t* toff = nullptr;
  uint32_t* tadj = nullptr;
  bool unranked = false;  // total degree gives no topological order
  std::vector<uint32_t> h_rank;
  // SYMMETRIC graphs: block mask of the counting formulation's prefilter,
  // bmask[v] bit b set when v has a neighbour w with (w >> bmask_shift) == b,
  // built on first use.
  unsigned long long* bmask = nullptr;
  uint32_t bmask_shift = 0;
  // SYMMETRIC graphs: adjacency bit matrices of the fixed patterns
  // (pattern_bits.hip), built on first use; nbits_off: they cannot be built,
  // nbits_mirrored: every edge is in both its lists.
  uint32_t* nbits = nullptr;
  bool nbits_off = false, nbits_mirrored = false;
};

namespace gpm {

// Host-to-device copy ordered on the handle's stream and complete on return.
// (A plain hipMemcpy runs on the null stream, which does not order against
// the handle's non-blocking stream, and may return before a pageable
// source's DMA lands: a kernel launched next on the handle's stream could
// read the old contents.)
int h2d(gpm_graph* g, void* dst, const void* src, size_t bytes);
// A non-blocking stream of the current device (a call for a handle of another device
// gets one too), its caller's until stream_give, which waits for its work.
hipError_t stream_take(hipStream_t* stream);
void stream_give(hipStream_t stream);
// Grows g->scratch to at least `bytes`; returns status.
int ensure_scratch(gpm_graph* g, size_t bytes);
// Builds g->src (COO sources) if missing.
int ensure_src(gpm_graph* g);
// Zeroes the first `count` counters with a kernel (no memset node, so the
// sequence stays valid inside a captured graph).
int zero_counters(gpm_graph* g, int count);
// Starts / stops event timing around the kernels of one mining call.
int timing_begin(gpm_graph* g);
// Records an event after the kernel just launched; `name` must be static.
int timing_mark(gpm_graph* g, const char* name);
// The results at src go to dst behind the stop mark: one wait for both.
int timing_end(gpm_graph* g, void* dst = nullptr, const void* src = nullptr, size_t bytes = 0);
// Mean list length an adjacency entry meets, dw = sum d^2 / sum d, and (g->met_skew) the
// mean square over its square, sum d^3 / (dw^2 sum d): 1 where all lists have one
// length.  Kept on the handle.
double mean_met_degree(gpm_graph* g);
// Number of compute units of the handle's device.
int device_cus(const gpm_graph* g);
// Builds g->toff/tadj/h_rank if missing; GPM_EINVAL if the graph has a cycle.
int ensure_topo(gpm_graph* g);
// The same where the order by total degree is topological; otherwise (and where
// its buffers do not fit) g->toff stays null and the status is GPM_OK.
int try_topo(gpm_graph* g);
// Orients the SYMMETRIC graph by (degree, id) (prep.hip): CSR in new device buffers
// *d_off, *d_adj, the caller's, and the offsets on the host; lists keep their order.
int orient_device(gpm_graph* sym, uint32_t** d_off, uint32_t** d_adj, std::vector<uint32_t>* h_off);
// The vertices [first, first + count) by decreasing out-degree, equal ones by id, as
// rank[v] where rank (a host array of all vertices) is given, to out (prep.hip).
int degree_order_device(gpm_graph* g, uint32_t first, uint32_t count, const uint32_t* rank,
                        uint32_t* out);
// Relabels the ORIENTED graph g by (out-degree + in-degree, id) on the device
// (prep.hip).  Where every edge goes up in that order -- gpm_graph_orient and
// gpm_csr_orient give such graphs -- *ordered is set and *toff / *tadj /
// *rank hold the relabelled CSR (the caller's) and the new id of every
// vertex; otherwise the caller has to find a topological order itself.
int topo_relabel_device(gpm_graph* g, uint32_t** toff, uint32_t** tadj, std::vector<uint32_t>* rank,
                        bool* ordered);
// Wraps a CSR already resident on the device (d_off: n + 1 entries, d_adj:
// m) into a new handle that owns d_off, d_adj and `stream`; h_off is the host
// copy of the offsets, h_adj the host copy of the adjacency (needed only
// with labels, for the label index).  On failure everything given is freed.
int adopt_device_csr(uint32_t n, uint64_t m, uint32_t* d_off, uint32_t* d_adj,
                     std::vector<uint32_t>&& h_off, const uint32_t* h_adj, const uint32_t* labels,
                     uint32_t n_labels, uint32_t flags, hipStream_t stream, gpm_graph** out);
// Floats of a packed MLP: mean[4], std[4], W1[64x4], b1[64], W2[64x64],
// b2[64], W3[64], b3[1] (the order of gpm_mlp_predict's arguments).
constexpr size_t kMlpWeights = 4 + 4 + 64 * 4 + 64 + 64 * 64 + 64 + 64 + 1;
// log1p-domain outputs of the packed MLP at d_packed for n feature rows
// (4 floats each, raw -- log1p and normalisation happen inside), enqueued on
// `stream` (mlp.hip).
int mlp_forward(const float* d_feat, uint32_t n, const float* d_packed, float* d_out, int cus,
                hipStream_t stream);
// Fixed patterns on adjacency bit matrices (pattern_bits.hip).  *ok: pattern `pid` in
// this form is counted that way; the matrices are there.
int prepare_pattern_bits(gpm_graph* g, int pid, bool counting, bool* ok);
// Enqueues the count of pattern `pid` (the direct formulation's h[0 .. 5], or the
// counting one's h[1], h[2]) into the zeroed out[6]; *queue is zero on entry.
int launch_pattern_bits(gpm_graph* g, int pid, bool counting, unsigned long long* queue,
                        unsigned long long* out);
// Releases the cached matching batch of g (match.hip).
void free_match_cache(gpm_graph* g);

}  // namespace gpm
