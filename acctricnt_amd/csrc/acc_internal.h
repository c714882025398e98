// Internal declarations shared by the HIP translation units of libacc_cn.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "acc_cn.h"
#include "fwd_plan.h"

// Sets the thread's last error and returns code.
int acc_set_error(int code, const std::string &msg);

struct acc_graph;
// Records a named HIP event on the graph's stream; acc_cn_timings reports the
// intervals between consecutive events under the later event's name.
int record_event(acc_graph *g, const char *name);

#define ACC_HIP_TRY(expr)                                                                   \
  do {                                                                                      \
    hipError_t acc_e_ = (expr);                                                             \
    if (acc_e_ != hipSuccess)                                                               \
      return acc_set_error(ACC_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(acc_e_)); \
  } while (0)

#define ACC_TRY(expr)        \
  do {                       \
    int acc_rc_ = (expr);    \
    if (acc_rc_) return acc_rc_; \
  } while (0)

// One lane of the staged host copies: a stream and two pinned buffers.
struct CopyLane {
  hipStream_t stream = nullptr;
  void *buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
};

// Device memory of a context's graphs and workspaces.  Freed blocks are kept
// for the next allocation of their size (up to an eighth and 64 KiB larger),
// at most kPoolBytes of them, the largest going back to the device first;
// all go back when an allocation fails and when the context ends.  A
// hipMalloc and a hipFree take 30 and 40 us, and an upload with a SCAN query
// made some 40 of each: 2.8 of its 7.6 ms at 262,144 vertices and 7.3M slots.
// A block is reused without waiting: whoever frees one has waited for the
// work that uses it, or that work is queued on the context's stream.  So a block
// used on another stream is not touched there before that stream has waited for
// an event recorded on the context's stream after the alloc.  Safe from several
// threads.
class DevicePool {
 public:
  hipError_t alloc(void **p, size_t bytes);
  void free(void *p);
  void trim();
  uint64_t idle_bytes();
  ~DevicePool() { trim(); }

 private:
  void give_back(size_t most);  // with mu_ held
  static constexpr size_t kPoolBytes = size_t(4) << 30;
  std::mutex mu_;
  std::multimap<size_t, void *> idle_;
  std::unordered_map<void *, size_t> size_;  // of every block, idle or not
  size_t idle_bytes_ = 0;
};

// Words of pinned host memory that kernels write results to: a total is there
// once the stream is synchronized, without a copy.  A call takes a word for as
// long as it waits; with none left (or none to be had) it copies instead.  Safe from
// several threads.
struct HostWord {
  volatile unsigned long long *host = nullptr;
  unsigned long long *dev = nullptr;
};
class HostWords {
 public:
  bool init();
  bool take(HostWord *w);
  void give(const HostWord &w);
  ~HostWords();

 private:
  static constexpr uint32_t kWords = 64;
  std::mutex mu_;
  unsigned long long *base_ = nullptr;
  std::vector<HostWord> idle_;
};

struct acc_ctx {
  DevicePool pool;
  HostWords words;
  int device = 0;
  hipStream_t stream = nullptr;
  int num_cus = 0;
  size_t lds_per_block = 0;
  std::mutex copy_mu;             // the copy lanes serve one transfer at a time
  std::vector<CopyLane> lanes;    // allocated at the first large pageable transfer
  unsigned long long *na_scratch = nullptr;  // device address of the allocation-free entry point's scratch
};

namespace accnoalloc {
// Device address of acc_noalloc.hip's file-scope scratch array on `device`
// (the current device), looked up once per device.
int bind_scratch(int device, unsigned long long **addr);
}  // namespace accnoalloc



// Per-edge plans (bitmap and merge paths): chunks of at most kChunk upper
// slots of every source, by d_u.  Wave units: a source with d_u <= 256 and at
// most 64 upper slots, one wave each, N(u) in a wave-private LDS table or
// sorted run.  Block units: the bitmap path keeps N(u) in an LDS hash table
// of 2^12, 2^14 or 2^15 keys (d_u up to half of that) or, for hubs, in an HBM
// bitmap; the merge path stages N(u) in LDS windows of 2^11 ids (the first
// class, and the units behind the hub units) or 2^13 ids (the others).
enum EdgeClass { kEdgeWave = 0, kEdgeHash12, kEdgeHash14, kEdgeHash15, kEdgeHub, kEdgeClasses };
constexpr uint32_t kEdgeWaveDeg = 256;  // d_u of a wave unit
constexpr int kEdgeWaveLog = 8;         // log2 kEdgeWaveDeg
static_assert((1u << kEdgeWaveLog) == kEdgeWaveDeg, "wave-unit runs are searched in kEdgeWaveLog steps");
constexpr uint32_t kEdgeWaveUp = 64;    // upper slots of a wave unit
struct EdgePlan {
  FwdUnit *d_units[kEdgeClasses] = {};  // hub units: nlow = the hub's bitmap in its batch's pool
  uint32_t n_units[kEdgeClasses] = {};
  uint32_t n_small = 0;                 // units with d_u <= 256 behind the hub units, where hub bitmaps lie in LDS
  uint32_t *d_hubs = nullptr;           // hub sources in order
  uint32_t n_hubs = 0;
  std::vector<uint32_t> hub_batch;       // batch k: hubs [hub_batch[k], hub_batch[k+1])
  std::vector<uint32_t> hub_unit_batch;  // ... and hub units [hub_unit_batch[k], hub_unit_batch[k+1])
  uint32_t *d_pool = nullptr;            // bitmaps of one batch of hubs, zero between passes
  uint32_t pool_hubs = 0;
  uint64_t pool_words = 0;               // words per bitmap: ceil(n / 32)
  int idx_shift = 0;                     // LDS index of the hash units: one bit per 2^idx_shift bitmap words
  int hub_idx_shift = 0;                 // LDS index of the hub units: one bit per 16 << hub_idx_shift ids
  bool valid = false;
};
constexpr uint32_t kEdgeHashMax = 1u << 14;  // largest d_u an LDS hash table holds

// Dense sources of the forward path (k_dense.hip): graph k of the partition
// (one graph without a partition) starts at vertex first[k] and its first
// limit[k] vertices are its dense sources.
struct DensePlan {
  std::vector<uint32_t> first, limit;
  uint32_t most = 0;              // largest limit
  uint32_t max_low = 0;           // most lower neighbors of a dense source
  FwdUnit *d_units = nullptr;     // units of the shard's dense sources (nlow unused)
  uint32_t n_units = 0;
  uint4 *d_vmeta = nullptr;       // per vertex: first slot, first low group, hit base, rows
  uint4 *d_low = nullptr;         // low lists, groups of eight 16-bit ids
  uint32_t *d_large = nullptr;    // vertices with large hit matrices, then (one allocation)
  uint32_t *d_mid = nullptr;      // those with medium ones
  uint32_t n_large = 0, n_mid = 0;
  uint32_t hit_cap = 0;           // most rows of a matrix that is kept
  uint64_t hit_bytes = 0;         // of all matrices
  uint8_t *d_hits = nullptr;      // allocated at the first per-slot pass
  bool no_hits = false;           // ... which found no memory for them: every row is counted by atomics
  uint64_t bytes = 0, hits_held = 0;
  bool allowed = true;            // the plan may have dense sources
  bool tables = false;            // d_vmeta, d_low and d_large match first and limit
};

constexpr uint32_t kAdjPad = 64;  // ids allocated past the adjacency array's end, 0

struct acc_graph {
  acc_ctx *ctx = nullptr;
  uint32_t n = 0;
  uint64_t m = 0;
  uint32_t max_deg = 0;
  uint32_t max_low = 0;  // max |N<(b)|
  // resident CSR and outputs
  uint32_t *d_off = nullptr;
  int32_t *d_adj = nullptr;
  int32_t *d_cnt = nullptr;
  uint32_t *d_hs = nullptr;             // first upper slot of every vertex
  uint32_t *d_rev = nullptr;            // reverse slot of every upper slot, ~0 elsewhere (built at upload)
  unsigned long long *d_sum = nullptr;  // sum over upper slots of the raw counts (3T) in sum_parts; [1]: T alone
  int32_t *d_flags = nullptr;           // validation flags
  unsigned long long *d_tri_parts = nullptr;  // partial sums of the triangle-only pass
  bool tri_parts_zero = false;                // the last pass left them zero
  int32_t *d_src = nullptr;             // source vertex of every slot (built for SCAN)
  int32_t *d_old = nullptr;             // caller vertex ids for cluster ids (NULL: identity)
  // similarity index (built for serving): every vertex's slots sorted by a
  // monotone float key of cn^2 / ((d_u+1)(d_v+1)), descending
  float *d_skey = nullptr;     // sorted keys
  int32_t *d_snbr = nullptr;   // neighbor of every sorted position
  uint32_t *d_sslot = nullptr; // original slot of every sorted position
  bool cnt_plus2 = true;                // counts stored as 2 + |N(u) ∩ N(v)|
  bool relabelled = false;              // relabelled by degree at upload (d_old holds the old ids)
  // forward plan, binned by degree skew
  FwdUnit *d_fwd_wave = nullptr;  // wave packs of small sources: {b0, b1, upper slots, lower entries}
  uint32_t n_fwd_wave = 0;
  FwdUnit *d_fwd_block = nullptr;  // one workgroup per chunk of upper slots, N<(b) in LDS
  uint32_t n_fwd_block = 0;
  FwdUnit *d_fwd_big = nullptr;  // |N<(b)| beyond the LDS table: global-memory lookups
  uint32_t n_fwd_big = 0;
  DensePlan dense;           // dense sources and their tables
  bool symmetric = false;    // every slot has its reverse (checked when the reverse slots are built)
  bool split_counts = false; // leave per-probe hits in the upper slots (the shard work estimate reads them)
  std::vector<uint32_t> h_gvoff;  // the partition's vertex offsets
  EdgePlan edge;  // per-edge plans, built at the first bitmap or merge pass
  uint64_t device_bytes = 0;
  // tuning parameters (acc_graph_set_param)
  int fwd_unroll = 4;
  int auto_path = ACC_PATH_FORWARD;  // what ACC_PATH_AUTO runs
  uint32_t wave_slots = accfwd::kWaveSlots;  // wave-unit bin: at most this many upper slots
  uint32_t wave_low = accfwd::kWaveCap;      // ... and |N<(b)| at most this
  uint32_t chunk = accfwd::kChunk;           // upper slots per workgroup unit
  uint32_t persist = 256;                    // counting grid: 0 one workgroup per task, else at most this many
                                             // workgroups per CU looping over the tasks
  uint32_t bmp_hash_max = 256;               // bitmap path: d_u above this goes to the HBM bitmaps
  uint32_t bmp_batch = 4096;                 // bitmap path: hub bitmaps built and probed per batch
  uint32_t shard_lo = 0, shard_hi = 0;       // forward sources [shard_lo, shard_hi) (the whole graph: 0, n)
  std::vector<uint64_t> h_work;              // prefix of the forward probe work per source (n + 1), for shards
  // host copies kept for plan rebuilds: offsets, first upper slot and smallest
  // neighbor (the vertex itself when it has no lower neighbor) of every vertex
  std::vector<uint32_t> h_off;
  std::vector<uint32_t> h_hs;
  std::vector<int32_t> h_lo;
  // multi-graph partition: graph k owns vertices [gvoff[k], gvoff[k+1])
  uint32_t num_parts = 0;
  uint32_t *d_gvoff = nullptr;
  uint32_t *d_gsoff = nullptr;           // slot offsets: graph k owns slots [gsoff[k], gsoff[k+1])
  unsigned long long *d_gtot = nullptr;  // per-graph sum of raw counts (= 6 T_k)
  bool totals_valid = false;             // d_gtot holds the last pass's totals
  // captured counting pass
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  bool graph_plus2 = true;  // count format the captured pass writes
  // last results / timing
  bool have_result = false;
  bool counts_share = false;  // the counts are one share's (a forward pass restricted by acc_graph_set_shard)
  bool graph_share = false;   // the captured pass counts one share
  std::vector<hipEvent_t> events;
  std::vector<std::string> event_names;
  bool timing_valid = false;
};

// Per-edge path launchers (k_paths.hip).
namespace accpaths {
// Graphs of at most this many vertices keep a hub's bitmap in LDS.
constexpr uint32_t kLdsBitmapIds = 1u << 19;
inline bool hubs_in_lds(const acc_graph *g) { return g->n <= kLdsBitmapIds; }
int launch_bitmap(acc_graph *g, int plus);
int launch_merge(acc_graph *g, int plus);
}  // namespace accpaths

// acc_graph_upload, with dense sources or without (acc_runtime.hip).
int acc_upload(acc_ctx *ctx, uint32_t n, uint64_t m, const uint32_t *node_off, const int32_t *edge_dst, uint32_t flags,
               bool dense, acc_graph **out);

// Builds the slot -> source array (acc_scan.hip).
int acc_graph_ensure_src(acc_graph *g);

constexpr int kScanCounters = 16;
constexpr uint32_t kItem = 256;  // list positions per work item of the index path

// One SCAN query as the batched SCAN kernels see it (acc_scan.hip): the
// resident graph's arrays, the query's buffers and its exact eps = p/q, mu.
struct ScanJob {
  const uint32_t *off;
  const int32_t *adj;
  const int32_t *src;
  const int32_t *cnt;
  const int32_t *old;  // caller vertex ids, or NULL
  uint8_t *sim;
  const float *skey;     // similarity index (NULL: per-slot kernels)
  const int32_t *snbr;
  const uint32_t *sslot;
  uint32_t *send;        // per vertex: end of the possibly-similar prefix
  int2 *work;            // work items (vertex, first list position) of the index path
  int32_t *core_cnt;
  int32_t *label;
  int32_t *parent;
  int32_t *rmin;
  int32_t *rmax;
  int32_t *cl;
  int32_t *cid;
  unsigned long long *counters;  // core, cluster, hub, outlier, pairs, index-path sums (5..7), item counts (8, 9)
  int8_t *out_label;             // host-mapped copies of the results (NULL: none)
  int32_t *out_cid;
  unsigned long long *out_counters;
  int2 *pairs;
  unsigned long long pairs_cap;
  unsigned long long p2, q2;
  uint64_t m;
  uint32_t n;
  int32_t add;  // added to cnt to get 2 + |N(u) ∩ N(v)|
  int32_t mu;
  uint32_t symmetric;  // every slot has its reverse (an upload trusted without validation may not)
  uint32_t vb0, vbn;  // workgroups of vertex-sized launches
  uint32_t sb0, sbn;  // workgroups of slot-sized launches
};

// A launch's job table, passed by value as a kernel argument (no copy to
// device memory before the kernels): at most kMaxJobs jobs per launch.
constexpr int kMaxJobs = 14;
struct JobTable {
  ScanJob jobs[kMaxJobs];
  int32_t nj;
};
static_assert(sizeof(JobTable) <= 3800, "kernel arguments are limited to 4 KiB");

// Per-query device buffers, grown on demand.
struct ScanBuffers {
  uint8_t *sim = nullptr;
  uint32_t *send = nullptr;
  int2 *work = nullptr;
  int32_t *core_cnt = nullptr;
  int32_t *label = nullptr;
  int32_t *parent = nullptr;
  int32_t *rmin = nullptr;
  int32_t *rmax = nullptr;
  int32_t *cl = nullptr;
  int32_t *cid = nullptr;
  unsigned long long *counters = nullptr;
  uint32_t n_cap = 0;
  uint64_t m_cap = 0;
  uint64_t bytes = 0;
  DevicePool *pool = nullptr;  // the context's
  bool pooled = false;         // the buffers come from the pool, else from hipMalloc (the pool then
                               // gives its idle blocks back where that fails)
};

namespace accscan {
void free_buffers(ScanBuffers *b);
int reserve_buffers(ScanBuffers *b, uint32_t n, uint64_t m);
uint64_t buffer_bytes(uint32_t n, uint64_t m);
int check_eps(int64_t eps_num, int64_t eps_den);
ScanJob make_job(const acc_graph *g, const ScanBuffers &b, int64_t eps_num, int64_t eps_den, int32_t mu);
void plan_jobs(ScanJob *jobs, int nj, int cus, uint32_t *vblocks, uint32_t *sblocks);
// Enqueues the eight per-slot SCAN kernels over the jobs of jt (planned).
int launch_jobs(const JobTable &jt, uint32_t vblocks, uint32_t sblocks, hipStream_t s);
int launch_pairs(const JobTable &jt, uint32_t sblocks, hipStream_t s);
// Builds the similarity index of a resident graph (counts computed, slot
// sources built); enqueued on the graph's context stream.
int build_index(acc_graph *g);
// Whether the index decides eps = p/q exactly (p, q < 2^26) on graph g.
bool index_usable(const acc_graph *g, int64_t p, int64_t q);
// The six index-path SCAN kernels over nj jobs whose skey is set.
int launch_index_jobs(const JobTable &jt, uint32_t vblocks, uint32_t sblocks, hipStream_t s);
}  // namespace accscan

// Dense sources (k_dense.hip).
namespace accdense {
constexpr uint32_t kMaxRows = 4096;  // most rows of a hit matrix that is kept
// Most bytes of a graph's hit matrices: 32-bit offsets, 16 bytes per slot.
inline uint64_t most_hit_bytes(uint64_t m) {
  const uint64_t by_slots = 16 * m + (1u << 20);
  return by_slots < 0xe0000000ull ? by_slots : 0xe0000000ull;
}
// The vertex records, low lists and matrix offsets for dense.first / limit.
int build_tables(acc_graph *g);
void free_tables(acc_graph *g);
// What a pass needs, where the plan has dense units: the tables and, with
// `slots`, the hit matrices (allocated once; zeroed where only a share's rows
// are written; passes count by atomics where there is no memory for them, or
// where the stream is recorded before they are there).
int ensure(acc_graph *g, bool slots);
int clear_hits(acc_graph *g);
int launch_count(acc_graph *g);
int launch_triangles(acc_graph *g, unsigned long long *total);
// Adds the hit matrices' row and column sums to the lower slots.
int launch_rows(acc_graph *g);
}  // namespace accdense

// Kernel launchers (k_forward.hip).
namespace accfwd {
// Partial triangle totals of the triangle-only pass: kTriParts counters one
// 128-byte line apart, workgroup w adding into counter w mod kTriParts, so
// the atomics of many small units do not queue on one address.
constexpr int kTriParts = 256;
// A pass's total likewise, in kSumParts counters at sum_parts(g): d_sum[0] takes
// their sum where no pinned word is to be had, d_sum[1] the triangle-only total.
constexpr int kSumParts = 64;
constexpr int kSumStride = 16;
inline unsigned long long *sum_parts(const acc_graph *g) { return g->d_sum + kSumStride; }
constexpr int kTriStride = 16;  // unsigned long longs per 128-byte line
// Whether a pass collects every edge's count in its lower slot, which the
// combine copies to the upper one.  Otherwise (an upload trusted without
// validation that is not symmetric, the shard work estimate) the upper slot holds
// its probe's hits, the lower slot the rest, and the combine adds them.
inline bool lower_counts(const acc_graph *g) { return g->symmetric && !g->split_counts; }
// Workgroups per compute unit of k_fwd_count's grid, at most, for a `persist` parameter.
// A workgroup holds its place until the slowest of its waves has ended, so
// several tasks a workgroup even out unequal packs: at 64 workgroups per
// compute unit 512 packed graphs (average degree 22) took 5.60 ms against
// 6.03 at 256, Erdos-Renyi n = 2M, degree 26, 1.48 against 1.55, n = 3M,
// degree 40, 4.05 against 4.19.  Below an average degree of 16 packs are
// short and alike and the finer grid ends evenly: n = 8M, degree 8, 1.76 ms at
// 256 against 1.81 at 64; degrees 16 and 20 are within 1% either way.
inline uint32_t count_persist(const acc_graph *g, uint32_t persist) {
  return g->m >= 16ull * g->n && persist > 64 ? 64 : persist;
}
// Every slot gets `fill`.
int launch_init(acc_graph *g, int fill);
// Slot-parallel over the sources in d_cnt (accprep::slot_sources).  With
// validate, d_flags[0] gets flag 8 for an upper slot without reverse and
// d_flags[2..3] (a uint64) the number of upper slots.
int launch_build_rev(acc_graph *g, bool validate);
// Triangle total only (forward path, no per-slot counts) into d_sum[1].
// The total goes to d_sum[1], and to *copy (device-visible host memory) if given.
int launch_triangles(acc_graph *g, unsigned long long *copy);
// *to = the sum of the pass's total counters.
int launch_publish(acc_graph *g, unsigned long long *to);
int launch_count(acc_graph *g);
int launch_count_big(acc_graph *g);
// Copies the lower slots' counts to the upper ones or adds the two
// (lower_counts); with a partition, also the per-graph totals (which
// launch_init zeroes).
int launch_combine(acc_graph *g, int plus);
int launch_graph_totals(acc_graph *g, int plus);
// Slot-parallel over the sources in d_cnt (accprep::slot_sources).
int launch_validate(acc_graph *g);
// Per-vertex plan inputs into g->d_hs (first upper slot) and lo (min(N(v) ∪ {v}));
// each of the vertex_meta_blocks(g) workgroups w leaves the max |N<(v)| of its
// vertices in maxes[2 w] and their max degree in maxes[2 w + 1].
uint32_t vertex_meta_blocks(const acc_graph *g);
int launch_vertex_meta(acc_graph *g, int32_t *lo, uint32_t *maxes);
// Forward work estimate of every source b into work[b]: the sum over its
// upper slots (b, c) of |N(c) ∩ [0, b)| + 4 + 2 hits, plus |N<(b)| + 256 per
// unit, hits read from d_cnt's upper slots after a pass without the combine.
int launch_source_work(acc_graph *g, unsigned long long *work);
}  // namespace accfwd

// Upload-time preparation (k_prepare.hip).  slot_sources writes the source
// vertex of every slot into d_cnt (d_rev is its scratch); both arrays are
// free until the reverse slots are built and the first pass runs.
// relabel_degree, given those sources, rewrites d_off and d_adj in place by
// degree (d_rev is its scratch) and keeps the old id of every new vertex in
// d_old; the sources must be recomputed after it.  reverse_slots, given the
// sources and d_hs, fills d_rev (d_cnt is its scratch) and returns the number
// of upper slots; an upper slot without its reverse sets flag 8 in d_flags,
// and with validate a count other than m / 2 leaves d_rev unbuilt.
namespace accprep {
int slot_sources(acc_graph *g);
int relabel_degree(acc_graph *g);
int reverse_slots(acc_graph *g, bool validate, uint64_t *upper);
}  // namespace accprep
