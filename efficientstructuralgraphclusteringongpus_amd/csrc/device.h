// Device-side structures shared by the C-ABI implementation and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "scan_rules.h"

#define SGC_HIP(call)                                                                             \
  do {                                                                                            \
    hipError_t e_ = (call);                                                                       \
    if (e_ != hipSuccess)                                                                         \
      return ::sgc::fail(SGC_EDEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, \
                         __LINE__);                                                               \
  } while (0)

namespace sgc {

constexpr int kWave = 64;
constexpr int32_t kNoLabel = 0x7FFFFFFF;


// Counters written by the kernels (64-bit words of one buffer).
//
// Atomics on one word are done one after the other, about 12 ns each on
// this card, so a word that every block of a grid adds to costs 50 us per
// 4096 blocks.  Sums are therefore kept in kStripes copies (count_add; a
// block's copy goes by its index), read on the device by count_total /
// count_any and summed on the host by fold_counters; counters whose atomics
// return a value (queues, reservations) have a 128-byte line each.
// k_finalize on 1M vertices: 101 us with single words, 9 with stripes.
enum Counter {
  // sums, striped
  kCntUEdges = 0,
  kCntSimilar,
  kCntCores,
  kCntClusters,
  kCntBorders,
  kCntHubs,
  kCntOutliers,
  kCntProbes,
  kCntLoaded,   // short-row elements loaded by the claims (consumed or not)
  kCntClaims,   // claims taken
  kCntLabeled,  // entries of labelled rows (cores, borders): picks the classify pass's side
  kCntMarked,   // cores marked by the core pass: none lets the later edge passes return at once
  kCntRedo,     // deferred edges the union-find and border passes need: decided after all
  kCntRedoOwned,  // owned undecided entries of that second similarity round
  kCntDeferred,   // edges deferred by the core-check pruning and never needed
  kStripeSlots = 16,
  // single words
  kCntOverflow = 16,  // owned undecided entries, when more than the unit array holds (asymmetric input)
  kCntStamp0 = 17,    // device clock when each phase's first kernel started (Stamp; 0: it was not launched)
  kCntTimer0 = 32,    // phase timers of debug builds (SGC_PHASE_TIMERS): 5 per tier
  kCntSlots = 48,     // host copies: the sums and single words above
  kCntUnits1 = 48,    // small-tier work units
  kCntUnits2 = 64,    // workgroup-tier work units
  kCntQueue1 = 80,    // small-tier units claimed beyond each block's first
  kCntQueue2 = 96,    // workgroup-tier units, likewise
  kCntDense = 112,    // owned undecided entries listed for the one-wave-per-edge kernel
  kCntTiny = 128,     // tiny owners listed by the planner for the tiny-owner kernel, or wave-filter owners
  kCntFUnits1 = 144,  // units of the workgroup filter
  kCntFUnits2 = 160,  // units of the large owners
  kCntFQueue1 = 176,
  kCntFQueue2 = 192,
  kCntHUnits = 208,   // units of the hash filter
  kCntHQueue = 224,
  kCntRecords = 224,  // chips, which have no hash filter: packed edge records placed
  kCntPieces = 240,   // pieces of labelled rows for the classify pass
  kCntWPieces = 248,  // pieces of wave-filter owners beyond their first (the line is the other's only later)
  kStripe0 = 256,
  kStripes = 32,
  kCntWords = kStripe0 + kStripes * kStripeSlots
};

// Phase times come from the device clock, read by the first block of a phase's
// first kernel: an event between two kernels holds the second back by about
// 2 us, which a pass of 150 us feels.
enum Stamp {
  kStampInit = 0,
  kStampSim,         // first similarity kernel
  kStampSimRest,     // first similarity kernel of the short owners
  kStampExactLarge,  // workgroup-tier exact kernel
  kStampExactSmall,
  kStampCore,
  kStampCluster,
  kStampBorder,
  kStampClassify,
  kStampEnd,
  kStamps
};

// Adds the stripes of a counter buffer's host copy to its sums.
inline void fold_counters(uint64_t* c) {
  for (int i = 0; i < kStripes; ++i)
    for (int q = 0; q < kStripeSlots; ++q) c[q] += c[kStripe0 + i * kStripeSlots + q];
}

// Similarity kernels selectable per context.
enum SimImpl { kSimTiered = 0, kSimWavePerEdge = 1 };

// Results of a pass up to this size go to host memory through the context's
// page-locked staging, written by the pass's last kernel (R-MAT-16, 320 KB:
// 246 us through two pageable copies, 215 staged).
constexpr size_t kStageBytes = 512u << 10;

// Page-locked staging of a context: kBounces buffers of kBounceBytes.
constexpr int kBounces = 4;
constexpr size_t kBounceBytes = 8u << 20;

// Most memory of a freed graph's row copies that a context keeps: releasing it
// takes 0.25 ms, and a caller that uploads, runs and releases graphs of 3e7
// entries one after another (6.0 ms each) had 6.4 ms with it released each time.
constexpr size_t kSpareBytes = 512u << 20;

// Grow-only device (or page-locked host) allocation owned by a context.
struct DevBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
};

}  // namespace sgc

struct sgc_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  char name[256] = {0};
  int cu_count = 0;
  sgc::DevBuf work;      // per-pass arrays
  sgc::DevBuf counters;  // kCntWords x uint64
  uint64_t* host_counters = nullptr;  // page-locked: kCntWords words, then kStageBytes for small results
  uint64_t* host_counters_dev = nullptr;  // its device address
  double clock_khz = 100000.0;  // rate of the device clock (Stamp)
  hipEvent_t ev[8] = {};
  int sim_impl = sgc::kSimTiered;
  void* scratch = nullptr;  // this GPU's static scratch (sgc_scan_device_noalloc)
  // page-locked staging for copies from and to pageable memory (one
  // allocation of sgc::kBounces buffers, made at the first such copy and
  // kept until destroy)
  char* bounce = nullptr;
  hipEvent_t bounce_done[sgc::kBounces] = {};
  sgc::DevBuf host_work;    // page-locked work memory of out-of-core passes
  bool prune = false;       // core-check pruning in passes that return no similarity flags (sgc_ctx_set_pruning)
  size_t work_pass = 0;  // bytes of `work` that the passes so far needed (uploads reserve them, and may sort in more)
  sgc_dgraph* packed = nullptr;  // the graphs that have compact row copies, linked by next_packed
  sgc::DevBuf spare;     // the row copies' memory of a graph freed earlier, for the next one (sgc::kSpareBytes)
};

namespace sgc {
// Planner knobs of the tiered similarity kernels (see sgc_tuning).
struct SimTuning {
  uint32_t small_max_degree = 1024;  // owners up to this degree take the small tier (<= 1024)
  double small_unit_work = 262144.0;  // short-row elements per small-tier unit
  double large_unit_work = 8388608.0;  // per workgroup-tier unit
  uint32_t hash_tables = 1;  // 1: cuckoo hashes where they fit; 0: linear probing and bitmap windows only
  uint32_t tiny_work = 2048;  // owners with sum over their edges of d(a) + d(b) <= this: merged, one edge per lane
};
}  // namespace sgc

namespace sgc {
// Out-of-core chip of two row blocks [lo0, hi0) and [lo1, hi1) (equal for a
// chip of one block): the prep kernel keeps only owned edges whose endpoints
// lie one in each block.
// keep0: entries of rows in [lo0, hi0) outside the pair keep their flag (an
// earlier chip of the same group of blocks decided them); every other entry
// outside the pair is marked kFlagUSkip.
struct PairFilter {
  uint32_t lo0 = 0, hi0 = 0, lo1 = 0, hi1 = 0;
  bool on = false;
  bool keep0 = false;
};
}  // namespace sgc

struct sgc_dgraph {
  sgc_ctx* ctx = nullptr;
  uint32_t n = 0;
  uint32_t m = 0;
  uint32_t max_degree = 0;
  uint32_t* row_ptr = nullptr;  // n + 1
  int32_t* adj = nullptr;       // m
  uint32_t* src = nullptr;      // m: row of each entry
  // m: position of the reverse entry (v, u) of each entry (u, v); resident
  // graphs only (null: the similarity kernels find it themselves)
  uint32_t* mirror = nullptr;
  // m: degree of each entry's neighbour, d(adj[k]); resident graphs only
  // (null: the prep kernel gathers it from the row offsets)
  uint32_t* ndeg = nullptr;
  // Row x is adj[row_begin[x], row_end[x]) for every row the similarity
  // kernels read; row_end[x] - row_begin[x] is x's degree for every x.  A
  // resident graph uses row_ptr and row_ptr + 1; an out-of-core chip holds
  // only some rows (absent rows: a range of the right length that is never
  // read).
  const uint32_t* row_begin = nullptr;
  const uint32_t* row_end = nullptr;
  sgc::SimTuning tuning;
  sgc::PairFilter pair;
  // Window-offset index of a resident graph with n > 2^20 (null otherwise):
  // (wcount + 1) positions per row, where the row crosses each 2^20-id
  // window boundary; the workgroup tier then streams exact window slices.
  uint32_t* woff = nullptr;
  uint32_t wcount = 0;
  // Compact copies of the rows for the filter stages (filter.hip: bitmaps
  // and hash groups, 9 bytes per entry); graphs of a serving engine, and
  // uploads without room, have none (null).  An allocation of their own: the
  // context takes them back when it finds no room for something else.
  char* packed = nullptr;
  size_t packed_cap = 0;  // bytes of that allocation
  sgc_dgraph* next_packed = nullptr;
  sgc_dgraph** link_packed = nullptr;  // the pointer that holds this graph in the context's list, or null
  // the allocations that hold the other arrays: one for all of them, or,
  // where that much was not free in one piece, one for each that was
  void* blocks[4] = {};
};

namespace sgc {

// Arrays one SCAN pass needs on the device.
struct PassBuffers {
  uint8_t* flag;     // m
  uint32_t* sd;      // n: similar-degree counts
  int32_t* parent;   // n: union-find forest over cores (parent < child)
  int32_t* label;    // n: cluster id (roots written by the flatten kernel)
  int32_t* lo;       // n: classify min neighbour label
  int32_t* hi;       // n: classify max neighbour label
  uint8_t* core;     // n
  uint32_t* cnt_u;   // n: undecided edges owned by each vertex (kFlagUDown entries)
  uint64_t* work_u;  // n: sum of the short-row lengths of those edges
  // m: owner b's undecided edges at [rb[b], rb[b] + cnt_u[b]) as (entry,
  // its reverse entry, row start of a, d(a))
  uint4* uedge;
  // ucap work units (begin, end in uedge, the owner's row begin and end):
  // small tier from the front, workgroup tier from the back
  uint4* units;
  // n: ids of the tiny owners (cnt[kCntTiny] of them).  Shares label's
  // memory, which is free until the core pass writes it.
  uint32_t* tiny;
  // Pruned core check, until the core pass: similar (ny) and dissimilar (nn)
  // edges seen per vertex, in lo's and hi's memory, and each vertex's
  // state (kVUndecided / kVCore / kVNonCore) in core's.
  uint32_t* ny;
  uint32_t* nn;
  // Packed edge records of out-of-core chips (launch_prep_packed): each
  // owner's first record (n) and its cursor (n).
  uint32_t* rec_start = nullptr;
  uint32_t* rec_cur = nullptr;
  uint32_t ucap;
  uint64_t* cnt;     // kCntWords
};

struct ScanParams {
  double eps;
  int32_t mu;
  // core-check pruning (GPUSCAN++/GPUScan.cu:303): the workgroup tier defers
  // an edge whose endpoints are both decided (core or not) when it starts
  bool prune = false;
  bool count_all = false;  // no filter stage (sgc_dgraph_autotune)
};

// Per-vertex state of the pruned core check, kept in PassBuffers::core until
// the core pass writes the final flags there.
enum : uint8_t { kVUndecided = 0, kVCore = 1, kVNonCore = 2 };

// Carves the arrays of one pass over g from the context's work buffer.
int carve_pass_buffers(sgc_ctx* ctx, const sgc_dgraph* g, PassBuffers* pb);

// Units of both tiers together are bounded by the number of owned undecided
// edges: every edge is owned once and has two entries, so at most m / 2.
inline size_t unit_capacity(uint64_t m) { return (size_t)(m / 2) + 2; }

// Status for a pass whose planner found more owned undecided entries than
// unit_capacity (counters as read back from the device): an input in which
// some entry has no reverse entry.  SGC_OK otherwise.
int check_unit_overflow(const uint64_t* cnt_host, uint64_t m);

// Device memory of the context's device, or null.  Where there is not enough,
// the context gives back what it can do without, if that makes room: spare
// memory, work memory beyond a pass's, then its graphs' compact row copies.
// Called with nothing of the work buffer in use.
void* device_alloc(sgc_ctx* ctx, size_t bytes);
// Frees g's compact row copies, or (keep) leaves their memory to its context.
void drop_packed(sgc_dgraph* g, bool keep = false);
// The context's work buffer grown to at least `bytes`, or null when the
// device has not that much (the buffer then has the size it had).
void* work_memory(sgc_ctx* ctx, size_t bytes);
// At least `bytes` of page-locked host memory, the context's until
// release_host_work; null when the system will not lock that much.
void* host_work_memory(sgc_ctx* ctx, size_t bytes);
// Gives that memory back if it is more than a context keeps.
void release_host_work(sgc_ctx* ctx);
// Copies between host memory and the device on the context stream.  Pageable
// memory goes through the context's page-locked staging, chunk by chunk, the
// host's share of one chunk overlapping the transfer of the others.  A
// pageable source or destination is done with on return; a page-locked one
// when the stream is.
hipError_t upload_bytes(sgc_ctx* ctx, void* dst, const void* src, size_t bytes, bool src_pinned);
struct HostCopy {
  void* dst;
  const void* src;
  size_t bytes;
};
// Device to host; every copy is done on return.
hipError_t download(sgc_ctx* ctx, const HostCopy* copies, int count);

// Uploads g; `scans`: also builds what only one-shot passes read (the packed
// rows of the filter stage).
int upload_graph(sgc_ctx* ctx, const sgc_host_graph* g, bool scans, sgc_dgraph** out);

// Kernel launchers (kernels.hip, similarity.hip, filter.hip).  All run on `s` and never
// synchronise.
// src[k] = base + the row of entry k, for n rows that start at rp[0 .. n]
void launch_fill_rows(const uint32_t* rp, uint32_t n, uint32_t m, uint32_t base, uint32_t* src, hipStream_t s);
// Fills g->ndeg and g->mirror (after g->src), whichever are there.  Entries
// without a reverse entry get mirror word 0xFFFFFFFF.  Works in the context's
// work buffer; without its memory the reverse entries are searched one by
// one.  May synchronise the stream.  index_work_bytes: what it takes of the
// buffer at most.
hipError_t build_indexes(sgc_ctx* ctx, const sgc_dgraph* g);
size_t index_work_bytes(const sgc_dgraph* g);
// 2^20-id windows of the large-tier bitmap covering n ids, and the kernel
// filling g->woff (see sgc_dgraph).
uint32_t window_count(uint32_t n);
// Bytes of the window-offset index a resident graph of n vertices and m
// entries keeps: n * (W + 1) words when there is more than one window and
// that is at most max(16 m, 1 GiB) bytes (four times the adjacency); else 0.
uint64_t window_index_bytes(uint64_t n, uint64_t m);
void launch_window_offsets(const sgc_dgraph* g, hipStream_t s);
// Bytes of the compact row copies (filter.hip) of m entries, and the kernels
// that write them, after the reverse-entry and neighbour-degree indexes;
// they use the context's work buffer and leave g without the copies when its
// memory is not there.
size_t packed_bytes(uint64_t m);
hipError_t build_packed_rows(sgc_ctx* ctx, sgc_dgraph* g);
// Whether a pass runs the filter stage: its plan then comes from
// launch_plan_filter, and launch_filter leaves the survivors as the exact
// kernels' units.
bool filter_stage(const sgc_dgraph* g, ScanParams p);
void launch_plan_filter(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s);
void launch_filter(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s);
// Whether launch_filter can leave units to the exact kernels.
bool filter_leaves_units(const sgc_dgraph* g);
// Exact units by teams (exact.hip): whether it takes the small or large units
// of a graph of n vertices, and the kernel.
bool exact_units_cover(uint32_t n, bool large);
void launch_exact_units(const sgc_dgraph* g, const PassBuffers& b, const uint4* units, uint32_t ucap, ScanParams p,
                        int cu_count, hipStream_t s, bool large, uint32_t* cn_out);
void launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t s);
void launch_init(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s);
// count_all: every edge is left to its owner (for exact common-neighbour
// counts) instead of the degree-only decision.
// With p.prune, also counts each row's degree-decided similar and dissimilar
// entries (ny, nn).
void launch_prep(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s, bool count_all = false);
// Packed edge records, for chips whose record array holds fewer records than
// the chip has entries: the prep kernel writes flags and per-owner counts,
// every owner gets its place in b.rec_start (and b.rec_cur); then
// launch_similarity_packed decides the owned edges in `rounds` rounds, round
// r taking the owners whose records start in [r w, (r + 1) w), packed into
// b.uedge (which must hold w plus the largest owned count); rounds past the
// chip's records return at once.
void launch_prep_packed(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s);
void launch_similarity_packed(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, int impl,
                              hipEvent_t mid, hipStream_t s, uint32_t w, uint32_t rounds);
// With p.prune, also sets every vertex's state from those counts.
void launch_plan(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s);
// Second similarity round of a pruned pass (after the union-find pass): the
// deferred edges the cluster and border passes need (core-core edges whose
// roots differ, core-non-core edges) are marked undecided again, planned and
// decided, and the union-find pass repeats.  Every kernel returns at once
// when no deferred edge is needed.
void launch_redo(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s);
// `mid` (optional) is recorded between the workgroup-tier and wave-tier
// kernels.  With cn_out the tiered kernels count every owned edge fully and
// write |N(a) & N(b)| to both of its entries instead of flags.
void launch_similarity(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, int impl, hipEvent_t mid,
                       hipStream_t s, uint32_t* cn_out = nullptr);
void launch_similarity_wave(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s);
void launch_core(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s);
// flatten: launch_flatten's work too (small graphs: a launch less)
void launch_border(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, bool flatten = false);
// Graphs on which a launch costs more than what it saves.
bool small_graph(const sgc_dgraph* g);
void launch_classify(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s);
// The single kernels the four launchers above are made of (edge passes over
// entries [0, g->m), vertex passes over all g->n vertices); the out-of-core
// path runs the edge passes once per chip.
void launch_core_count(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s);
// mu_dev (optional): read mu from device memory instead of p (captured launches)
void launch_core_mark(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s,
                      const int32_t* mu_dev = nullptr);
// gate >= 0: the kernel runs only when the sum `gate` is not 0
void launch_union(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, int gate = -1);
// marks the deferred edges a pruned pass needs after its union-find pass
// (count in cnt[kCntRedo]); needs g->mirror
void launch_redo_mark(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s);
void launch_flatten(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s);
// m_all: entries of the whole graph when g is one of several row chips
void launch_classify_edges(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, uint64_t m_all = 0);
// The pass's end: counters (sums folded) to host_cnt (page-locked, device
// address), and the results to the device addresses given (any may be null);
// after an overflow (kCntOverflow) the results are left alone.
// All that follows the similarity phase, and the pass's end, in one launch:
// graphs of few vertices and entries (tiny_graph), without the core-check
// pruning.
bool tiny_graph(const sgc_dgraph* g);
void launch_tail(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, uint64_t* host_cnt, int32_t* labels,
                 uint8_t* core, uint8_t* sim, hipStream_t s);
void launch_publish(const sgc_dgraph* g, const PassBuffers& b, uint64_t* host_cnt, int32_t* labels, uint8_t* core,
                    uint8_t* sim, hipStream_t s);
void launch_finalize(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s,
                     const int32_t* mu_dev = nullptr);

}  // namespace sgc
