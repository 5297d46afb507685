// SCAN kernels for gfx950 (wave64) after the similarity phase, plus graph
// preparation and the one-wave-per-edge similarity kernel.  Every kernel is a
// grid-stride loop over vertices or directed CSR entries; per-row aggregation
// inside a wave uses a segmented shuffle reduction (entries of one row are
// consecutive lanes) so each row issues at most one atomic per wave.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include <hipcub/device/device_radix_sort.hpp>

#include "device.h"
#include "device_util.h"
#include "scan_phases.h"

namespace sgc {

namespace {

// ---------------------------------------------------------------------------
// Graph preparation
// ---------------------------------------------------------------------------

// The last of rows [lo, hi] that starts at k or before, given that lo does: 64
// pivots to a round.
__device__ __forceinline__ uint32_t wave_row_of(const uint32_t* __restrict__ rp, uint32_t lo, uint32_t hi, uint32_t k) {
  const uint32_t lane = lane_id();
  while (hi - lo >= kWave) {
    const uint64_t w = (uint64_t)hi - lo + 1;
    const uint32_t le = (uint32_t)__popcll(__ballot(rp[lo + (uint32_t)(w * lane / kWave)] <= k));  // at least 1
    const uint32_t at = lo;
    lo = at + (uint32_t)(w * (le - 1) / kWave);
    if (le < kWave) hi = at + (uint32_t)(w * le / kWave) - 1;
  }
  return lo + (uint32_t)__popcll(__ballot(lane <= hi - lo && rp[lo + lane] <= k)) - 1;
}

// src[k] = base + the row of entry k.  A wave takes 1024 entries, finds the
// rows of the first and the last and searches the others between them: stores
// are whole lines and no row is long or short for it.  A wave to a row took
// 256 us on R-MAT-20 (3.1e7 entries) and 59 on R-MAT-18.
constexpr uint32_t kFillTile = 1024;

__global__ void __launch_bounds__(kBlock) k_fill_rows(uint32_t n, uint32_t m, uint32_t base,
                                                      const uint32_t* __restrict__ rp, uint32_t* __restrict__ src) {
  constexpr uint32_t C = 4;
  const uint32_t lane = lane_id();
  const uint64_t step = (uint64_t)gridDim.x * (kBlock / kWave) * kFillTile;
  for (uint64_t t = ((uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave) * kFillTile; t < m; t += step) {
    const uint32_t t0 = (uint32_t)t, len = min(m - t0, kFillTile);
    const uint32_t first = wave_row_of(rp, 0, n - 1, t0), last = wave_row_of(rp, first, n - 1, t0 + len - 1);
    for (uint32_t i = lane; i < len; i += kWave * C) {
      uint32_t lo[C], hi[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) lo[j] = first, hi[j] = last;
      for (uint32_t left = last - first; left; left >>= 1) {
#pragma unroll
        for (uint32_t j = 0; j < C; ++j) {
          const uint32_t mid = lo[j] + ((hi[j] - lo[j] + 1) >> 1);
          if (rp[mid] <= t0 + min(i + j * kWave, len - 1))
            lo[j] = mid;
          else
            hi[j] = mid - 1;  // above lo: mid = lo only when lo = hi, and then rp[lo] <= k
        }
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j)
        if (i + j * kWave < len) src[t0 + i + j * kWave] = base + lo[j];
    }
  }
}

// mirror[k] = position of the reverse entry (v, u) of entry k = (u, v).  Of
// the two entries of an edge only the one whose neighbour row is the shorter,
// (d(v), v) <= (d(u), u), searches: a binary search of u in the sorted row of
// v, which writes both mirror[k] and mirror[p].  A pair is found only from
// entry k, so each word has one writer.  Entries whose reverse entry is
// missing (asymmetric input) get 0xFFFFFFFF.  Four searches per thread run
// in lockstep so that their loads overlap; each halves its window only down
// to eight entries and reads those with eight independent loads, which ends
// the searches in short rows (most rows) after one round trip.
__global__ void __launch_bounds__(kBlock) k_mirror(uint32_t m, const uint32_t* __restrict__ rp,
                                                   const uint32_t* __restrict__ src, const int32_t* __restrict__ adj,
                                                   uint32_t* __restrict__ mirror) {
  constexpr uint32_t C = 4;  // searches per thread
  constexpr uint32_t W = 7;  // windows [lo, hi] of at most W + 1 entries end in one round of loads
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k0 = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k0 < m; k0 += stride * C) {
    // lower bound of key in [lo, end): it lies in [lo, hi], and entries from
    // hi on are >= key
    uint32_t lo[C], hi[C], end[C];
    int32_t key[C];
    bool on[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      const uint64_t k = k0 + j * stride;
      lo[j] = hi[j] = end[j] = 0;
      key[j] = 0;
      on[j] = false;
      if (k < m) {
        const uint32_t v = (uint32_t)adj[k], u = src[k];
        const uint32_t vb = rp[v], ve = rp[v + 1], du = rp[u + 1] - rp[u], dv = ve - vb;
        key[j] = (int32_t)u;
        on[j] = dv < du || (dv == du && v <= u);
        if (on[j]) {
          lo[j] = vb;
          hi[j] = end[j] = ve;
        }
      }
    }
    // halve the windows longer than W, all searches in lockstep
    for (;;) {
      bool any = false;
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) any |= hi[j] - lo[j] > W;
      if (!any) break;
      int32_t val[C];
      uint32_t mid[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        mid[j] = lo[j] + ((hi[j] - lo[j]) >> 1);
        val[j] = hi[j] - lo[j] > W ? adj[mid[j]] : 0;
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j)
        if (hi[j] - lo[j] > W) {
          if (val[j] < key[j])
            lo[j] = mid[j] + 1;
          else
            hi[j] = mid[j];
        }
    }
    // the last window [lo, hi] (clipped to the row) in one round of loads:
    // the key's position is lo + (entries below it)
    int32_t val[C][W + 1];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j)
#pragma unroll
      for (uint32_t t = 0; t <= W; ++t)
        val[j][t] = on[j] && lo[j] + t <= hi[j] && lo[j] + t < end[j] ? adj[lo[j] + t] : 0x7FFFFFFF;
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      if (!on[j]) continue;
      uint32_t below = 0;
      bool found = false;
#pragma unroll
      for (uint32_t t = 0; t <= W; ++t) {
        below += val[j][t] < key[j];
        found |= val[j][t] == key[j];
      }
      const uint32_t k = (uint32_t)(k0 + j * stride), p = lo[j] + below;
      mirror[k] = found ? p : 0xFFFFFFFFu;
      if (found) mirror[p] = k;
    }
  }
}

// The reverse-entry index by sorting.  In a symmetric CSR with sorted rows,
// the entries stably sorted by neighbour id come in the order of their
// reverse entries: row v lists its neighbours u ascending, and the entries
// (u, v) ordered by v, then by position (so by u), are ordered the same way.
// So the entry (u, v) at k that the sort puts at j has its reverse at j
// exactly when entry j is (v, u), and then entry j's reverse is k: the index
// is written at j, in order, not scattered.  Each pair is checked, and an
// input where some is not falls back to the search (k_mirror).  The sort's
// values carry the entry's row beside its position, so the check reads no
// other row.
__global__ void __launch_bounds__(kBlock) k_rows_and_positions(uint32_t m, const uint32_t* __restrict__ src,
                                                               uint64_t* __restrict__ vals) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < m; k += stride)
    vals[k] = ((uint64_t)src[k] << 32) | k;
}

__global__ void __launch_bounds__(kBlock) k_mirror_from_sorted(uint32_t m, const uint32_t* __restrict__ src,
                                                               const int32_t* __restrict__ adj,
                                                               const uint32_t* __restrict__ keys,
                                                               const uint64_t* __restrict__ vals,
                                                               uint32_t* __restrict__ mirror,
                                                               unsigned long long* __restrict__ bad) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  unsigned long long miss = 0;
  for (uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x; j < m; j += stride) {
    const uint64_t val = vals[j];
    const uint32_t k = (uint32_t)val, u = (uint32_t)(val >> 32), v = keys[j];
    const bool ok = src[j] == v && (uint32_t)adj[j] == u;
    mirror[j] = ok ? k : 0xFFFFFFFFu;
    miss += ok ? 0u : 1u;
  }
  block_atomic_add(bad, miss);
}

// The reverse-entry index of mid-size graphs by splitting: the searches of
// k_mirror whose rows start in the same 2^15 entries of the adjacency meet in
// one bucket, whose rows then lie in LDS.  k_split_searches writes one item a
// search, (entry, its row, where its neighbour's row starts in the bucket and
// its length), in runs of a tile's items for a bucket, and the neighbour
// degrees on the way; k_bucket_searches finds and writes.  Searches in rows
// over kBucketRow, and those a bucket has no room for (input whose entries
// lack their reverse), are done on the spot.  Bound by the item and index
// traffic, about 40 bytes an entry: R-MAT-20 (3.1e7 entries) 0.64 ms with the
// neighbour degrees, 1.44 by the sort; R-MAT-22 2.9 and 4.8.
constexpr uint32_t kBucketBits = 15, kBucketRow = 4096;
constexpr uint32_t kBucketCap = (1u << kBucketBits) + kBucketRow;  // a bucket's rows hold no more
constexpr uint32_t kBuckets = 4096;
constexpr uint32_t kSplitEntries = kBuckets << kBucketBits;  // largest graph

// The position of x in the sorted row a[lo, hi), or 0xFFFFFFFF.
__device__ __forceinline__ uint32_t find_in_row(const int32_t* a, uint32_t lo, uint32_t hi, int32_t x) {
  const uint32_t end = hi;
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (a[mid] < x)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo < end && a[lo] == x ? lo : 0xFFFFFFFFu;
}

struct SplitItem {
  uint32_t k, u, row;  // row: its start in the bucket, length << kBucketBits
};

__global__ void __launch_bounds__(1024) k_split_searches(uint32_t m, const uint32_t* __restrict__ rp,
                                                         const uint32_t* __restrict__ src,
                                                         const int32_t* __restrict__ adj, uint32_t* __restrict__ ndeg,
                                                         uint32_t* __restrict__ mirror, uint32_t* __restrict__ cursor,
                                                         SplitItem* __restrict__ items, uint32_t buckets) {
  constexpr uint32_t T = 1024, C = 16;
  __shared__ uint32_t s_count[kBuckets], s_base[kBuckets];
  const uint32_t tid = threadIdx.x;
  for (uint32_t b = tid; b < buckets; b += T) s_count[b] = 0;
  __syncthreads();
  for (uint64_t t0 = (uint64_t)blockIdx.x * T * C; t0 < m; t0 += (uint64_t)gridDim.x * T * C) {  // block-uniform
    uint32_t u[C], start[C], len[C], at[C];  // len 0: no search; at: its place among the tile's items of its bucket
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      const uint64_t k = t0 + j * T + tid;
      u[j] = k < m ? src[k] : 0u;
      at[j] = k < m ? (uint32_t)adj[k] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      const uint64_t k = t0 + j * T + tid;
      const uint32_t v = at[j], du = rp[u[j] + 1] - rp[u[j]];
      start[j] = rp[v];
      const uint32_t dv = rp[v + 1] - start[j];
      if (k < m) ndeg[k] = dv;
      len[j] = k < m && (dv < du || (dv == du && v <= u[j])) ? dv : 0u;
      if (len[j] > kBucketRow) {
        const uint32_t p = find_in_row(adj, start[j], start[j] + dv, (int32_t)u[j]);
        if (p != 0xFFFFFFFFu) {
          mirror[k] = p;
          mirror[p] = (uint32_t)k;
        }
        len[j] = 0;
      }
      if (len[j]) at[j] = atomicAdd(&s_count[start[j] >> kBucketBits], 1u);
    }
    __syncthreads();
    for (uint32_t b = tid; b < buckets; b += T) {
      const uint32_t c = s_count[b];
      if (c) s_base[b] = atomicAdd(&cursor[b], c);
      s_count[b] = 0;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      if (!len[j]) continue;
      const uint32_t k = (uint32_t)(t0 + j * T + tid), b = start[j] >> kBucketBits, i = s_base[b] + at[j];
      if (i < kBucketCap) {
        items[(uint64_t)b * kBucketCap + i] =
            SplitItem{k, u[j], (start[j] & ((1u << kBucketBits) - 1)) | len[j] << kBucketBits};
      } else {
        const uint32_t p = find_in_row(adj, start[j], start[j] + len[j], (int32_t)u[j]);
        if (p != 0xFFFFFFFFu) {
          mirror[k] = p;
          mirror[p] = k;
        }
      }
    }
    __syncthreads();  // s_base is rewritten
  }
}

// Block b: bucket b.
__global__ void __launch_bounds__(1024) k_bucket_searches(uint32_t m, const int32_t* __restrict__ adj,
                                                          const uint32_t* __restrict__ cursor,
                                                          const SplitItem* __restrict__ items,
                                                          uint32_t* __restrict__ mirror) {
  constexpr uint32_t T = 1024, C = 4;
  __shared__ __align__(16) int32_t rows[kBucketCap];
  const uint32_t b0 = blockIdx.x << kBucketBits, span = min(m - b0, kBucketCap), tid = threadIdx.x;
  const uint32_t count = min(cursor[blockIdx.x], kBucketCap);
  if (!count) return;
  for (uint32_t t = tid * 4; t < span / 4 * 4; t += T * 4)
    *reinterpret_cast<int4*>(rows + t) = *reinterpret_cast<const int4*>(adj + b0 + t);
  if (tid < span % 4) rows[span / 4 * 4 + tid] = adj[b0 + span / 4 * 4 + tid];
  __syncthreads();
  const SplitItem* const it = items + (uint64_t)blockIdx.x * kBucketCap;
  for (uint32_t i0 = tid; i0 < count; i0 += T * C) {
    SplitItem q[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) q[j] = it[min(i0 + j * T, count - 1)];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      if (i0 + j * T >= count) break;
      const uint32_t lo = q[j].row & ((1u << kBucketBits) - 1);
      const uint32_t p = find_in_row(rows, lo, lo + (q[j].row >> kBucketBits), (int32_t)q[j].u);
      if (p != 0xFFFFFFFFu) {
        mirror[q[j].k] = b0 + p;
        mirror[b0 + p] = q[j].k;
      }
    }
  }
}

// ndeg[k] = d(adj[k]), so the prep kernel streams the neighbour degrees
// instead of gathering two row offsets per entry on every pass.
__global__ void __launch_bounds__(kBlock) k_neighbor_degrees(uint32_t m, const uint32_t* __restrict__ rp,
                                                             const int32_t* __restrict__ adj,
                                                             uint32_t* __restrict__ ndeg) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < m; k += stride) {
    const uint32_t v = (uint32_t)adj[k];
    ndeg[k] = rp[v + 1] - rp[v];
  }
}

// ---------------------------------------------------------------------------
// Per-pass initialisation
// ---------------------------------------------------------------------------

// lo / hi hold the pruned core check's similar / dissimilar counts and core
// its vertex states until the core pass (k_core_mark) gives them their
// final meaning.
__global__ void __launch_bounds__(kBlock) k_init(uint32_t n, uint32_t* __restrict__ sd, int32_t* __restrict__ lo,
                                                 int32_t* __restrict__ hi, uint8_t* __restrict__ core,
                                                 uint32_t* __restrict__ cnt_u,
                                                 uint64_t* __restrict__ work_u, uint64_t* __restrict__ cnt) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride) {
    sd[x] = 0;
    lo[x] = 0;
    hi[x] = 0;
    core[x] = kVUndecided;
    cnt_u[x] = 0;
    work_u[x] = 0;
  }
  if (blockIdx.x == 0) {
    for (uint32_t t = threadIdx.x; t < kCntWords; t += kBlock) cnt[t] = 0;
    __syncthreads();
    stamp(cnt, kStampInit);
  }
}

// ---------------------------------------------------------------------------
// Similarity, one wave per undecided edge (GPUSCAN++/GPUScan.cu:174-222)
// ---------------------------------------------------------------------------

// Dense list of the owned undecided entries (kFlagUDown), in any order, for
// the one-wave-per-edge kernel: 16 consecutive entries per thread, one
// append per block iteration.
__global__ void __launch_bounds__(kBlock) k_list_owned(uint32_t m, const uint8_t* __restrict__ flag,
                                                       uint32_t* __restrict__ list, uint64_t* __restrict__ cnt) {
  stamp(cnt, kStampSim);
  constexpr uint32_t E = 16;
  unsigned long long* const ctr[1] = {(unsigned long long*)&cnt[kCntDense]};
  const uint64_t tile = (uint64_t)kBlock * E;
  for (uint64_t base = (uint64_t)blockIdx.x * tile; base < m; base += (uint64_t)gridDim.x * tile) {  // block-uniform
    const uint64_t k0 = base + (uint64_t)threadIdx.x * E;
    uint32_t sel = 0;
#pragma unroll
    for (uint32_t j = 0; j < E; ++j)
      if (k0 + j < m && flag[k0 + j] == kFlagUDown) sel |= 1u << j;
    uint32_t pos[1] = {(uint32_t)__popc(sel)};
    block_reserve<1>(pos, ctr);
    for (uint32_t j = 0; j < E; ++j)
      if ((sel >> j) & 1u) list[pos[0]++] = (uint32_t)(k0 + j);
  }
}

// One wave per undecided edge (a, b), s = d(a) <= l = d(b): lanes take the
// short row 64 elements at a time and binary-search each in the long row,
// keeping a per-lane lower bound (each lane's keys increase).  The count is
// checked against the exact threshold after every 64 elements: reached ->
// similar, unreachable -> not similar.  Writes the flag of both directed
// entries.  Kept beside the tiered kernels as an independent second
// implementation (selectable per context).
__global__ void __launch_bounds__(kBlock) k_similarity_wave(const uint32_t* __restrict__ rb,
                                                            const uint32_t* __restrict__ re,
                                                            const int32_t* __restrict__ adj,
                                                            const uint32_t* __restrict__ src, double eps,
                                                            uint8_t* __restrict__ flag,
                                                            const uint32_t* __restrict__ list,
                                                            uint64_t* __restrict__ cnt) {
  const uint32_t lane = lane_id();
  const uint64_t nU = cnt[kCntDense];
  const uint64_t waves = (uint64_t)gridDim.x * (kBlock / kWave);
  uint64_t probes = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; i < nU; i += waves) {
    const uint32_t k = list[i];
    const uint32_t b = src[k];
    const uint32_t a = (uint32_t)adj[k];
    const uint32_t ab = rb[a], ae = re[a], bb = rb[b], be = re[b];
    const uint32_t s = ae - ab, l = be - bb;
    const double rhs = predicate_rhs(eps, s, l);
    const bool thresholded = s <= kMaxThresholdRow;
    const uint32_t cstar = thresholded ? min_common_threshold(rhs, s) : 0u;
    uint32_t cn = 0;
    uint32_t lo = bb;
    uint32_t off = 0;
    bool decided = false, sim = false;
    if (thresholded && cstar == 0) {
      decided = true;
      sim = true;
    } else if (thresholded && cstar > s) {
      decided = true;
      sim = false;
    }
    while (!decided && off < s) {
      bool hit = false;
      if (off + lane < s) {
        const int32_t x = adj[ab + off + lane];
        uint32_t h = be;
        while (lo < h) {
          const uint32_t mid = (lo + h) >> 1;
          if (adj[mid] < x)
            lo = mid + 1;
          else
            h = mid;
        }
        hit = lo < be && adj[lo] == x;
      }
      cn += (uint32_t)__popcll(__ballot(hit));
      off += kWave;
      if (thresholded) {
        const uint32_t rest = off < s ? s - off : 0u;
        if (cn >= cstar) {
          decided = true;
          sim = true;
        } else if (cn + rest < cstar) {
          decided = true;
          sim = false;
        }
      }
    }
    probes += off < s ? off : s;
    if (!decided) sim = thresholded ? cn >= cstar : predicate_exact(cn, rhs);
    const uint32_t mpos = wave_lower_bound(adj, ab, ae, (int32_t)b);
    if (lane == 0) {
      const uint8_t f = sim ? kFlagY : kFlagN;
      flag[k] = f;
      if (mpos < ae && adj[mpos] == (int32_t)b) flag[mpos] = f;
    }
  }
  count_add<1>(cnt, {kCntProbes}, {lane == 0 ? probes : 0ull});
}

// ---------------------------------------------------------------------------
// Core check (GPUSCAN++/GPUScan.cu:115-131, :276-367)
// ---------------------------------------------------------------------------

// Similar entries per row, from the flags' similar entries alone: one
// atomic per run of a row's entries in a wave's 64.
template <uint32_t TILE>
__global__ void __launch_bounds__(kBlock) k_core_count(uint64_t m, const uint32_t* __restrict__ src,
                                                       const uint8_t* __restrict__ flag, uint32_t* __restrict__ sd,
                                                       uint64_t* __restrict__ cnt) {
  stamp(cnt, kStampCore);
  __shared__ uint16_t s_at[kBlock / kWave][TILE];
  const uint32_t wv = threadIdx.x / kWave;
  PhaseView v{};
  v.m = (uint32_t)m, v.src = src, v.flag = flag, v.sd = sd;
  const uint64_t step = (uint64_t)gridDim.x * (kBlock / kWave) * TILE;
  for (uint64_t base = ((uint64_t)blockIdx.x * (kBlock / kWave) + wv) * TILE; base < m; base += step)
    core_count_tile<TILE>(v, base, s_at[wv]);
}

// core(x) <=> #similar neighbours >= mu (mu <= 0: >= 1).  The reference's
// sd/ed state machine reaches exactly this fixed point: sd only counts
// similar edges, ed only discounts dissimilar ones, and every edge of a
// still-undecided vertex is evaluated.
// mu comes from mu_dev when given (parameters of a captured launch), else mu.
// Also adds the entries of the core rows to kCntLabeled when the row
// offsets are given (rb null: views without them count nothing here).
__global__ void __launch_bounds__(kBlock) k_core_mark(uint32_t n, const uint32_t* __restrict__ sd, int32_t mu,
                                                      const int32_t* __restrict__ mu_dev,
                                                      const uint32_t* __restrict__ rb,
                                                      const uint32_t* __restrict__ re, uint8_t* __restrict__ core,
                                                      int32_t* __restrict__ parent, int32_t* __restrict__ label,
                                                      int32_t* __restrict__ lo, int32_t* __restrict__ hi,
                                                      uint64_t* __restrict__ cnt) {
  if (mu_dev) mu = *mu_dev;
  PhaseView v{};
  v.n = n;
  v.sd = const_cast<uint32_t*>(sd);
  v.rb = rb, v.re = re, v.core = core, v.parent = parent, v.label = label, v.lo = lo, v.hi = hi;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  uint64_t labeled = 0, marked = 0;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride) {
    uint32_t mk;
    labeled += core_mark_vertex(v, (uint32_t)x, mu, &mk);
    marked += mk;
  }
  count_add<2>(cnt, {kCntLabeled, kCntMarked}, {labeled, marked});
}

// ---------------------------------------------------------------------------
// Clusters: lock-free union-find, parents always smaller than children
// (GPUSCAN++/GPUScan.cu:465-528, :632-652; scan_phases.h)
// ---------------------------------------------------------------------------

// Two rounds over the similar core-core edges, each visited from its larger
// endpoint: the first joins one edge per run of a row's entries (HEADS), then
// k_compress points every core at its root, and the second joins what is
// left; by then nearly every edge's endpoints have the same parent, which two
// plain loads show (a parent read from a stale cache line is still an
// ancestor).  Joining every edge at once met in long chains and contended
// swaps: on planted communities (n = 3e5, 3.6e6 similar edges, 64k cores)
// 0.97 ms, 0.26 in two rounds.
// gate >= 0: runs only when the sum `gate` is not 0 (the union-find pass
// repeated after the second similarity round of a pruned pass).
constexpr uint64_t kFewCores = 1024;  // up to here the first round costs more than it saves

template <bool HEADS, uint32_t TILE>
__global__ void __launch_bounds__(kBlock) k_union(uint64_t m, const uint32_t* __restrict__ src,
                                                  const int32_t* __restrict__ adj, const uint8_t* __restrict__ flag,
                                                  const uint8_t* __restrict__ core, int32_t* parent,
                                                  uint64_t* __restrict__ cnt, int gate) {
  stamp(cnt, kStampCluster);
  const uint64_t cores = count_total(cnt, kCntMarked);
  if (cores == 0) return;  // no core-core edge to join
  if (HEADS && cores <= kFewCores) return;
  if (gate >= 0 && !count_any(cnt, gate)) return;
  __shared__ uint16_t s_at[kBlock / kWave][TILE];
  const uint32_t wv = threadIdx.x / kWave;
  PhaseView v{};
  v.m = (uint32_t)m, v.src = src, v.adj = adj, v.flag = flag, v.core = const_cast<uint8_t*>(core), v.parent = parent;
  const uint64_t step = (uint64_t)gridDim.x * (kBlock / kWave) * TILE;
  for (uint64_t base = ((uint64_t)blockIdx.x * (kBlock / kWave) + wv) * TILE; base < m; base += step)
    union_tile<HEADS, TILE>(v, base, s_at[wv]);
}

__global__ void __launch_bounds__(kBlock) k_compress(uint32_t n, const uint8_t* __restrict__ core, int32_t* parent,
                                                     const uint64_t* __restrict__ cnt) {
  if (count_total(cnt, kCntMarked) <= kFewCores) return;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride)
    if (core[x]) st_coherent(parent + x, uf_find(parent, (int32_t)x));
}

__global__ void __launch_bounds__(kBlock) k_flatten(uint32_t n, const uint8_t* __restrict__ core, int32_t* parent,
                                                    int32_t* __restrict__ label) {
  PhaseView v{};
  v.n = n, v.core = const_cast<uint8_t*>(core), v.parent = parent, v.label = label;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride) flatten_vertex(v, (uint32_t)x);
}

// Deferred edges of a pruned pass that the later passes need, after the
// union-find pass over the known similar core-core edges: a core-core edge
// whose endpoints are still in different trees (GPUSCAN++/GPUScan.cu:
// 557-585 computes these on demand) and a core-non-core edge (a border
// candidate, :692-719).  They are marked undecided again (owner side
// kFlagUDown, the other kFlagUUp) for a second similarity round and counted
// in kCntRedo.  A non-core-non-core edge is never needed: classify
// reads labels only.  Edges deferred with both endpoints in one tree cannot
// join anything.
__global__ void __launch_bounds__(kBlock) k_redo_mark(uint32_t m, const uint32_t* __restrict__ src,
                                                      const int32_t* __restrict__ adj,
                                                      const uint32_t* __restrict__ mirror, uint8_t* flag,
                                                      const uint8_t* __restrict__ core, int32_t* parent,
                                                      uint64_t* __restrict__ cnt) {
  if (!count_any(cnt, kCntMarked) || !count_any(cnt, kCntDeferred)) return;
  constexpr uint32_t C = kEdgeChunks;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  uint32_t redo = 0;
  for (uint64_t k0 = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k0 < m; k0 += stride * C) {
    bool d[C];
    uint32_t b[C], a[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      const uint64_t k = k0 + j * stride;
      d[j] = k < m && flag[k] == kFlagDeferDown;
      b[j] = d[j] ? src[k] : 0u;
      a[j] = d[j] ? (uint32_t)adj[k] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      if (!d[j]) continue;
      const bool ca = core[a[j]], cb = core[b[j]];
      const bool need =
          ca && cb ? uf_find(parent, (int32_t)a[j]) != uf_find(parent, (int32_t)b[j]) : ca != cb;
      if (!need) continue;
      const uint64_t k = k0 + j * stride;
      flag[k] = kFlagUDown;
      const uint32_t mk = mirror[k];  // 0xFFFFFFFF: no reverse entry (asymmetric input)
      if (mk < m) flag[mk] = kFlagUUp;
      ++redo;
    }
  }
  count_add<1>(cnt, {kCntRedo}, {redo});
}

// ---------------------------------------------------------------------------
// Borders (GPUSCAN++/GPUScan.cu:654-730): minimum candidate cluster id
// ---------------------------------------------------------------------------

template <bool FLATTEN, uint32_t TILE>
__global__ void __launch_bounds__(kBlock) k_border(uint32_t n, uint64_t m, int32_t* parent,
                                                   const uint32_t* __restrict__ src,
                                                   const int32_t* __restrict__ adj, const uint8_t* __restrict__ flag,
                                                   const uint8_t* __restrict__ core, const uint32_t* __restrict__ rb,
                                                   const uint32_t* __restrict__ re, int32_t* label,
                                                   uint64_t* __restrict__ cnt) {
  stamp(cnt, kStampBorder);
  if (!count_any(cnt, kCntMarked)) return;  // no core: no border
  // FLATTEN: cluster ids of the cores too (roots go to label, as k_flatten
  // does for larger graphs); the edges below then find a core's root themselves
  if (FLATTEN) {
    PhaseView f{};
    f.core = const_cast<uint8_t*>(core), f.parent = parent, f.label = label;
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride) flatten_vertex(f, (uint32_t)x);
  }
  __shared__ uint16_t s_at[kBlock / kWave][TILE];
  PhaseView v{};
  v.m = (uint32_t)m, v.src = src, v.adj = adj, v.flag = flag, v.core = const_cast<uint8_t*>(core);
  v.rb = rb, v.re = re, v.label = label, v.parent = parent;
  const uint32_t wv = threadIdx.x / kWave;
  const uint64_t step = (uint64_t)gridDim.x * (kBlock / kWave) * TILE;
  // entries of the border rows this lane labels first; the core rows'
  // entries were counted by k_core_mark
  uint64_t labeled = 0;
  for (uint64_t base = ((uint64_t)blockIdx.x * (kBlock / kWave) + wv) * TILE; base < m; base += step)
    labeled += border_tile<FLATTEN, TILE>(v, base, s_at[wv]);
  count_add<1>(cnt, {kCntLabeled}, {labeled});
}

// ---------------------------------------------------------------------------
// Hubs and outliers (GPUSCAN++/GPUScan.cu:732-798)
// ---------------------------------------------------------------------------

// The side of the classify pass, the same for every launch over the graph's
// m_all entries (maybe in several row chips): from the labelled rows when
// they hold fewer than a third of the entries.
__device__ __forceinline__ bool classify_from_labeled(const uint64_t* cnt, uint64_t m_all) {
  return 3 * count_total(cnt, kCntLabeled) < m_all;
}

// listed: the labelled side is left to k_classify_rows.
__global__ void __launch_bounds__(kBlock) k_classify(uint32_t m, uint64_t m_all, const uint32_t* __restrict__ src,
                                                     const int32_t* __restrict__ adj,
                                                     const int32_t* __restrict__ label, int32_t* __restrict__ lo,
                                                     int32_t* __restrict__ hi, uint64_t* __restrict__ cnt,
                                                     bool listed) {
  stamp(cnt, kStampClassify);
  // no core means no label anywhere: lo and hi keep their initial values
  if (!count_any(cnt, kCntMarked)) return;
  PhaseView v{};
  v.m = m, v.src = src, v.adj = adj, v.label = const_cast<int32_t*>(label), v.lo = lo, v.hi = hi;
  const bool from_labeled = classify_from_labeled(cnt, m_all);
  if (from_labeled && listed) return;
  const uint64_t waves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t base = ((uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave) * (kWave * kEdgeChunks);
       base < m; base += waves * kWave * kEdgeChunks)
    classify_chunk(v, base, from_labeled);
}

// The labelled side without a walk over all entries: the labelled rows in
// pieces of kRowPiece entries, listed, then one wave per piece.  At most one
// piece per labelled row and one per kRowPiece entries: under m of them.
// R-MAT-24 with 304 cores: 1.45 ms for the walk, 0.73 listed.
constexpr uint32_t kRowPiece = 1024;

__global__ void __launch_bounds__(kBlock) k_label_pieces(uint32_t n, uint64_t m, const uint32_t* __restrict__ rb,
                                                         const uint32_t* __restrict__ re,
                                                         const int32_t* __restrict__ label, uint2* __restrict__ piece,
                                                         uint64_t* __restrict__ cnt) {
  stamp(cnt, kStampClassify);
  if (!count_any(cnt, kCntMarked) || !classify_from_labeled(cnt, m)) return;
  constexpr uint32_t V = 8;
  unsigned long long* const ctr[1] = {(unsigned long long*)&cnt[kCntPieces]};
  const uint64_t tile = (uint64_t)kBlock * V;
  for (uint64_t base = (uint64_t)blockIdx.x * tile; base < n; base += (uint64_t)gridDim.x * tile) {  // block-uniform
    uint32_t len[V], need[1] = {0};
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint64_t x = base + j * kBlock + threadIdx.x;
      len[j] = x < n && label[x] != kNoLabel ? re[x] - rb[x] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) need[0] += (len[j] + kRowPiece - 1) / kRowPiece;
    if (!__syncthreads_or(need[0] != 0)) continue;
    block_reserve<1>(need, ctr);
#pragma unroll
    for (uint32_t j = 0; j < V; ++j)
      for (uint32_t at = 0; at < len[j]; at += kRowPiece)
        piece[need[0]++] = make_uint2((uint32_t)(base + j * kBlock + threadIdx.x), at);
  }
}

__global__ void __launch_bounds__(kBlock) k_classify_rows(const uint32_t* __restrict__ rb,
                                                          const uint32_t* __restrict__ re,
                                                          const int32_t* __restrict__ adj,
                                                          const int32_t* __restrict__ label, int32_t* lo, int32_t* hi,
                                                          const uint2* __restrict__ piece,
                                                          const uint64_t* __restrict__ cnt) {
  const uint64_t count = cnt[kCntPieces];  // 0 when the other side is taken
  const uint64_t waves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t i = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; i < count; i += waves) {
    const uint2 p = piece[i];
    const uint32_t b = rb[p.x] + p.y, len = min(re[p.x] - b, kRowPiece);
    const int32_t l = label[p.x];
    for (uint32_t t0 = lane_id(); t0 < len; t0 += kWave * kEdgeChunks) {
      int32_t nb[kEdgeChunks];
      bool to[kEdgeChunks];
#pragma unroll
      for (uint32_t j = 0; j < kEdgeChunks; ++j) {
        to[j] = t0 + j * kWave < len;
        nb[j] = to[j] ? adj[b + t0 + j * kWave] : 0;
      }
#pragma unroll
      for (uint32_t j = 0; j < kEdgeChunks; ++j) to[j] = to[j] && label[nb[j]] == kNoLabel;
      // a bound that is there already needs no atomic (a stale one is looser)
#pragma unroll
      for (uint32_t j = 0; j < kEdgeChunks; ++j)
        if (to[j]) {
          if (l < lo[nb[j]]) atomicMin(&lo[nb[j]], l);
          if (l > hi[nb[j]]) atomicMax(&hi[nb[j]], l);
        }
    }
  }
}

// Also counts the similar entries: sd[x] holds those of row x.
__global__ void __launch_bounds__(kBlock) k_finalize(uint32_t n, int32_t mu, const int32_t* __restrict__ mu_dev,
                                                     const uint32_t* __restrict__ sd, const int32_t* __restrict__ lo,
                                                     const int32_t* __restrict__ hi, const uint8_t* __restrict__ core,
                                                     int32_t* __restrict__ label, uint64_t* __restrict__ cnt) {
  if (mu_dev) mu = *mu_dev;
  PhaseView v{};
  v.n = n, v.sd = const_cast<uint32_t*>(sd), v.lo = const_cast<int32_t*>(lo), v.hi = const_cast<int32_t*>(hi);
  v.core = const_cast<uint8_t*>(core), v.label = label;
  RoleCounts rc;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride)
    finalize_vertex(v, (uint32_t)x, mu, &rc);
  count_roles(cnt, rc);
}

// Copies `bytes` bytes by the whole grid: 16 at a time where both ends allow
// it.
__device__ __forceinline__ void grid_copy(const void* __restrict__ from, void* __restrict__ to, uint64_t bytes) {
  const uint64_t at = (uint64_t)blockIdx.x * kBlock + threadIdx.x, stride = (uint64_t)gridDim.x * kBlock;
  uint64_t done = 0;
  if ((((uintptr_t)from | (uintptr_t)to) & 15) == 0) {
    const uint64_t v = bytes / 16;
    for (uint64_t i = at; i < v; i += stride) ((uint4*)to)[i] = ((const uint4*)from)[i];
    done = v * 16;
  }
  for (uint64_t i = done + at; i < bytes; i += stride) ((uint8_t*)to)[i] = ((const uint8_t*)from)[i];
}

__global__ void __launch_bounds__(kBlock) k_publish(uint32_t n, uint64_t m, uint64_t* cnt, uint64_t* host_cnt,
                                                    const int32_t* label, const uint8_t* core, const uint8_t* flag,
                                                    int32_t* to_label, uint8_t* to_core, uint8_t* to_sim) {
  stamp(cnt, kStampEnd);
  if (blockIdx.x == 0) {
    __syncthreads();
    if (threadIdx.x < kCntSlots) {
      uint64_t v = cnt[threadIdx.x];
      if (threadIdx.x < kStripeSlots)
        for (uint32_t i = 0; i < kStripes; ++i) v += cnt[kStripe0 + i * kStripeSlots + threadIdx.x];
      host_cnt[threadIdx.x] = v;
    }
  }
  if (cnt[kCntOverflow]) return;
  if (to_label) grid_copy(label, to_label, (uint64_t)n * 4);
  if (to_core) grid_copy(core, to_core, n);
  if (to_sim) grid_copy(flag, to_sim, m);
}

// Everything after the similarity phase of a tiny graph, from the core count
// to the results, by one workgroup with the per-vertex state in LDS: the seven
// kernels it replaces do less than a microsecond of work each in launches 2-5
// us apart.  LDS: sd, then the lower label bound; parent, then the upper
// bound; label; core.  Bound by the latency of one CU's loads, so only where
// the entries are few: R-MAT with 10 / 12 thousand entries 67 / 66 -> 54 / 56
// us a pass on the device, but 40 / 80 / 120 thousand 148 / 110 / 120 ->
// 154 / 114 / 136.
constexpr uint32_t kTailVertices = 8192, kTailEntries = 1u << 15;

struct TailArgs {
  uint32_t n, m;
  const uint32_t* src;
  const int32_t* adj;
  const uint32_t* rb;
  const uint32_t* re;
  const uint8_t* flag;
  int32_t mu;
  int32_t* label;
  uint8_t* core;
  const uint64_t* cnt;
  uint64_t* host_cnt;
  int32_t* to_label;
  uint8_t* to_core;
  uint8_t* to_sim;
};

__global__ void __launch_bounds__(1024) k_tail(TailArgs a) {
  constexpr uint32_t T = 1024;
  extern __shared__ __align__(16) int32_t sh[];
  __shared__ uint64_t s_stamp[4];
  __shared__ unsigned long long s_sum[kStripeSlots];  // this kernel's share of the striped sums
  const uint32_t tid = threadIdx.x, n = a.n, m = a.m;
  int32_t* const lo = sh;
  int32_t* const hi = sh + n;
  int32_t* const label = sh + 2 * n;
  uint8_t* const core = (uint8_t*)(sh + 3 * n);
  uint32_t* const sd = (uint32_t*)lo;
  volatile int32_t* const parent = hi;
  auto start = [&](int i) {
    __syncthreads();
    if (tid == 0) s_stamp[i] = (uint64_t)wall_clock64();
  };
  // fn(k) for this thread's similar entries
  auto for_similar = [&](auto fn) {
    for (uint32_t k0 = tid * 16; k0 < m; k0 += T * 16) {
      uint32_t mask = similar_mask(*reinterpret_cast<const uint4*>(a.flag + k0));
      if (k0 + 16 > m) mask &= (1u << (m - k0)) - 1u;
      for (; mask; mask &= mask - 1) fn(k0 + (uint32_t)__ffs(mask) - 1);
    }
  };
  auto sum = [&](int slot, unsigned long long v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_down(v, off);
    if (lane_id() == 0 && v) atomicAdd(&s_sum[slot], v);
  };
  auto find = [&](int32_t x) {
    int32_t p = parent[x];
    while (p != x) {
      const int32_t gp = parent[p];
      if (gp != p) parent[x] = gp;  // path splitting
      x = p;
      p = gp;
    }
    return x;
  };
  for (uint32_t x = tid; x < n; x += T) sd[x] = 0;
  if (tid < kStripeSlots) s_sum[tid] = 0;
  start(0);
  // ---- cores
  for_similar([&](uint32_t k) { atomicAdd(&sd[a.src[k]], 1u); });
  __syncthreads();
  const uint32_t thr = a.mu >= 1 ? (uint32_t)a.mu : 1u;
  uint32_t marked = 0, labeled = 0, similar = 0;
  for (uint32_t x = tid; x < n; x += T) {
    const bool c = sd[x] >= thr;
    similar += sd[x];
    core[x] = c;
    marked += c;
    if (c) labeled += a.re[x] - a.rb[x];
    lo[x] = kNoLabel;
    parent[x] = (int32_t)x;
    label[x] = kNoLabel;
  }
  sum(kCntMarked, marked);
  sum(kCntLabeled, labeled);
  sum(kCntSimilar, similar);
  start(1);
  const bool any = s_sum[kCntMarked] != 0;
  if (any) {
    // ---- clusters
    for_similar([&](uint32_t k) {
      const uint32_t u = a.src[k];
      const int32_t w = a.adj[k];
      if ((uint32_t)w >= u || !core[u] || !core[w]) return;
      for (;;) {
        const int32_t ru = find((int32_t)u), rw = find(w);
        if (ru == rw) return;
        const int32_t top = ru > rw ? ru : rw, low = ru > rw ? rw : ru;
        if (atomicCAS((int32_t*)&parent[top], top, low) == top) return;
      }
    });
    __syncthreads();
    for (uint32_t x = tid; x < n; x += T)
      if (core[x]) label[x] = find((int32_t)x);
    start(2);
    // ---- borders: the minimum candidate id; core labels do not change
    labeled = 0;
    for_similar([&](uint32_t k) {
      const uint32_t u = a.src[k];
      const int32_t w = a.adj[k];
      if (core[u] || !core[w]) return;
      if (atomicMin(&label[u], label[w]) == kNoLabel) labeled += a.re[u] - a.rb[u];
    });
    sum(kCntLabeled, labeled);
    for (uint32_t x = tid; x < n; x += T) hi[x] = -1;
    start(3);
    // ---- hubs and outliers, from the same side as k_classify
    const bool from_labeled = 3 * s_sum[kCntLabeled] < m;
    constexpr uint32_t C = 8;
    for (uint32_t k0 = tid; k0 < m; k0 += T * C) {
      uint32_t row[C];
      int32_t nb[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        const uint32_t k = k0 + j * T;
        row[j] = k < m ? a.src[k] : 0u;
        nb[j] = k < m ? a.adj[k] : 0;
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        if (k0 + j * T >= m) continue;
        const uint32_t from = from_labeled ? row[j] : (uint32_t)nb[j], to = from_labeled ? (uint32_t)nb[j] : row[j];
        const int32_t l = label[from];
        if (l == kNoLabel || label[to] != kNoLabel) continue;
        if (l < lo[to]) atomicMin(&lo[to], l);
        if (l > hi[to]) atomicMax(&hi[to], l);
      }
    }
  } else {
    start(2);
    start(3);
  }
  __syncthreads();
  // ---- roles and results
  const bool publish = a.cnt[kCntOverflow] == 0;
  RoleCounts rc;
  PhaseView v{};
  v.sd = nullptr, v.core = core, v.label = label, v.lo = lo, v.hi = hi;
  for (uint32_t x = tid; x < n; x += T) {
    const int32_t l = role_label(v, x, a.mu, &rc);
    a.label[x] = l;
    a.core[x] = core[x];
    if (publish && a.to_label) a.to_label[x] = l;
    if (publish && a.to_core) a.to_core[x] = core[x];
  }
  if (publish && a.to_sim) {
    uint32_t done = 0;
    if (((uintptr_t)a.to_sim & 15) == 0) {
      done = m / 16 * 16;
      for (uint32_t k = tid * 16; k < done; k += T * 16)
        *reinterpret_cast<uint4*>(a.to_sim + k) = *reinterpret_cast<const uint4*>(a.flag + k);
    }
    for (uint32_t k = done + tid; k < m; k += T) a.to_sim[k] = a.flag[k];
  }
  sum(kCntCores, rc.cores);
  sum(kCntClusters, rc.clusters);
  sum(kCntBorders, rc.borders);
  sum(kCntHubs, rc.hubs);
  sum(kCntOutliers, rc.outliers);
  __syncthreads();
  if (tid < kCntSlots) {
    uint64_t v = a.cnt[tid];
    if (tid < kStripeSlots) {
      for (uint32_t i = 0; i < kStripes; ++i) v += a.cnt[kStripe0 + i * kStripeSlots + tid];
      v += s_sum[tid];
    }
    const int i = (int)tid - kCntStamp0;
    if (i >= kStampCore && i < kStampEnd) v = s_stamp[i - kStampCore];
    if (i == kStampEnd) v = (uint64_t)wall_clock64();
    a.host_cnt[tid] = v;
  }
}

// Plain streaming copy (16 bytes per lane per step), the reference point for
// the HBM byte counters.
__global__ void __launch_bounds__(kBlock) k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

}  // namespace

void launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t s) {
  const uint64_t n = bytes / sizeof(uint4);
  if (n) k_copy<<<grid_for(n, kBlock), kBlock, 0, s>>>((const uint4*)src, (uint4*)dst, n);
}

void launch_fill_rows(const uint32_t* rp, uint32_t n, uint32_t m, uint32_t base, uint32_t* src, hipStream_t s) {
  if (n && m) k_fill_rows<<<grid_for(m, kFillTile * (kBlock / kWave)), kBlock, 0, s>>>(n, m, base, rp, src);
}

static void launch_neighbor_degrees(const sgc_dgraph* g, hipStream_t s) {
  if (g->m && g->ndeg)
    k_neighbor_degrees<<<grid_for(g->m, kBlock), kBlock, 0, s>>>(g->m, g->row_ptr, g->adj, g->ndeg);
}

static void launch_mirror(const sgc_dgraph* g, hipStream_t s) {
  if (!g->m || !g->mirror) return;
  // words of entries without a reverse entry are never written by k_mirror
  (void)hipMemsetAsync(g->mirror, 0xFF, (size_t)g->m * 4, s);
  k_mirror<<<grid_for(g->m, kBlock), kBlock, 0, s>>>(g->m, g->row_ptr, g->src, g->adj, g->mirror);
}

// Up to here one search an entry is as fast (its rows come from L2): with the
// neighbour degrees, 1.8e6 entries 65 us against 63 split, but 4e6 161 against
// 76, 7.6e6 (R-MAT-18) 366 / 145.  Above kSplitEntries the sort takes over: a
// bucket's rows no longer fit LDS, or its items come one by one.
constexpr uint32_t kSearchEntries = 1u << 21;

// Work memory of the sort: keys out, values in and out, its scratch and the
// mismatch count.
struct SortLayout {
  size_t vin, vout, tmp, bad, bytes, tmp_bytes;
  int key_bits;
};

static SortLayout sort_layout(const sgc_dgraph* g, hipStream_t s) {
  SortLayout L{};
  const size_t m = g->m;
  L.key_bits = 1;
  while (L.key_bits < 32 && (1ull << L.key_bits) < (uint64_t)g->n) ++L.key_bits;
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, L.tmp_bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr,
                                           (const uint64_t*)nullptr, (uint64_t*)nullptr, g->m, 0, L.key_bits, s);
  L.vin = (m * 4 + 255) / 256 * 256;
  L.vout = L.vin + m * 8;
  L.tmp = L.vout + m * 8;
  L.bad = L.tmp + (L.tmp_bytes + 255) / 256 * 256;
  L.bytes = L.bad + 256;
  return L;
}

static size_t split_bytes(uint32_t m) {
  return (size_t)((m + (1u << kBucketBits) - 1) >> kBucketBits) * (kBucketCap * sizeof(SplitItem) + 4);
}

size_t index_work_bytes(const sgc_dgraph* g) {
  if (!g->mirror || g->m <= kSearchEntries) return 0;
  return g->m <= kSplitEntries && g->ndeg ? split_bytes(g->m) : sort_layout(g, g->ctx->stream).bytes;
}

static hipError_t build_mirror(sgc_ctx* ctx, const sgc_dgraph* g);

hipError_t build_indexes(sgc_ctx* ctx, const sgc_dgraph* g) {
  hipStream_t s = ctx->stream;
  const uint32_t m = g->m;
  if (m > kSearchEntries && m <= kSplitEntries && g->mirror && g->ndeg) {
    const uint32_t buckets = (m + (1u << kBucketBits) - 1) >> kBucketBits;
    char* const mem = (char*)work_memory(ctx, split_bytes(m));
    if (mem) {
      uint32_t* const cursor = (uint32_t*)(mem + (size_t)buckets * kBucketCap * sizeof(SplitItem));
      hipError_t e = hipMemsetAsync(cursor, 0, (size_t)buckets * 4, s);
      if (e == hipSuccess) e = hipMemsetAsync(g->mirror, 0xFF, (size_t)m * 4, s);
      if (e != hipSuccess) return e;
      k_split_searches<<<std::min(grid_for(m, 16384), 1024u), 1024, 0, s>>>(m, g->row_ptr, g->src, g->adj, g->ndeg,
                                                                             g->mirror, cursor, (SplitItem*)mem, buckets);
      k_bucket_searches<<<buckets, 1024, 0, s>>>(m, g->adj, cursor, (const SplitItem*)mem, g->mirror);
      return hipGetLastError();
    }
  }
  launch_neighbor_degrees(g, s);
  return build_mirror(ctx, g);
}

static hipError_t build_mirror(sgc_ctx* ctx, const sgc_dgraph* g) {
  if (!g->m || !g->mirror) return hipSuccess;
  hipStream_t s = ctx->stream;
  const uint32_t m = g->m;
  if (m <= kSearchEntries) {
    launch_mirror(g, s);
    return hipGetLastError();
  }
  SortLayout L = sort_layout(g, s);
  char* const mem = (char*)work_memory(ctx, L.bytes);
  if (!mem) {
    launch_mirror(g, s);  // not enough room to sort: search each reverse entry
    return hipGetLastError();
  }
  uint32_t* keys = (uint32_t*)mem;
  uint64_t* vin = (uint64_t*)(mem + L.vin);
  uint64_t* vout = (uint64_t*)(mem + L.vout);
  unsigned long long* bad = (unsigned long long*)(mem + L.bad);
  k_rows_and_positions<<<grid_for(m, kBlock), kBlock, 0, s>>>(m, g->src, vin);
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(mem + L.tmp, L.tmp_bytes, (const uint32_t*)g->adj, keys, vin,
                                                     vout, m, 0, L.key_bits, s);
  if (e == hipSuccess) e = hipMemsetAsync(bad, 0, 8, s);
  if (e == hipSuccess) {
    k_mirror_from_sorted<<<grid_for(m, kBlock), kBlock, 0, s>>>(m, g->src, g->adj, keys, vout, g->mirror, bad);
    e = hipGetLastError();
  }
  unsigned long long h_bad = 0;
  if (e == hipSuccess) e = hipMemcpyAsync(&h_bad, bad, 8, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess && h_bad) {  // some entry lacks its reverse: the search finds those that exist
    launch_mirror(g, s);
    e = hipGetLastError();
  }
  return e;
}

void launch_init(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  k_init<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, b.sd, b.lo, b.hi, b.core, b.cnt_u, b.work_u, b.cnt);
}

void launch_similarity_wave(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s) {
  if (g->m == 0) return;
  const uint32_t blocks = (uint32_t)(cu_count > 0 ? cu_count : 256) * 8;
  // the list takes the tiered kernels' uedge array, which this kernel replaces
  uint32_t* list = reinterpret_cast<uint32_t*>(b.uedge);
  k_list_owned<<<grid_for(g->m, kBlock), kBlock, 0, s>>>(g->m, b.flag, list, b.cnt);
  k_similarity_wave<<<blocks, kBlock, 0, s>>>(g->row_begin, g->row_end, g->adj, g->src, p.eps, b.flag, list,
                                              b.cnt);
}

// Graphs below this many entries skip the launches that only pay on large
// ones (the list of labelled rows, a flatten kernel of its own): a launch
// costs 2-5 us, and the walk of all entries it saves no more than that.
// R-MAT with 1.8 / 3.8 million entries: 159 / 437 us a pass with them, 155 /
// 405 without.
constexpr uint64_t kSmallGraph = 1u << 22;

// The first union round pays from here on: planted communities with 0.7 / 1.4
// million entries 80 / 81 -> 37 / 37 us in two rounds (and 3.4 million 300 ->
// 78); without cores the two launches cost 3.
constexpr uint64_t kUnionRounds = 1u << 19;

// Passes over fewer flags than this take the short tile: planted communities
// with 0.7 / 3.4 / 8.1 million entries 109 / 121 / 143 us in the core count,
// union-find and borders with the long one, 50 / 98 / 127 with the short (in
// two union rounds).  Above, tiles keep every wave busy, and the short one
// reads a graph with few similar entries at half the rate (R-MAT-20: 64 us
// against 90; planted with 55 million entries 338 against 263).
constexpr uint64_t kShortTiles = 1u << 24;

// Blocks of a pass over the flags by similar_tile.
static uint32_t flag_grid(uint64_t m) {
  return std::min(grid_for(m, (m < kShortTiles ? kShortTile : kFlagTile) * (kBlock / kWave)), m < kShortTiles ? 4096u : 2048u);
}

// Calls fn with the tile's size as a constant.
template <typename Fn>
static void with_tile(uint64_t m, Fn fn) {
  if (m < kShortTiles)
    fn(std::integral_constant<uint32_t, kShortTile>());
  else
    fn(std::integral_constant<uint32_t, kFlagTile>());
}

// Edge passes take the entries [0, g->m) of g (a whole graph or one chip of
// rows); vertex passes cover all g->n vertices.
void launch_core_count(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  if (!g->m) return;
  with_tile(g->m, [&](auto tile) {
    k_core_count<tile><<<flag_grid(g->m), kBlock, 0, s>>>(g->m, g->src, b.flag, b.sd, b.cnt);
  });
}

void launch_core_mark(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s,
                      const int32_t* mu_dev) {
  k_core_mark<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, b.sd, p.mu, mu_dev, g->row_begin, g->row_end, b.core,
                                                       b.parent, b.label, b.lo, b.hi, b.cnt);
}

void launch_union(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, int gate) {
  if (!g->m) return;
  const uint32_t grid = flag_grid(g->m);
  with_tile(g->m, [&](auto tile) {
    if (g->m >= kUnionRounds) {
      k_union<true, tile><<<grid, kBlock, 0, s>>>(g->m, g->src, g->adj, b.flag, b.core, b.parent, b.cnt, gate);
      k_compress<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, b.core, b.parent, b.cnt);
    }
    k_union<false, tile><<<grid, kBlock, 0, s>>>(g->m, g->src, g->adj, b.flag, b.core, b.parent, b.cnt, gate);
  });
}

void launch_redo_mark(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  if (g->m && g->mirror)
    k_redo_mark<<<grid_for(g->m, kBlock), kBlock, 0, s>>>(g->m, g->src, g->adj, g->mirror, b.flag, b.core, b.parent,
                                                         b.cnt);
}

void launch_flatten(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  k_flatten<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, b.core, b.parent, b.label);
}

void launch_border(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, bool flatten) {
  if (!g->m) return;
  with_tile(g->m, [&](auto tile) {
    if (flatten)
      k_border<true, tile><<<std::max(flag_grid(g->m), std::min(grid_for(g->n, kBlock), 1024u)), kBlock, 0, s>>>(
          g->n, g->m, b.parent, g->src, g->adj, b.flag, b.core, g->row_begin, g->row_end, b.label, b.cnt);
    else
      k_border<false, tile><<<flag_grid(g->m), kBlock, 0, s>>>(g->n, g->m, b.parent, g->src, g->adj, b.flag, b.core,
                                                               g->row_begin, g->row_end, b.label, b.cnt);
  });
}

bool small_graph(const sgc_dgraph* g) { return g->m < kSmallGraph; }

void launch_classify_edges(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s, uint64_t m_all) {
  if (!g->m) return;
  // a whole graph lists its labelled rows, in the edge records' memory (free
  // by now; serving slots have none)
  const bool listed = !m_all && b.uedge && g->row_begin && g->m >= kSmallGraph;
  if (listed) {
    uint2* const piece = reinterpret_cast<uint2*>(b.uedge);
    k_label_pieces<<<grid_for(g->n, kBlock * 8), kBlock, 0, s>>>(g->n, g->m, g->row_begin, g->row_end, b.label, piece,
                                                                 b.cnt);
    k_classify_rows<<<2048, kBlock, 0, s>>>(g->row_begin, g->row_end, g->adj, b.label, b.lo, b.hi, piece, b.cnt);
  }
  k_classify<<<grid_for(g->m, kBlock), kBlock, 0, s>>>(g->m, m_all ? m_all : g->m, g->src, g->adj, b.label, b.lo, b.hi,
                                                       b.cnt, listed);
}

void launch_finalize(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s,
                     const int32_t* mu_dev) {
  k_finalize<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, p.mu, mu_dev, b.sd, b.lo, b.hi, b.core, b.label, b.cnt);
}


bool tiny_graph(const sgc_dgraph* g) { return g->m && g->n <= kTailVertices && g->m <= kTailEntries; }

void launch_tail(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, uint64_t* host_cnt, int32_t* labels,
                 uint8_t* core, uint8_t* sim, hipStream_t s) {
  const TailArgs a{g->n, g->m, g->src, g->adj, g->row_begin, g->row_end, b.flag, p.mu, b.label, b.core, b.cnt,
                   host_cnt, labels, core, sim};
  k_tail<<<1, 1024, (size_t)g->n * 13, s>>>(a);
}

void launch_publish(const sgc_dgraph* g, const PassBuffers& b, uint64_t* host_cnt, int32_t* labels, uint8_t* core,
                    uint8_t* sim, hipStream_t s) {
  const uint64_t bytes = (labels ? (uint64_t)g->n * 4 : 0) + (core ? g->n : 0) + (sim ? g->m : 0);
  k_publish<<<std::min(grid_for(bytes / 16, kBlock), 2048u), kBlock, 0, s>>>(g->n, g->m, b.cnt, host_cnt, b.label,
                                                                             b.core, b.flag, labels, core, sim);
}

void launch_core(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s) {
  launch_core_count(g, b, s);
  launch_core_mark(g, b, p, s);
}

void launch_classify(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, hipStream_t s) {
  launch_classify_edges(g, b, s);
  launch_finalize(g, b, p, s);
}

}  // namespace sgc
