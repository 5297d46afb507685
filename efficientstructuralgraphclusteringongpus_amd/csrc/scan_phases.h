// The SCAN phases after the similarity phase as wave- and thread-level device
// functions over one graph's arrays: the single-graph kernels (kernels.hip)
// run them over grid-stride loops, the batched query kernels (serve.hip) over
// the tiles of many queries in one launch.  Semantics:
// GPUSCAN++/GPUScan.cu:276-367 (core), :465-652 (union-find, minimum-id
// roots), :654-730 (borders, canonical minimum candidate), :732-798 (hubs and
// outliers).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device.h"
#include "device_util.h"

namespace sgc {

// Arrays of one query over one graph (entries [0, m), vertices [0, n)).
struct PhaseView {
  uint32_t n, m;
  const uint32_t* src;  // m: row of each entry
  const int32_t* adj;   // m
  const uint32_t* rb;   // row starts and ends (null: labelled-entry counts are skipped)
  const uint32_t* re;
  const uint8_t* flag;  // m
  uint32_t* sd;         // n: similar entries per row
  uint8_t* core;        // n
  int32_t* parent;      // n
  int32_t* label;       // n
  int32_t* lo;          // n
  int32_t* hi;          // n
};

// ---- core check: core(x) <=> #similar neighbours >= mu (mu <= 0: >= 1).
// Returns x's row length when x is a core and row offsets are known (the
// labelled entries classify chooses its side by), else 0; *marked = core.
__device__ __forceinline__ uint32_t core_mark_vertex(const PhaseView& v, uint32_t x, int32_t mu, uint32_t* marked) {
  const uint32_t thr = mu >= 1 ? (uint32_t)mu : 1u;
  const bool c = v.sd[x] >= thr;
  v.core[x] = c;
  v.parent[x] = (int32_t)x;
  v.label[x] = kNoLabel;
  v.lo[x] = kNoLabel;  // classify's neighbour-label bounds
  v.hi[x] = -1;
  *marked = c;
  return c && v.rb ? v.re[x] - v.rb[x] : 0u;
}

// ---- union-find, parents always smaller than children
__device__ __forceinline__ int32_t uf_find(int32_t* parent, int32_t x) {
  int32_t p = ld_coherent(parent + x);
  while (p != x) {
    const int32_t gp = ld_coherent(parent + p);
    if (gp != p) st_coherent(parent + x, gp);  // path splitting
    x = p;
    p = gp;
  }
  return x;
}

__device__ __forceinline__ void uf_union(int32_t* parent, int32_t a, int32_t b) {
  for (;;) {
    const int32_t ra = uf_find(parent, a), rb = uf_find(parent, b);
    if (ra == rb) return;
    const int32_t hi = ra > rb ? ra : rb, lo = ra > rb ? rb : ra;
    if (atomicCAS(parent + hi, hi, lo) == hi) return;
  }
}

// Bit i: flag i of 16 says similar.
__device__ __forceinline__ uint32_t similar_mask(const uint4 w) {
  const uint32_t x[4] = {w.x, w.y, w.z, w.w};
  uint32_t mask = 0;
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) {
    const uint32_t z = x[q] ^ (0x01010101u * kFlagY);
    const uint32_t t = ~(((z & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | z | 0x7F7F7F7Fu);  // 0x80 in zero bytes
    mask |= (((t >> 7) & 1u) | ((t >> 14) & 2u) | ((t >> 21) & 4u) | ((t >> 28) & 8u)) << (4 * q);
  }
  return mask;
}

// The similar entries of the wave's tile [base, base + TILE) of the flag
// array, ascending, into `at` (the wave's TILE words of LDS, offsets from
// base); returns their number (uniform).  Flags come 16 to a load, or 4 in the
// short tile (flag must be 16-byte aligned and readable up to the next
// multiple of 16): a byte a lane read them at 0.9 TB/s.  The short tile is for
// graphs that fill the chip with few waves otherwise, where a wave with 2048
// similar entries is the whole pass.
constexpr uint32_t kFlagTile = 2048, kShortTile = 256;

template <uint32_t TILE>
__device__ __forceinline__ uint32_t similar_tile(const uint8_t* __restrict__ flag, uint64_t m, uint64_t base,
                                                 uint16_t* at) {
  static_assert(TILE == kFlagTile || TILE == kShortTile, "flags per lane and load");
  constexpr uint32_t F = TILE == kShortTile ? 4 : 16, L = TILE / (kWave * F);
  const uint32_t lane = lane_id();
  uint4 w[L];
#pragma unroll
  for (uint32_t j = 0; j < L; ++j) {
    const uint64_t k = base + (j * kWave + lane) * F;
    w[j] = make_uint4(0, 0, 0, 0);
    if (k < m) {
      if (F == 16)
        w[j] = *reinterpret_cast<const uint4*>(flag + k);
      else
        w[j].x = *reinterpret_cast<const uint32_t*>(flag + k);
    }
  }
  uint32_t total = 0;
#pragma unroll
  for (uint32_t j = 0; j < L; ++j) {
    const uint64_t k = base + (j * kWave + lane) * F;
    uint32_t mask = similar_mask(w[j]);
    if (k + F > m) mask &= k < m ? (1u << (uint32_t)(m - k)) - 1u : 0u;
    if (!__ballot(mask != 0)) continue;
    const uint32_t incl = wave_incl_scan((uint32_t)__popc(mask));
    uint32_t pos = total + incl - (uint32_t)__popc(mask);
    for (uint32_t b = mask; b; b &= b - 1) at[pos++] = (uint16_t)((j * kWave + lane) * F + (uint32_t)__ffs(b) - 1);
    total += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
  }
  wave_lds_sync();
  return total;
}

// The core count and the union-find take this many wave loads of listed
// entries at a time: each entry costs two to four dependent gathers, and one
// load at a time left them waiting (planted communities, n = 3e5, 7e6 similar
// entries: core count 65 -> 39 us, union-find 260 -> 225; the border pass,
// whose entries rarely pass the first gather, gains nothing: 72 / 76).
constexpr uint32_t kListed = 4;

// Similar entries per row among the wave's tile at `base`: one atomic per run
// of a row's entries in a wave's 64.
template <uint32_t TILE = kFlagTile>
__device__ __forceinline__ void core_count_tile(const PhaseView& v, uint64_t base, uint16_t* at) {
  const uint32_t lane = lane_id();
  const uint32_t total = similar_tile<TILE>(v.flag, v.m, base, at);
  for (uint32_t i0 = 0; i0 < total; i0 += kWave * kListed) {
    uint32_t row[kListed];
#pragma unroll
    for (uint32_t j = 0; j < kListed; ++j) {
      const uint32_t i = i0 + j * kWave + lane;
      row[j] = i < total ? v.src[base + at[i]] : 0xFFFFFFFFu;
    }
#pragma unroll
    for (uint32_t j = 0; j < kListed; ++j) {
      if (i0 + j * kWave >= total) break;
      const bool head = wave_seg_head(row[j]);
      const uint64_t after = __ballot(head) & ~lanemask_le(lane);
      const uint32_t stop = after ? (uint32_t)(__ffsll((long long)after) - 1) : (uint32_t)kWave;
      if (head && row[j] != 0xFFFFFFFFu) atomicAdd(&v.sd[row[j]], stop - lane);
    }
  }
  wave_lds_sync();  // the list is rewritten
}

// Joins the similar core-core edges of the wave's tile, each visited from its
// larger endpoint.  HEADS: one edge per run of a row's entries only.
template <bool HEADS, uint32_t TILE = kFlagTile>
__device__ __forceinline__ void union_tile(const PhaseView& v, uint64_t base, uint16_t* at) {
  const uint32_t lane = lane_id();
  const uint32_t total = similar_tile<TILE>(v.flag, v.m, base, at);
  for (uint32_t i0 = 0; i0 < total; i0 += kWave * kListed) {
    uint32_t u[kListed];
    int32_t w[kListed];
    bool on[kListed];
#pragma unroll
    for (uint32_t j = 0; j < kListed; ++j) {
      const uint32_t i = i0 + j * kWave + lane;
      const uint64_t k = base + (i < total ? at[i] : 0);
      u[j] = i < total ? v.src[k] : 0u;
      w[j] = i < total ? v.adj[k] : 0;
    }
#pragma unroll
    for (uint32_t j = 0; j < kListed; ++j) on[j] = (uint32_t)w[j] < u[j] && v.core[u[j]] && v.core[w[j]];
    if (!HEADS) {
#pragma unroll
      for (uint32_t j = 0; j < kListed; ++j) on[j] = on[j] && v.parent[u[j]] != v.parent[w[j]];
    }
#pragma unroll
    for (uint32_t j = 0; j < kListed; ++j) {
      if (HEADS) {
        // the first of the row's entries among the lanes that are on
        const uint64_t below = __ballot(on[j]) & lanemask_lt(lane);
        const uint32_t prev = below ? 63u - (uint32_t)__clzll((long long)below) : lane;
        const uint32_t pu = (uint32_t)__shfl((int)u[j], (int)prev);
        on[j] = on[j] && (!below || pu != u[j]);
      }
      if (on[j]) uf_union(v.parent, (int32_t)u[j], w[j]);
    }
  }
  wave_lds_sync();  // the list is rewritten
}

// Roots go to label: the finds keep splitting paths in parent (stores of
// ancestors only), which must not land on a finished label.
__device__ __forceinline__ void flatten_vertex(const PhaseView& v, uint32_t x) {
  if (v.core[x]) v.label[x] = uf_find(v.parent, (int32_t)x);
}

// ---- borders: the minimum candidate cluster id over similar edges to cores,
// for one similar entry k per lane (on; ascending over the lanes).  A row's
// candidates may lie in several runs of lanes (other entries between them get
// a marker row), each run's minimum is added.  Returns the entries of the
// border rows this lane labelled first (rows known only).  FIND: the cores'
// cluster ids are not in label yet.  All 64 lanes must call it.
template <bool FIND>
__device__ __forceinline__ uint32_t border_entry(const PhaseView& v, uint64_t k, bool on) {
  const uint32_t row = on ? v.src[k] : 0xFFFFFFFFu;
  const int32_t c = on ? v.adj[k] : 0;
  const bool y = on && v.core[c] && !v.core[row];
  if (!__ballot(y)) return 0;
  const int32_t cand = !y ? kNoLabel : FIND ? uf_find(v.parent, c) : v.label[c];
  const uint32_t r = y ? row : 0xFFFFFFFFu;
  const int32_t best = wave_seg_reduce(r, cand, OpMin());
  if (wave_seg_head(r) && best != kNoLabel && atomicMin(&v.label[r], best) == kNoLabel && v.rb)
    return v.re[r] - v.rb[r];
  return 0;
}

// The same for the wave's tile at `base`.
template <bool FIND, uint32_t TILE = kFlagTile>
__device__ __forceinline__ uint32_t border_tile(const PhaseView& v, uint64_t base, uint16_t* at) {
  const uint32_t total = similar_tile<TILE>(v.flag, v.m, base, at);
  uint32_t labeled = 0;
  for (uint32_t i0 = 0; i0 < total; i0 += kWave) {
    const bool on = i0 + lane_id() < total;
    labeled += border_entry<FIND>(v, base + (on ? at[i0 + lane_id()] : 0), on);
  }
  wave_lds_sync();  // the list is rewritten
  return labeled;
}

// ---- hubs and outliers: every unlabelled vertex's min and max neighbour
// label, for the wave chunk at `base`.  from_labeled: walk the labelled rows
// and hand each label to the unlabelled neighbours (few labelled entries),
// else walk the unlabelled rows and gather.  Two different labels <=> the
// reference finds a first labelled neighbour and a later one with another.
__device__ __forceinline__ void classify_chunk(const PhaseView& v, uint64_t base, bool from_labeled) {
  constexpr uint32_t C = kEdgeChunks;
  const uint32_t lane = lane_id();
  uint32_t row[C];
#pragma unroll
  for (uint32_t j = 0; j < C; ++j) {
    const uint64_t k = base + j * kWave + lane;
    row[j] = k < v.m ? v.src[k] : 0xFFFFFFFFu;
  }
  int32_t lr[C];
#pragma unroll
  for (uint32_t j = 0; j < C; ++j) lr[j] = row[j] != 0xFFFFFFFFu ? v.label[row[j]] : kNoLabel;
  // neighbours only where this side needs them
  int32_t nb[C];
#pragma unroll
  for (uint32_t j = 0; j < C; ++j)
    nb[j] = row[j] != 0xFFFFFFFFu && (from_labeled ? lr[j] != kNoLabel : lr[j] == kNoLabel)
                ? v.adj[base + j * kWave + lane]
                : 0;
  if (from_labeled) {
    bool to[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) to[j] = lr[j] != kNoLabel && v.label[nb[j]] == kNoLabel;
#pragma unroll
    for (uint32_t j = 0; j < C; ++j)
      if (to[j]) {
        atomicMin(&v.lo[nb[j]], lr[j]);
        atomicMax(&v.hi[nb[j]], lr[j]);
      }
    return;
  }
  int32_t ly[C];
#pragma unroll
  for (uint32_t j = 0; j < C; ++j) ly[j] = row[j] != 0xFFFFFFFFu && lr[j] == kNoLabel ? v.label[nb[j]] : kNoLabel;
#pragma unroll
  for (uint32_t j = 0; j < C; ++j) {
    const bool has = ly[j] != kNoLabel;
    if (!__ballot(has)) continue;
    const int32_t vmin = wave_seg_reduce(row[j], has ? ly[j] : kNoLabel, OpMin());
    const int32_t vmax = wave_seg_reduce(row[j], has ? ly[j] : -1, OpMax());
    if (wave_seg_head(row[j]) && vmax >= 0) {
      atomicMin(&v.lo[row[j]], vmin);
      atomicMax(&v.hi[row[j]], vmax);
    }
  }
}

// Final label of vertex x and its role, added to the counts: cores, the
// clusters (roots), borders, hubs, outliers, and x's similar entries.
struct RoleCounts {
  uint32_t cores = 0, clusters = 0, borders = 0, hubs = 0, outliers = 0;
  uint64_t similar = 0;
};

__device__ __forceinline__ void count_roles(uint64_t* cnt, const RoleCounts& rc) {
  count_add<6>(cnt, {kCntCores, kCntClusters, kCntBorders, kCntHubs, kCntOutliers, kCntSimilar},
               {rc.cores, rc.clusters, rc.borders, rc.hubs, rc.outliers, rc.similar});
}

__device__ __forceinline__ int32_t role_label(const PhaseView& v, uint32_t x, int32_t mu, RoleCounts* rc) {
  int32_t l = v.label[x];
  if (v.core[x]) {
    ++rc->cores;
    rc->clusters += l == (int32_t)x;
  } else if (l != kNoLabel) {
    ++rc->borders;
  } else {
    // mu <= 0: the reference classifies only role -2 vertices and there are
    // none, so every non-core keeps role -1 (GPUScan.cu:978-984).
    const bool hub = mu <= 0 || (v.lo[x] != kNoLabel && v.lo[x] != v.hi[x]);
    l = hub ? -1 : -2;
    v.label[x] = l;
    rc->hubs += hub;
    rc->outliers += !hub;
  }
  return l;
}

__device__ __forceinline__ int32_t finalize_vertex(const PhaseView& v, uint32_t x, int32_t mu, RoleCounts* rc) {
  rc->similar += v.sd[x];
  return role_label(v, x, mu, rc);
}

}  // namespace sgc
