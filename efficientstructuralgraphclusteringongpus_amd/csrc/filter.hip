// Filter stage of the similarity phase for resident graphs.
//
// Almost every edge that the degree-only test leaves undecided is dissimilar,
// and with room to spare: on R-MAT the common neighbours of half of them are
// under half of the threshold c*.  This stage rejects them from a compact
// copy of the rows, and leaves the few others to the exact kernels.
//
// Packed rows (built at upload).  A vertex v has a 16-bit hash and one of 16
// classes by its degree, cut so that each class holds a sixteenth of all
// entries, rarest vertices first.  A row is a list of 16-byte groups: a
// 16-bit header and seven hashes.  In wide rows (kWideRow entries or more)
// every group holds one class, named in its header, rarest class first; in
// narrow rows the classes are mixed and the header says "fold".  That is 2.3
// to 2.4 bytes an entry instead of 4.
//
// Filter.  The owner's row N(b) is a bit set in LDS: one window of 2^16 bits
// per pair of classes and one fold window over all of them (2^13 bits for
// short owner rows).  A clear bit proves that an element of N(a) is not in
// N(b), so an edge that needs c* common neighbours is dissimilar once
// d(a) - c* + 1 elements have missed: an exact rejection.  Hits may be false
// (l / 2^16 to l / 2^19 of the probes), so an edge whose row ends first
// survives and is decided by counting.  Rare neighbours first means misses
// first: 10-20 % fewer elements than in id order (CPU replay of R-MAT-20 and
// 22).
//
// R-MAT-24 (2.6e8 edges), eps 0.2: 62.5 ms for the three filters and 4.8 for
// the survivors, where the exact kernels alone took 129 (owners above degree
// 1024) + 19.5 (below) + 3.6 (tiny owners); the build takes 6 ms at upload.
#include <hip/hip_runtime.h>

#include <algorithm>

#include <hipcub/device/device_scan.hpp>

#include "device.h"
#include "device_util.h"

namespace sgc {

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kGroup = 7;            // elements per group
constexpr uint32_t kClasses = 16;
constexpr uint32_t kWideRow = 512;        // rows of at least this many entries are ordered by class
constexpr uint32_t kWindowWords16 = 2048;   // 2^16 bits
constexpr uint32_t kDegBuckets = 512;       // degree buckets: 16 per power of two

// Group headers: 0 = fold, else 2 + class; header >> 1 is the filter window
// (0 fold, 1..8 pairs of classes).
__device__ __forceinline__ uint32_t class_header(uint32_t c) { return 2 + c; }

// 0xFFFF is the padding element, whose bit is set in every filter.
__device__ __forceinline__ uint32_t hash16(uint32_t x) {
  const uint32_t h = (x * 0x9E3779B1u) >> 16;
  return h < 0xFFFFu ? h : 0xFFFEu;
}

__device__ __forceinline__ uint32_t degree_bucket(uint32_t d) {
  if (d < 16) return d;
  const uint32_t e = 31 - __clz(d);
  return (e - 3) * 16 + ((d >> (e - 4)) & 15);
}

// Class of vertex x of degree d: tab[bucket] = (first, width) of the bucket's
// share of all entries in sixteenths; a second hash of x places it inside.
__device__ __forceinline__ uint32_t vertex_class(uint32_t x, uint32_t d, const float2* tab) {
  const float2 t = tab[degree_bucket(d)];
  const float u = (float)((x * 0x85EBCA77u) >> 8) * (1.0f / 16777216.0f);
  const int c = (int)(t.x + t.y * u);
  return c < (int)kClasses - 1 ? (uint32_t)c : kClasses - 1;
}

// ---------------------------------------------------------------------------
// Packed rows
// ---------------------------------------------------------------------------

__global__ void k_degree_clear(unsigned long long* __restrict__ mass, uint32_t* __restrict__ wide_count) {
  if (threadIdx.x < kDegBuckets) mass[threadIdx.x] = 0;
  if (threadIdx.x == 0) *wide_count = 0;
}

// Entries per degree bucket of the neighbour.
__global__ void __launch_bounds__(kBlock) k_degree_mass(uint32_t n, const uint32_t* __restrict__ rp,
                                                        unsigned long long* __restrict__ mass) {
  __shared__ unsigned long long h[kDegBuckets];
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock) h[t] = 0;
  __syncthreads();
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n; x += stride) {
    const uint32_t d = rp[x + 1] - rp[x];
    if (d) atomicAdd(&h[degree_bucket(d)], (unsigned long long)d);
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock)
    if (h[t]) atomicAdd(&mass[t], h[t]);
}

__global__ void __launch_bounds__(kDegBuckets) k_degree_table(const unsigned long long* __restrict__ mass,
                                                              float2* __restrict__ tab) {
  __shared__ unsigned long long s[kDegBuckets];
  const uint32_t t = threadIdx.x;
  const unsigned long long own = mass[t];
  s[t] = own;
  __syncthreads();
  for (uint32_t off = 1; off < kDegBuckets; off <<= 1) {
    const unsigned long long v = t >= off ? s[t - off] : 0ull;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  const double total = (double)(s[kDegBuckets - 1] ? s[kDegBuckets - 1] : 1ull);
  tab[t] = make_float2((float)(kClasses * ((double)(s[t] - own) / total)), (float)(kClasses * ((double)own / total)));
}

// Groups of every narrow row; the wide rows are listed.
__global__ void __launch_bounds__(kBlock) k_pack_count(uint32_t n, const uint32_t* __restrict__ rp,
                                                       uint32_t* __restrict__ groups, uint32_t* __restrict__ wide,
                                                       uint32_t* __restrict__ wide_count) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x <= n; x += stride) {
    const uint32_t d = x < n ? rp[x + 1] - rp[x] : 0u;
    if (d >= kWideRow)
      wide[atomicAdd(wide_count, 1u)] = (uint32_t)x;
    else
      groups[x] = (d + kGroup - 1) / kGroup;
  }
}

// Class sizes of the row [b, e) into h[kClasses] (LDS), by the whole block.
__device__ __forceinline__ void count_classes(uint32_t b, uint32_t e, const int32_t* __restrict__ adj,
                                              const uint32_t* __restrict__ ndeg, const float2* tab, uint32_t* h) {
  constexpr uint32_t C = 4;
  if (threadIdx.x < kClasses) h[threadIdx.x] = 0;
  __syncthreads();
  for (uint64_t k0 = b; k0 < e; k0 += kBlock * C) {
    uint32_t x[C], d[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      const uint64_t k = k0 + j * kBlock + threadIdx.x;
      x[j] = k < e ? (uint32_t)adj[k] : 0u;
      d[j] = k < e ? ndeg[k] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < C; ++j)
      if (d[j]) atomicAdd(&h[vertex_class(x[j], d[j], tab)], 1u);
  }
  __syncthreads();
}

// Groups of the wide rows, one block per row.
__global__ void __launch_bounds__(kBlock) k_wide_count(const uint32_t* __restrict__ rp, const int32_t* __restrict__ adj,
                                                       const uint32_t* __restrict__ ndeg,
                                                       const float2* __restrict__ tab_g,
                                                       const uint32_t* __restrict__ wide,
                                                       const uint32_t* __restrict__ wide_count,
                                                       uint32_t* __restrict__ groups) {
  __shared__ float2 tab[kDegBuckets];
  __shared__ uint32_t h[kClasses];
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock) tab[t] = tab_g[t];
  __syncthreads();
  const uint32_t count = *wide_count;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t x = wide[i];
    count_classes(rp[x], rp[x + 1], adj, ndeg, tab, h);
    if (threadIdx.x == 0) {
      uint32_t g = 0;
      for (uint32_t c = 0; c < kClasses; ++c) g += (h[c] + kGroup - 1) / kGroup;
      groups[x] = g;
    }
    __syncthreads();
  }
}

// Narrow rows: entry i of a row is element i % 7 of the row's group i / 7.
__global__ void __launch_bounds__(kBlock) k_pack_narrow(uint32_t m, const uint32_t* __restrict__ rp,
                                                        const uint32_t* __restrict__ src,
                                                        const int32_t* __restrict__ adj,
                                                        const uint32_t* __restrict__ gs, uint16_t* __restrict__ packed) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < m; k += stride) {
    const uint32_t u = src[k], b = rp[u], d = rp[u + 1] - b;
    if (d >= kWideRow) continue;
    const uint32_t i = (uint32_t)k - b, q = i / kGroup, r = i % kGroup, h = hash16((uint32_t)adj[k]);
    uint16_t* const g = packed + ((uint64_t)gs[u] + q) * 8;
    if (r == 0)
      *reinterpret_cast<uint32_t*>(g) = h << 16;  // header 0: fold
    else
      g[1 + r] = (uint16_t)h;
    if (i + 1 == d)
      for (uint32_t t = r + 1; t < kGroup; ++t) g[1 + t] = 0xFFFF;
  }
}

// Wide rows, one block per row: classes in order, each from a group of its own.
__global__ void __launch_bounds__(kBlock) k_pack_wide(const uint32_t* __restrict__ rp, const int32_t* __restrict__ adj,
                                                      const uint32_t* __restrict__ ndeg,
                                                      const float2* __restrict__ tab_g,
                                                      const uint32_t* __restrict__ wide,
                                                      const uint32_t* __restrict__ wide_count,
                                                      const uint32_t* __restrict__ gs, uint16_t* __restrict__ packed) {
  constexpr uint32_t C = 4;
  __shared__ float2 tab[kDegBuckets];
  __shared__ uint32_t h[kClasses], first[kClasses], cur[kClasses];
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock) tab[t] = tab_g[t];
  __syncthreads();
  const uint32_t count = *wide_count;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t x = wide[i], b = rp[x], e = rp[x + 1];
    count_classes(b, e, adj, ndeg, tab, h);
    if (threadIdx.x == 0) {
      uint32_t g = gs[x];
      for (uint32_t c = 0; c < kClasses; ++c) {
        first[c] = g;
        cur[c] = 0;
        g += (h[c] + kGroup - 1) / kGroup;
      }
    }
    __syncthreads();
    for (uint64_t k0 = b; k0 < e; k0 += kBlock * C) {
      uint32_t v[C], d[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        const uint64_t k = k0 + j * kBlock + threadIdx.x;
        v[j] = k < e ? (uint32_t)adj[k] : 0u;
        d[j] = k < e ? ndeg[k] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        if (!d[j]) continue;
        const uint32_t c = vertex_class(v[j], d[j], tab), pos = atomicAdd(&cur[c], 1u);
        const uint32_t q = pos / kGroup, r = pos % kGroup, hv = hash16(v[j]);
        uint16_t* const g = packed + ((uint64_t)first[c] + q) * 8;
        if (r == 0)
          *reinterpret_cast<uint32_t*>(g) = (hv << 16) | class_header(c);
        else
          g[1 + r] = (uint16_t)hv;
      }
    }
    if (threadIdx.x < kClasses) {
      const uint32_t c = threadIdx.x, used = h[c] % kGroup;
      if (used)
        for (uint32_t t = used; t < kGroup; ++t)
          packed[((uint64_t)first[c] + h[c] / kGroup) * 8 + 1 + t] = 0xFFFF;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Planning
// ---------------------------------------------------------------------------

// Owners by the kernel that filters their edges:
//   wave       rows of at most kWaveRow entries and at most kWaveEdges edges:
//              one wave per owner, which also decides the survivors
//   workgroup  up to kSmallRow entries (or many edges): 256 threads, the fold
//              window alone
//   large      1024 threads, nine windows
constexpr uint32_t kWaveRow = 512;
constexpr uint32_t kWaveEdges = 256;
constexpr uint32_t kSmallRow = 2048;
constexpr uint32_t kSmallEdges = 256;  // edges per unit
constexpr uint32_t kLargeEdges = 768;

// Units of the workgroup and large filters (small from the front of funits,
// large from the back) and the wave list.  A unit's edges are capped so that
// a small graph still gives every workgroup slot several units.
__global__ void __launch_bounds__(kBlock) k_plan_filter(uint32_t n, const uint32_t* __restrict__ rb,
                                                        const uint32_t* __restrict__ re,
                                                        const uint32_t* __restrict__ cnt_u,
                                                        const uint64_t* __restrict__ work_u,
                                                        uint4* __restrict__ funits, uint32_t fcap, uint32_t ucap,
                                                        uint32_t* __restrict__ wl_b, uint32_t* __restrict__ wl_e,
                                                        uint32_t* __restrict__ wl_k, uint64_t* __restrict__ cnt) {
  constexpr uint32_t V = 4;  // vertices per thread per block iteration
  const uint64_t owned_all = count_total(cnt, kCntUEdges);
  if (owned_all > ucap) {  // asymmetric input: reported by the host, no unit is written
    if (blockIdx.x == 0 && threadIdx.x == 0) cnt[kCntOverflow] = owned_all;
    return;
  }
  const uint32_t cap_s = (uint32_t)min((uint64_t)kSmallEdges, max((uint64_t)32, owned_all / 8192));
  const uint32_t cap_l = (uint32_t)min((uint64_t)kLargeEdges, max((uint64_t)64, owned_all / 2048));
  unsigned long long* const ctr[3] = {(unsigned long long*)&cnt[kCntFUnits1], (unsigned long long*)&cnt[kCntFUnits2],
                                      (unsigned long long*)&cnt[kCntTiny]};
  const uint64_t tile = (uint64_t)kBlock * V;
  for (uint64_t base = (uint64_t)blockIdx.x * tile; base < n; base += (uint64_t)gridDim.x * tile) {  // block-uniform
    uint32_t owned[V], c1[V], c2[V], c3[V], per[V], start[V], stop[V];
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint64_t x = base + j * kBlock + threadIdx.x;
      owned[j] = x < n ? cnt_u[x] : 0u;
    }
    uint32_t need[3] = {0, 0, 0};
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint64_t x = base + j * kBlock + threadIdx.x;
      c1[j] = c2[j] = c3[j] = 0;
      per[j] = 1;
      start[j] = stop[j] = 0;
      if (owned[j]) {
        start[j] = rb[x];
        stop[j] = re[x];
        const uint32_t d = stop[j] - start[j];
        if (d <= kWaveRow && owned[j] <= kWaveEdges) {
          c3[j] = 1;
        } else {
          // long short rows: fewer edges per unit, at least 32
          const uint32_t cap = d <= kSmallRow ? cap_s : cap_l;
          const uint64_t target = (uint64_t)cap * (d <= kSmallRow ? 512 : 2048);
          const uint64_t avg = work_u[x] / owned[j] + 1, fit = target / avg;
          per[j] = fit >= cap ? cap : (fit < 32 ? 32u : (uint32_t)fit);
          const uint32_t c = (owned[j] + per[j] - 1) / per[j];
          if (d <= kSmallRow)
            c1[j] = c;
          else
            c2[j] = c;
        }
      }
      need[0] += c1[j];
      need[1] += c2[j];
      need[2] += c3[j];
    }
    block_reserve<3>(need, ctr);
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint32_t cu = c1[j] + c2[j];
      const uint64_t end = (uint64_t)start[j] + owned[j];
      for (uint32_t t = 0; t < cu; ++t) {
        const uint64_t j0 = (uint64_t)start[j] + (uint64_t)t * per[j];
        const uint64_t j1 = j0 + per[j] < end ? j0 + per[j] : end;
        const uint32_t at = c1[j] ? need[0] + t : fcap - 1 - (need[1] + t);
        funits[at] = make_uint4((uint32_t)j0, (uint32_t)j1, start[j], stop[j]);
      }
      if (c3[j]) {
        wl_b[need[2]] = start[j];
        wl_e[need[2]] = stop[j];
        wl_k[need[2]] = owned[j];
      }
      need[0] += c1[j];
      need[1] += c2[j];
      need[2] += c3[j];
    }
  }
}

// ---------------------------------------------------------------------------
// Filtering
// ---------------------------------------------------------------------------

// Sum over each team of 16 lanes, in all of them.
__device__ __forceinline__ uint32_t team_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, true);  // row_ror:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, true);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, true);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);
  return v;
}

constexpr uint32_t kTeam = 16;
constexpr uint32_t kTeamLoads = 4;  // groups per lane and round

// Filter shapes: 2^13 bits, the fold window, the fold window and eight class
// windows.
enum FilterKind { kFilterWave, kFilterFold, kFilterWindows };

// The absence bits of one group's seven elements in the top bits of a word,
// against a filter whose set bits are the absent elements.  An element costs
// four VALU instructions and one LDS read: address shift and mask, the word
// shifted by the element, and its low bit funnelled into the result.
template <int KIND>
__device__ __forceinline__ uint32_t group_absent(const uint4 v, const uint32_t* filt) {
  constexpr uint32_t mask = KIND == kFilterWave ? 0x3FCu : 0x1FFCu;
  const uint32_t base = KIND == kFilterWindows ? (v.x & 0x1Eu) << 12 : 0u;  // window (header >> 1) x 8 KB
  const char* const f = reinterpret_cast<const char*>(filt);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t lo[4], hi[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q) lo[q] = *reinterpret_cast<const uint32_t*>(f + (((w[q] >> 3) & mask) | base));
    hi[q] = *reinterpret_cast<const uint32_t*>(f + (((w[q] >> 19) & mask) | base));
  }
  uint32_t bits = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q) bits = __builtin_amdgcn_alignbit(lo[q] >> (w[q] & 31), bits, 1);
    bits = __builtin_amdgcn_alignbit(hi[q] >> ((w[q] >> 16) & 31), bits, 1);
  }
  return bits;
}

// Loads of a round: as many as reach `need` misses if an eighth of the
// elements hit, so that little is read past the decision.
__device__ __forceinline__ uint32_t round_loads(uint32_t need) {
  const uint32_t nl = (need + (need >> 3) + kTeam * kGroup - 1) / (kTeam * kGroup);
  return nl < kTeamLoads ? nl : kTeamLoads;
}

// One round of a team at group g: the misses found in the next `take`
// groups.  Lanes past them load the last one again (every address is valid,
// also a resting team's) and are left out of the count.
template <int KIND>
__device__ __forceinline__ uint32_t filter_round(uint32_t g, uint32_t take, const uint4* __restrict__ packed,
                                                 const uint32_t* filt) {
  const uint32_t tl = lane_id() & (kTeam - 1), last = take ? take - 1 : 0u;
  uint4 v[kTeamLoads];
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * kTeam < take)) break;
    v[j] = packed[g + min(j * kTeam + tl, last)];
  }
  uint32_t miss = 0;
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * kTeam < take)) break;
    const uint32_t bits = group_absent<KIND>(v[j], filt);
    miss += (uint32_t)__popc(j * kTeam + tl < take ? bits : 0u);
  }
  return team_sum(miss);
}

// Misses that make an edge (s = d(a), threshold c*) dissimilar; 0: decided
// without streaming, *survive says which way (true: by the exact kernels).
__device__ __forceinline__ uint32_t misses_needed(double eps, uint32_t s, uint32_t l, uint32_t* cstar, bool* survive) {
  *cstar = 0;
  *survive = true;
  if (s > kMaxThresholdRow) return 0;  // the reference's int32 wrap: counted in full
  const uint32_t c = min_common_threshold(predicate_rhs(eps, s, l), s);
  *cstar = c;
  if (c == 0) return 0;  // similar with any count
  if (c > s) {
    *survive = false;
    return 0;
  }
  return s - c + 1;
}

struct FilterArgs {
  uint32_t m;
  double eps;
  const uint32_t* rb;
  const uint32_t* src;
  const int32_t* adj;
  const uint32_t* gs;     // n + 1: first group of each row
  const uint4* packed;
  uint4* uedge;
  uint8_t* flag;
  uint64_t* cnt;
};

// Workgroup (LARGE = false) and large filters.  One unit = one owner and up
// to MAXE of its edges; each team of 16 lanes takes edges from the unit's
// cursor and streams their packed rows against the LDS filter.  Rejected
// edges get their flags; the survivors' records are moved to the front of
// the unit's range and become one unit of the exact kernels.
//
// The packed rows bound it by HBM reads: two 1024-thread workgroups of 80 KB
// share a CU (eight waves per SIMD, four 1 KB wave loads in flight each).
template <bool LARGE>
__global__ void __launch_bounds__(LARGE ? 1024 : 256, 8)
    k_filter_units(FilterArgs A, const uint4* __restrict__ funits, uint32_t fcap, uint4* __restrict__ eunits,
                   uint32_t ecap, uint32_t small_max_degree) {
  constexpr uint32_t T = LARGE ? 1024 : 256;
  constexpr uint32_t MAXE = LARGE ? kLargeEdges : kSmallEdges;
  constexpr uint32_t WORDS = LARGE ? 9 * kWindowWords16 : kWindowWords16;
  __shared__ __align__(16) uint32_t filt[WORDS];
  // the edges to stream, longest first: (first group, groups << 16 | misses
  // needed)
  __shared__ uint2 e_q[MAXE];
  __shared__ uint32_t s_surv[MAXE / 32], s_part[T / kWave], s_hist[32];
  __shared__ uint32_t s_unit, s_cursor;
  const uint32_t lane = lane_id(), tl = lane & (kTeam - 1), tid = threadIdx.x;
  const uint64_t nunits = A.cnt[LARGE ? kCntFUnits2 : kCntFUnits1];
  unsigned long long* const queue = (unsigned long long*)&A.cnt[LARGE ? kCntFQueue2 : kCntFQueue1];
  // the first unit is the block's own, the others come from the queue, one
  // ahead (atomics on one word take about 12 ns each, one after the other)
  uint32_t streamed = 0, rounds = 0, nxt = blockIdx.x;
  for (;;) {
    if (tid == 0) {
      s_unit = nxt;
      s_cursor = 0;
      if (nxt < nunits) nxt = nunits > gridDim.x ? gridDim.x + (uint32_t)atomicAdd(queue, 1ull) : kNone;
    }
    __syncthreads();
    const uint32_t u = s_unit;
    if (u >= nunits) break;
    const uint4 un = funits[LARGE ? fcap - 1 - u : u];
    const uint32_t ne = un.y - un.x, bb = un.z, l = un.w - un.z;
    const bool mine = tid < ne && tid < MAXE;
    uint4 ed = make_uint4(kNone, kNone, 0, 0);  // (entry, reverse entry, a, d(a))
    if (mine) ed = A.uedge[un.x + tid];
    const uint32_t b = A.src[bb];
    // every element absent but the padding
    uint4* const f4 = reinterpret_cast<uint4*>(filt);
    for (uint32_t t = tid; t < WORDS / 4; t += T)
      f4[t] = make_uint4(~0u, ~0u, ~0u, t % (kWindowWords16 / 4) == kWindowWords16 / 4 - 1 ? 0x7FFFFFFFu : ~0u);
    if (tid < MAXE / 32) s_surv[tid] = 0;
    if (tid < 32) s_hist[tid] = 0;
    uint32_t g0 = 0, g1 = 0;
    if (mine) {
      g0 = A.gs[ed.z];
      g1 = A.gs[ed.z + 1];
    }
    const uint32_t bg0 = A.gs[b], bg1 = A.gs[b + 1];
    __syncthreads();
    for (uint32_t i = bg0 + tid; i < bg1; i += T) {
      const uint4 v = A.packed[i];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      const uint32_t win = LARGE ? ((v.x & 0x1Eu) >> 1) * kWindowWords16 : 0u;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q == 0) continue;  // the header
        const uint32_t h = q & 1 ? w[q >> 1] >> 16 : w[q >> 1] & 0xFFFFu;
        if (LARGE) atomicAnd(&filt[win + (h >> 5)], ~(1u << (h & 31)));
        atomicAnd(&filt[h >> 5], ~(1u << (h & 31)));
      }
    }
    // Edges in order of the misses they need (two buckets per power of two),
    // most first: the teams of a wave then take edges of about the same
    // length, end their rounds and fetch their next edges together, and the
    // longest edges do not start last.
    bool keep = false;  // survives
    uint32_t need0 = 0, rank = 0, slot = 0;
    if (mine) {
      uint32_t cstar;
      need0 = misses_needed(A.eps, ed.w, l, &cstar, &keep);
    }
    const uint32_t lg = need0 ? 31 - __clz(need0) : 0u;  // need0 < 2^16
    const uint32_t bucket = 31 - (lg ? lg * 2 + ((need0 >> (lg - 1)) & 1) : 0u);
    if (need0) {
      keep = false;
      rank = atomicAdd(&s_hist[bucket], 1u);
    }
    __syncthreads();
    const uint32_t incl = wave_incl_scan(lane < 32 ? s_hist[lane] : 0u);
    const uint32_t todo = __builtin_amdgcn_readlane(incl, 31);
    slot = (uint32_t)__shfl((int)incl, (int)bucket) - s_hist[bucket] + rank;
    if (need0) e_q[slot] = make_uint2(g0, ((g1 - g0) << 16) | need0);
    __syncthreads();
    // ---- stream
    bool act = false, out = false;  // this team has an edge; the cursor is at its end
    uint32_t e = 0, g = bg0, ge = 0, need = 0;
    for (;;) {
      if (!act && !out) {
        uint32_t t = 0;
        if (tl == 0) t = atomicAdd(&s_cursor, 1u);
        t = (uint32_t)__shfl((int)t, (int)(lane & ~(kTeam - 1)));
        if (t < todo) {
          const uint2 q = e_q[t];
          e = t;
          g = q.x;
          ge = q.x + (q.y >> 16);
          need = q.y & 0xFFFFu;
          act = true;
        } else {
          out = true;
        }
      }
      if (!__ballot(act)) break;
      const uint32_t take = act ? min(round_loads(need) * kTeam, ge - g) : 0u;
      const uint32_t miss = filter_round<LARGE ? kFilterWindows : kFilterFold>(g, take, A.packed, filt);
      if (act) {
        streamed += take;
        ++rounds;
        g += take;
        if (miss >= need) {
          act = false;
        } else {
          need -= miss;
          if (g >= ge) {
            act = false;
            if (tl == 0) atomicOr(&s_surv[e >> 5], 1u << (e & 31));
          }
        }
      }
    }
    __syncthreads();
    // ---- results, and the survivors' records to the front of the range
    if (need0) keep = (s_surv[slot >> 5] >> (slot & 31)) & 1u;
    if (mine && !keep) {
      if (ed.x < A.m) A.flag[ed.x] = kFlagN;
      if (ed.y < A.m) A.flag[ed.y] = kFlagN;
    }
    const uint64_t km = __ballot(keep);
    if (lane == 0) s_part[tid / kWave] = (uint32_t)__popcll(km);
    uint4 rec = make_uint4(0, 0, 0, 0);
    if (keep) rec = A.uedge[un.x + tid];
    __syncthreads();  // also: every record that moves has been read
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < T / kWave; ++w) {
      const uint32_t c = s_part[w];
      before += w < tid / kWave ? c : 0u;
      total += c;
    }
    if (total) {
      if (keep) A.uedge[un.x + before + (uint32_t)__popcll(km & lanemask_lt(lane))] = rec;
      if (tid == 0) {
        const bool small = l <= small_max_degree;
        const uint32_t at = (uint32_t)atomicAdd((unsigned long long*)&A.cnt[small ? kCntUnits1 : kCntUnits2], 1ull);
        eunits[small ? at : ecap - 1 - at] = make_uint4(un.x, un.x + total, un.z, un.w);
      }
    }
  }
  const uint64_t elements = tl == 0 ? (uint64_t)streamed * kGroup : 0ull;
  count_add<3>(A.cnt, {kCntProbes, kCntLoaded, kCntClaims}, {elements, elements, tl == 0 ? rounds : 0u});
}

// Owners with short rows, one wave each: the row in LDS (sorted, for the
// exact counts) and a 2^13-bit filter of it; 64 edges at a time, four teams.
// Survivors are counted by binary search of the short row's elements in the
// owner's row, one team per edge, so nothing is left to the exact kernels.
__global__ void __launch_bounds__(kBlock, 8)
    k_filter_wave(FilterArgs A, const uint32_t* __restrict__ wl_b, const uint32_t* __restrict__ wl_e,
                  const uint32_t* __restrict__ wl_k) {
  constexpr uint32_t W = kBlock / kWave;
  __shared__ __align__(16) uint32_t s_filt[W][256];
  __shared__ int32_t s_row[W][kWaveRow];
  __shared__ uint2 s_q[W][kWave];
  __shared__ uint32_t s_list[W][kWave];
  const uint32_t lane = lane_id(), tl = lane & (kTeam - 1), wv = threadIdx.x / kWave;
  uint32_t* const filt = s_filt[wv];
  int32_t* const row = s_row[wv];
  uint2* const e_q = s_q[wv];
  uint32_t* const list = s_list[wv];
  const uint32_t count = (uint32_t)A.cnt[kCntTiny];
  const uint32_t waves = gridDim.x * W;
  uint32_t streamed = 0, rounds = 0, probed = 0;
  for (uint32_t idx = blockIdx.x * W + wv; idx < count; idx += waves) {
    const uint32_t bb = __builtin_amdgcn_readfirstlane(wl_b[idx]), be = __builtin_amdgcn_readfirstlane(wl_e[idx]);
    const uint32_t owned = __builtin_amdgcn_readfirstlane(wl_k[idx]), l = be - bb;
    uint4 ed = make_uint4(kNone, kNone, 0, 0);
    if (lane < owned) ed = A.uedge[bb + lane];
    // the row, padded to a power of two, and its filter
    uint32_t P = kWave;
    while (P < l) P <<= 1;
    reinterpret_cast<uint4*>(filt)[lane] = make_uint4(~0u, ~0u, ~0u, lane == kWave - 1 ? 0x7FFFFFFFu : ~0u);
    for (uint32_t t = lane; t < P; t += kWave) row[t] = t < l ? A.adj[bb + t] : 0x7FFFFFFF;
    wave_lds_sync();
    for (uint32_t t = lane; t < l; t += kWave) {
      const uint32_t h = hash16((uint32_t)row[t]);
      atomicAnd(&filt[(h >> 5) & 255u], ~(1u << (h & 31)));
    }
    for (uint32_t base = 0; base < owned; base += kWave) {
      const uint32_t ne = min(owned - base, (uint32_t)kWave);
      if (base) {
        ed = make_uint4(kNone, kNone, 0, 0);
        if (lane < ne) ed = A.uedge[bb + base + lane];
      }
      uint32_t cstar = 0;
      bool survive = false;
      uint2 q = make_uint2(0, 0);
      if (lane < ne) {
        const uint32_t g0 = A.gs[ed.z], g1 = A.gs[ed.z + 1];
        const uint32_t need = misses_needed(A.eps, ed.w, l, &cstar, &survive);
        q = make_uint2(g0, need ? ((g1 - g0) << 16) | need : 0u);
        if (need) survive = false;
      }
      e_q[lane] = q;
      wave_lds_sync();
      // ---- filter: teams take the edges in order
      bool act = false;
      uint32_t e = 0, g = 0, ge = 0, need = 0, next = 0;
      for (;;) {
        const uint64_t idle = __ballot(!act && tl == 0);
        if (idle && next < ne) {
          if (!act) {
            const uint32_t t = next + (uint32_t)__popcll(idle & lanemask_lt(lane & ~(kTeam - 1)));
            if (t < ne) {
              const uint2 p = e_q[t];
              e = t;
              g = p.x;
              ge = p.x + (p.y >> 16);
              need = p.y & 0xFFFFu;
              act = need != 0;
            }
          }
          next += (uint32_t)__popcll(idle);
        }
        if (!__ballot(act)) {
          if (next >= ne) break;
          continue;
        }
        const uint32_t take = act ? min(round_loads(need) * kTeam, ge - g) : 0u;
        const uint32_t miss = filter_round<kFilterWave>(g, take, A.packed, filt);
        if (act) {
          streamed += take;
          ++rounds;
          g += take;
          if (miss >= need) {
            act = false;
          } else {
            need -= miss;
            if (g >= ge) {
              act = false;
              if (tl == 0) e_q[e].y = kNone;  // survives
            }
          }
        }
      }
      wave_lds_sync();
      if (lane < ne && e_q[lane].y == kNone) survive = true;
      // ---- exact counts of the survivors
      bool sim = false;
      uint64_t sm = __ballot(survive);
      if (sm) {
        wave_lds_sync();
        if (survive) {
          e_q[lane] = make_uint2(A.rb[ed.z], (cstar << 16) | ed.w);  // d(a) <= l <= 512
          list[(uint32_t)__popcll(sm & lanemask_lt(lane))] = lane;
        }
        wave_lds_sync();
        const uint32_t ns = (uint32_t)__popcll(sm);
        uint32_t pos = 0, end = 0, hits = 0, cs = 0;
        act = false;
        next = 0;
        for (;;) {
          const uint64_t idle = __ballot(!act && tl == 0);
          if (idle && next < ns) {
            if (!act) {
              const uint32_t t = next + (uint32_t)__popcll(idle & lanemask_lt(lane & ~(kTeam - 1)));
              if (t < ns) {
                e = list[t];
                const uint2 p = e_q[e];
                pos = p.x;
                end = p.x + (p.y & 0xFFFFu);
                cs = p.y >> 16;
                hits = 0;
                act = cs != 0;  // c* = 0: similar with any count
                if (!act && tl == 0) e_q[e].y = kNone;
              }
            }
            next += (uint32_t)__popcll(idle);
          }
          if (!__ballot(act)) {
            if (next >= ns) break;
            continue;
          }
          int32_t x[4];
          uint32_t at[4];
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t k = j * kTeam + tl;
            x[j] = act && k < end - pos ? A.adj[pos + k] : -1;
            at[j] = 0;
          }
          for (uint32_t half = P >> 1; half; half >>= 1) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) at[j] += row[at[j] + half - 1] < x[j] ? half : 0u;
          }
          uint32_t h = 0;
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) h += row[at[j]] == x[j] ? 1u : 0u;
          h = team_sum(h);
          if (act) {
            const uint32_t took = min(4 * kTeam, end - pos);
            pos += took;
            hits += h;
            probed += took;
            if (hits >= cs) {
              act = false;
              if (tl == 0) e_q[e].y = kNone;  // similar
            } else if (hits + (end - pos) < cs) {
              act = false;
            }
          }
        }
        wave_lds_sync();
        sim = survive && e_q[lane].y == kNone;
      }
      if (lane < ne) {
        const uint8_t f = sim ? kFlagY : kFlagN;
        if (ed.x < A.m) A.flag[ed.x] = f;
        if (ed.y < A.m) A.flag[ed.y] = f;
      }
      wave_lds_sync();  // e_q is rewritten by the next batch
    }
    wave_lds_sync();
  }
  const uint64_t elements = tl == 0 ? (uint64_t)streamed * kGroup + probed : 0ull;
  count_add<3>(A.cnt, {kCntProbes, kCntLoaded, kCntClaims}, {elements, elements, tl == 0 ? rounds : 0u});
}

// Temporary memory of build_packed_rows.
struct PackScratch {
  size_t mass, tab, groups, wide, wide_count, scan, bytes, scan_bytes;
};

PackScratch pack_scratch(uint32_t n, uint32_t m) {
  PackScratch s;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) / 256 * 256;
    return o;
  };
  s.scan_bytes = 0;
  (void)hipcub::DeviceScan::ExclusiveSum(nullptr, s.scan_bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr, n + 1);
  s.mass = take(kDegBuckets * 8);
  s.tab = take(kDegBuckets * sizeof(float2));
  s.groups = take(((size_t)n + 1) * 4);
  s.wide = take(((size_t)m / kWideRow + 1) * 4);
  s.wide_count = take(4);
  s.scan = take(s.scan_bytes);
  s.bytes = off;
  return s;
}

}  // namespace

// At most 6 padding elements per narrow row and per class of a wide row.
uint64_t packed_row_groups(uint64_t n, uint64_t m) {
  return (m + 6 * std::min(n, m)) / kGroup + kClasses * (m / kWideRow) + 1;
}

hipError_t build_packed_rows(sgc_dgraph* g, hipStream_t s) {
  if (!g->m || !g->mirror || !g->ndeg) return hipSuccess;
  const uint32_t n = g->n, m = g->m;
  const PackScratch L = pack_scratch(n, m);
  char* mem = nullptr;
  if (hipMalloc(&g->gs, ((size_t)n + 1) * 4) != hipSuccess ||
      hipMalloc(&g->packed, packed_row_groups(n, m) * sizeof(uint4)) != hipSuccess ||
      hipMalloc(&mem, L.bytes) != hipSuccess) {
    (void)hipGetLastError();  // no room: every edge goes to the exact kernels
    if (g->gs) (void)hipFree(g->gs);
    if (g->packed) (void)hipFree(g->packed);
    g->gs = nullptr;
    g->packed = nullptr;
    return hipSuccess;
  }
  unsigned long long* mass = (unsigned long long*)(mem + L.mass);
  float2* tab = (float2*)(mem + L.tab);
  uint32_t* groups = (uint32_t*)(mem + L.groups);
  uint32_t* wide = (uint32_t*)(mem + L.wide);
  uint32_t* wide_count = (uint32_t*)(mem + L.wide_count);
  uint16_t* packed = (uint16_t*)g->packed;
  k_degree_clear<<<1, kDegBuckets, 0, s>>>(mass, wide_count);
  k_degree_mass<<<std::min(grid_for(n, kBlock), 512u), kBlock, 0, s>>>(n, g->row_ptr, mass);
  k_degree_table<<<1, kDegBuckets, 0, s>>>(mass, tab);
  k_pack_count<<<grid_for((uint64_t)n + 1, kBlock), kBlock, 0, s>>>(n, g->row_ptr, groups, wide, wide_count);
  const uint32_t wide_grid = grid_for(m / kWideRow + 1, 1);
  k_wide_count<<<wide_grid, kBlock, 0, s>>>(g->row_ptr, g->adj, g->ndeg, tab, wide, wide_count, groups);
  size_t scan_bytes = L.scan_bytes;
  hipError_t e = hipcub::DeviceScan::ExclusiveSum(mem + L.scan, scan_bytes, groups, g->gs, n + 1, s);
  k_pack_narrow<<<grid_for(m, kBlock), kBlock, 0, s>>>(m, g->row_ptr, g->src, g->adj, g->gs, packed);
  k_pack_wide<<<wide_grid, kBlock, 0, s>>>(g->row_ptr, g->adj, g->ndeg, tab, wide, wide_count, g->gs, packed);
  if (e == hipSuccess) e = hipGetLastError();
  const hipError_t w = hipStreamSynchronize(s);
  (void)hipFree(mem);
  return e != hipSuccess ? e : w;
}

bool filter_stage(const sgc_dgraph* g, ScanParams p) {
  return g->packed && g->mirror && !p.prune && g->tuning.hash_tables != 0;
}

void launch_plan_filter(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  // the lists share arrays that the core pass initialises later
  k_plan_filter<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, g->row_begin, g->row_end, b.cnt_u, b.work_u, b.units,
                                                          b.ucap / 2, b.ucap, (uint32_t*)b.label, (uint32_t*)b.parent,
                                                          (uint32_t*)b.lo, b.cnt);
}

void launch_filter(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s) {
  const uint32_t cus = (uint32_t)(cu_count > 0 ? cu_count : 256);
  const uint32_t fcap = b.ucap / 2, ecap = b.ucap - fcap;
  const FilterArgs A{g->m, p.eps, g->row_begin, g->src, g->adj, g->gs, g->packed, b.uedge, b.flag, b.cnt};
  k_filter_units<true><<<cus * 2, 1024, 0, s>>>(A, b.units, fcap, b.units + fcap, ecap, g->tuning.small_max_degree);
  k_filter_units<false><<<cus * 8, 256, 0, s>>>(A, b.units, fcap, b.units + fcap, ecap, g->tuning.small_max_degree);
  const uint64_t want = ((uint64_t)g->n + kBlock / kWave - 1) / (kBlock / kWave), cap = (uint64_t)cus * 8;
  k_filter_wave<<<(uint32_t)(want < cap ? want : cap), kBlock, 0, s>>>(A, (const uint32_t*)b.label,
                                                                       (const uint32_t*)b.parent,
                                                                       (const uint32_t*)b.lo);
}

}  // namespace sgc
