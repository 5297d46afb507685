// Filter stages of the similarity phase for resident graphs.
//
// Almost every edge that the degree-only test leaves undecided is dissimilar,
// and with room to spare: on R-MAT the common neighbours of half of them are
// under half of the threshold c*.  Two stages reject such edges from compact
// copies of the rows made at upload; the few others go to the exact kernels.
// An edge (a, b), a the short endpoint, is dissimilar once d(a) - c* + 1
// elements of N(a) are known to miss N(b), and every miss below is certain:
// the rejections are exact, only hits may be false.
//
// Bitmaps.  Row x as a bit set of M(x) = 4 to 8 times d(x) bits (a power of
// two), element v at bit hash(v) mod M: under a byte an entry.  The owner's
// row is built in LDS at the largest M its edges need and folded to the
// smaller ones, so an edge is ANDed word by word at its own M: 32 bits cost
// three instructions, without bank conflicts.  A clear bit of the owner's
// under a set bit of a's is a miss; elements of N(a) that share a bit count
// once and a dense owner hides misses, so about
// k (1 - e^(-1/k)) e^(-r/k) of the misses show (k = M / d(a), r = d(b) /
// d(a)): enough for eps >= 0.35 or so.  Rows of at most kFineRow entries also
// have one of 4 M bits, enough for eps >= 0.2.
//
// Hash groups, for long rows at low eps.  A vertex has a 16-bit hash and one
// of 16 classes by its degree, cut so that each class holds a sixteenth of
// all entries, rarest vertices first.  A row is a list of 16-byte groups: a
// 16-bit header and seven hashes.  In wide rows (kWideRow entries or more)
// every group holds one class, named in its header, rarest class first; in
// narrow rows the classes are mixed and the header says "fold".  That is 2.3
// to 2.4 bytes an entry.  The owner's row is a bit set in LDS: one window of
// 2^16 bits per pair of classes and one fold window over all of them.  Rare
// neighbours first means misses first: 10-20 % fewer elements than in id
// order (CPU replay of R-MAT-20 and 22).
//
// Similarity phase on R-MAT-24 (2.6e8 edges), exact kernels alone -> with the
// filters: eps 0.2 150 -> 67 ms, 0.3 119 -> 46, 0.4 80 -> 24, 0.6 32 -> 11,
// 0.8 22 -> 8.  (Hash groups alone: 67, 51, 35, 17, 11.)  The build takes
// 3.8 ms of the upload.  Lower eps: kHashEps.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.h"
#include "device_util.h"

namespace sgc {

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kGroup = 7;            // elements per hash group
constexpr uint32_t kClasses = 16;
constexpr uint32_t kMinRow = 16;          // shorter rows have no compact copy
constexpr uint32_t kWideRow = 512;        // rows of at least this many entries are ordered by class
constexpr uint32_t kFineRow = 1024;       // rows up to this length have a fine bitmap
constexpr uint32_t kWindowWords16 = 2048;   // 2^16 bits
constexpr uint32_t kDegBuckets = 512;       // degree buckets: 16 per power of two

// Two rounds of multiply and shift (odd constants); bitmaps use the low bits,
// hash groups the high ones.
__device__ __forceinline__ uint32_t vertex_hash(uint32_t x) {
  x *= 0x9E3779B1u;
  x ^= x >> 15;
  x *= 0x85EBCA77u;
  return x ^ (x >> 13);
}

// 0xFFFF is the padding element, whose bit is set in every filter.
__device__ __forceinline__ uint32_t group_element(uint32_t hash) {
  const uint32_t h = hash >> 16;
  return h < 0xFFFFu ? h : 0xFFFEu;
}

// Group headers: 0 = fold, else 2 + class; header >> 1 is the filter window
// (0 fold, 1..8 pairs of classes).
__device__ __forceinline__ uint32_t class_header(uint32_t c) { return 2 + c; }

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

// ---- where the copies of a row [b, b + d) lie, for d >= kMinRow: all from
// its first entry, so an edge record needs nothing else to find them.
//   bitmap: M(d) = max(128, 4 d rounded up to a power of two) <= 8 d bits at
//     16-byte word coarse_at(b) of the coarse array (16 bytes per 16
//     entries); M / 8 is at most d rounded down to a multiple of 16, so rows
//     do not overlap
//   fine bitmap: 4 M(d) bits at 4 coarse_at(b) of the fine array
//   groups: at b / 4, row_groups(d) of them (at most (d - 3) / 4)
__device__ __forceinline__ uint32_t coarse_words(uint32_t d) {  // of 16 bytes
  return d <= 32 ? 1u : 1u << (32 - __clz(d - 1) - 5);          // 2^ceil(log2 d) * 4 / 128
}
__device__ __forceinline__ uint32_t coarse_at(uint32_t b) { return (uint32_t)(((uint64_t)b + 15) >> 4); }
__device__ __forceinline__ uint32_t row_groups(uint32_t d) {
  return d < kWideRow ? (d + kGroup - 1) / kGroup : d / kGroup + kClasses;
}

// ---------------------------------------------------------------------------
// Building the copies
// ---------------------------------------------------------------------------

struct PackArgs {
  uint32_t n;
  const uint32_t* rp;
  const int32_t* adj;
  const uint32_t* ndeg;
  uint16_t* groups;  // 8 per group
  uint4* coarse;
  uint4* fine;
  unsigned long long* mass;  // entries per degree bucket
  float2* tab;
  uint32_t* narrow;  // rows of kMinRow .. kWideRow - 1 entries
  uint32_t* wide;    // longer ones
  unsigned long long* counts;  // of the two lists
};

__global__ void __launch_bounds__(kDegBuckets) k_pack_clear(PackArgs A) {
  A.mass[threadIdx.x] = 0;
  if (threadIdx.x < 2) A.counts[threadIdx.x * 16] = 0;
}

// Entries per degree bucket, and the two row lists.
__global__ void __launch_bounds__(kBlock) k_pack_lists(PackArgs A) {
  __shared__ unsigned long long h[kDegBuckets];
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock) h[t] = 0;
  __syncthreads();
  constexpr uint32_t V = 8;
  unsigned long long* const ctr[2] = {&A.counts[0], &A.counts[16]};
  const uint64_t tile = (uint64_t)kBlock * V;
  for (uint64_t base = (uint64_t)blockIdx.x * tile; base < A.n; base += (uint64_t)gridDim.x * tile) {
    uint32_t d[V], need[2] = {0, 0};
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint64_t x = base + j * kBlock + threadIdx.x;
      d[j] = x < A.n ? A.rp[x + 1] - A.rp[x] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      if (d[j]) atomicAdd(&h[degree_bucket(d[j])], (unsigned long long)d[j]);
      need[0] += d[j] >= kMinRow && d[j] < kWideRow;
      need[1] += d[j] >= kWideRow;
    }
    block_reserve<2>(need, ctr);
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint32_t x = (uint32_t)(base + j * kBlock + threadIdx.x);
      if (d[j] >= kWideRow)
        A.wide[need[1]++] = x;
      else if (d[j] >= kMinRow)
        A.narrow[need[0]++] = x;
    }
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock)
    if (h[t]) atomicAdd(&A.mass[t], h[t]);
}

__global__ void __launch_bounds__(kDegBuckets) k_pack_table(PackArgs A) {
  __shared__ unsigned long long s[kDegBuckets];
  const uint32_t t = threadIdx.x;
  const unsigned long long own = A.mass[t];
  s[t] = own;
  __syncthreads();
  for (uint32_t off = 1; off < kDegBuckets; off <<= 1) {
    const unsigned long long v = t >= off ? s[t - off] : 0ull;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  const double total = (double)(s[kDegBuckets - 1] ? s[kDegBuckets - 1] : 1ull);
  A.tab[t] = make_float2((float)(kClasses * ((double)(s[t] - own) / total)), (float)(kClasses * ((double)own / total)));
}

// Narrow rows, one wave each: element i of the row is element i % 7 of its
// group i / 7; the fine bitmap is collected in LDS and folded to the coarse.
__global__ void __launch_bounds__(kBlock) k_pack_narrow(PackArgs A) {
  __shared__ __align__(16) uint32_t s_bits[kBlock / kWave][256];  // 4 M(511) = 8192 bits
  const uint32_t lane = lane_id(), wv = threadIdx.x / kWave;
  uint32_t* const bits = s_bits[wv];
  uint4* const bits4 = reinterpret_cast<uint4*>(bits);
  const uint32_t count = (uint32_t)A.counts[0], waves = gridDim.x * (kBlock / kWave);
  for (uint32_t i = blockIdx.x * (kBlock / kWave) + wv; i < count; i += waves) {
    const uint32_t x = __builtin_amdgcn_readfirstlane(A.narrow[i]);
    const uint32_t b = __builtin_amdgcn_readfirstlane(A.rp[x]), d = __builtin_amdgcn_readfirstlane(A.rp[x + 1]) - b;
    const uint32_t cw = coarse_words(d), mask = cw * 512 - 1;  // 4 * 128 cw bits
    bits4[lane] = make_uint4(0, 0, 0, 0);
    wave_lds_sync();
    for (uint32_t t = lane; t < d; t += kWave) {
      const uint32_t h = vertex_hash((uint32_t)A.adj[b + t]);
      atomicOr(&bits[(h & mask) >> 5], 1u << (h & 31));
      const uint32_t q = t / kGroup, r = t % kGroup, e = group_element(h);
      uint16_t* const g = A.groups + ((uint64_t)(b / 4) + q) * 8;
      if (r == 0)
        *reinterpret_cast<uint32_t*>(g) = e << 16;  // header 0: fold
      else
        g[1 + r] = (uint16_t)e;
      if (t + 1 == d)
        for (uint32_t p = r + 1; p < kGroup; ++p) g[1 + p] = 0xFFFF;
    }
    wave_lds_sync();
    const uint32_t at = coarse_at(b);
    if (lane < 4 * cw) A.fine[(uint64_t)at * 4 + lane] = bits4[lane];
    if (lane < cw) {
      uint4 v = bits4[lane];
#pragma unroll
      for (uint32_t q = 1; q < 4; ++q) {
        const uint4 o = bits4[q * cw + lane];
        v.x |= o.x, v.y |= o.y, v.z |= o.z, v.w |= o.w;
      }
      A.coarse[at + lane] = v;
    }
    wave_lds_sync();
  }
}

// Wide rows, one block each: the groups by class (each class from a group of
// its own, the groups left over all padding), the bitmaps as above.  Rows
// beyond kMaxThresholdRow are never streamed: no bitmap.  Every entry goes in,
// whatever its degree: input that is not symmetric has neighbours without a
// row, and one that is left out would count as a certain miss.
__global__ void __launch_bounds__(kBlock) k_pack_wide(PackArgs A) {
  constexpr uint32_t C = 4;
  __shared__ __align__(16) uint32_t bits[8192];  // M(46338) = 2^18 bits; 4 M(1024) = 2^14
  __shared__ float2 tab[kDegBuckets];
  __shared__ uint32_t h[kClasses], first[kClasses + 1], cur[kClasses];
  uint4* const bits4 = reinterpret_cast<uint4*>(bits);
  for (uint32_t t = threadIdx.x; t < kDegBuckets; t += kBlock) tab[t] = A.tab[t];
  const uint32_t count = (uint32_t)A.counts[16];
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t x = A.wide[i], b = A.rp[x], d = A.rp[x + 1] - b, g0 = b / 4;
    const bool fine = d <= kFineRow, coarse = d <= kMaxThresholdRow;
    const uint32_t cw = coarse ? coarse_words(d) : 0u, words = fine ? 4 * cw : cw, mask = words * 128 - 1;
    if (threadIdx.x < kClasses) h[threadIdx.x] = cur[threadIdx.x] = 0;
    for (uint32_t t = threadIdx.x; t < words; t += kBlock) bits4[t] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    for (uint32_t t0 = 0; t0 < d; t0 += kBlock * C) {
      uint32_t v[C], dv[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        const uint32_t t = t0 + j * kBlock + threadIdx.x;
        v[j] = t < d ? (uint32_t)A.adj[b + t] : 0u;
        dv[j] = t < d ? A.ndeg[b + t] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        if (t0 + j * kBlock + threadIdx.x >= d) continue;
        atomicAdd(&h[vertex_class(v[j], dv[j], tab)], 1u);
        if (coarse) {
          const uint32_t hv = vertex_hash(v[j]);
          atomicOr(&bits[(hv & mask) >> 5], 1u << (hv & 31));
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t g = g0;
      for (uint32_t c = 0; c < kClasses; ++c) {
        first[c] = g;
        g += (h[c] + kGroup - 1) / kGroup;
      }
      first[kClasses] = g;
    }
    const uint32_t at = coarse_at(b);
    if (fine)
      for (uint32_t t = threadIdx.x; t < 4 * cw; t += kBlock) A.fine[(uint64_t)at * 4 + t] = bits4[t];
    for (uint32_t t = threadIdx.x; t < cw; t += kBlock) {
      uint4 v = bits4[t];
      if (fine)
        for (uint32_t q = 1; q < 4; ++q) {
          const uint4 o = bits4[q * cw + t];
          v.x |= o.x, v.y |= o.y, v.z |= o.z, v.w |= o.w;
        }
      A.coarse[at + t] = v;
    }
    __syncthreads();
    for (uint32_t t0 = 0; t0 < d; t0 += kBlock * C) {
      uint32_t v[C], dv[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        const uint32_t t = t0 + j * kBlock + threadIdx.x;
        v[j] = t < d ? (uint32_t)A.adj[b + t] : 0u;
        dv[j] = t < d ? A.ndeg[b + t] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        if (t0 + j * kBlock + threadIdx.x >= d) continue;
        const uint32_t c = vertex_class(v[j], dv[j], tab), pos = atomicAdd(&cur[c], 1u);
        const uint32_t q = pos / kGroup, r = pos % kGroup, e = group_element(vertex_hash(v[j]));
        uint16_t* const g = A.groups + ((uint64_t)first[c] + q) * 8;
        if (r == 0)
          *reinterpret_cast<uint32_t*>(g) = (e << 16) | class_header(c);
        else
          g[1 + r] = (uint16_t)e;
      }
    }
    if (threadIdx.x < kClasses) {
      const uint32_t c = threadIdx.x, used = h[c] % kGroup;
      if (used)
        for (uint32_t t = used; t < kGroup; ++t)
          A.groups[((uint64_t)first[c] + h[c] / kGroup) * 8 + 1 + t] = 0xFFFF;
    }
    for (uint32_t g = first[kClasses] + threadIdx.x; g < g0 + row_groups(d); g += kBlock)
      reinterpret_cast<uint4*>(A.groups)[g] = make_uint4(0xFFFF0000u, ~0u, ~0u, ~0u);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Planning
// ---------------------------------------------------------------------------

// Owners by the kernel that takes their edges first:
//   wave       rows of at most kWaveRow entries and at most kWaveEdges edges:
//              one wave per owner, which also decides the survivors
//   workgroup  up to kSmallRow entries (or many edges): 256 threads
//   large      1024 threads
constexpr uint32_t kWaveRow = 256;
constexpr uint32_t kXcds = 8;  // blocks go to the XCDs in turn
constexpr uint32_t kWaveEdges = 256;
constexpr uint32_t kSmallRow = 1024;
constexpr uint32_t kSmallEdges = 256;  // edges per unit
constexpr uint32_t kLargeEdges = 768;
// Below this eps the coarse bitmaps of long rows rarely show enough misses:
// the large owners' edges go to the hash filter at once.  R-MAT-24, with the
// bitmaps first / without: eps 0.25 63.1 / 58.0 ms, eps 0.3 46.4 / 50.6.
constexpr double kCoarseEps = 0.27;
// Below this one most edges are similar and the exact kernels see that after
// a few elements, where the hash filter reads the whole row to no end: there
// the large owners' edges pass the bitmap kernel (which rejects next to
// nothing) and are counted.  Similarity phase, with the hash filter / without:
// R-MAT-22 eps 0.01 31.4 / 19.8 ms, 0.02 39.7 / 29.2, 0.03 48.4 / 40.6,
// 0.05 49.0 / 54.5; R-MAT-24 eps 0.01 223 / 145, 0.02 323 / 271, 0.03 336 / 359,
// 0.05 246 / 351.
constexpr double kHashEps = 0.025;

// Pieces an owner's edges are cut into for the wave filter, beyond its first
// (row begin and end, first edge, edges): at most one for every 32 owned
// edges, so under an eighth of the quarter of the unit array they have.  A
// whole owner is a chain of waits of up to 256 edges, and with few owners the
// longest chains are the kernel: pieces are sized for kWavePieces of them, two
// to a wave slot.  Planted communities with 0.7 / 1.4 / 3.4 million entries,
// similarity phase: 227 / 286 / 722 us whole, 161 / 183 / 610 in pieces.
// Graphs of kPieceEntries and more have owners enough (8.1 million: 981 and
// 1006), and the registers the piece costs slow them (R-MAT-22 shuffled 1.65 ->
// 1.72 ms).
constexpr uint32_t kWavePieces = 12288;
constexpr uint32_t kPieceEntries = 1u << 22;
__host__ __device__ __forceinline__ uint4* wave_pieces(uint4* funits, uint32_t fcap) { return funits + fcap / 2; }

// Units of the workgroup and large filters (small from the front of funits,
// large from the back) and the wave list.  A unit's edges are capped so that
// a small graph still gives every workgroup slot several units; below 96
// edges a unit's row load and empty lanes cost more than the balance gives
// (at least 32 / 96 edges: R-MAT-14 177 / 151 us, R-MAT-16 250 / 246).
__global__ void __launch_bounds__(kBlock) k_plan_filter(uint32_t n, const uint32_t* __restrict__ rb,
                                                        const uint32_t* __restrict__ re,
                                                        const uint32_t* __restrict__ cnt_u,
                                                        const uint64_t* __restrict__ work_u,
                                                        uint4* __restrict__ funits, uint32_t fcap, uint32_t ucap,
                                                        uint32_t* __restrict__ wl_b, uint32_t* __restrict__ wl_e,
                                                        uint32_t* __restrict__ wl_k, bool pieces,
                                                        uint64_t* __restrict__ cnt) {
  constexpr uint32_t V = 4;  // vertices per thread per block iteration
  const uint64_t owned_all = count_total(cnt, kCntUEdges);
  if (owned_all > ucap) {  // asymmetric input: reported by the host, no unit is written
    if (blockIdx.x == 0 && threadIdx.x == 0) cnt[kCntOverflow] = owned_all;
    return;
  }
  const uint32_t cap_s = (uint32_t)min((uint64_t)kSmallEdges, max((uint64_t)96, owned_all / 8192));
  const uint32_t cap_l = (uint32_t)min((uint64_t)kLargeEdges, max((uint64_t)64, owned_all / 2048));
  const uint32_t cap_w =
      pieces ? (uint32_t)min((uint64_t)kWaveEdges, max((uint64_t)32, owned_all / kWavePieces)) : kWaveEdges;
  unsigned long long* const ctr[4] = {(unsigned long long*)&cnt[kCntFUnits1], (unsigned long long*)&cnt[kCntFUnits2],
                                      (unsigned long long*)&cnt[kCntTiny], (unsigned long long*)&cnt[kCntWPieces]};
  const uint64_t tile = (uint64_t)kBlock * V;
  for (uint64_t base = (uint64_t)blockIdx.x * tile; base < n; base += (uint64_t)gridDim.x * tile) {  // block-uniform
    uint32_t owned[V], c1[V], c2[V], c3[V], per[V], start[V], stop[V];
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint64_t x = base + j * kBlock + threadIdx.x;
      owned[j] = x < n ? cnt_u[x] : 0u;
    }
    uint32_t need[4] = {0, 0, 0, 0};
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
      need[3] += c3[j] ? (owned[j] - 1) / cap_w : 0u;
    }
    block_reserve<4>(need, ctr);
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
        wl_k[need[2]] = min(owned[j], cap_w);
        for (uint32_t at = cap_w; at < owned[j]; at += cap_w)
          wave_pieces(funits, fcap)[need[3]++] = make_uint4(start[j], stop[j], at, min(owned[j] - at, cap_w));
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

struct FilterArgs {
  uint32_t m;
  double eps;
  const int32_t* adj;
  const uint4* groups;
  const uint4* bits;   // coarse bitmaps, then (from fine0) the fine ones
  uint32_t fine0;
  uint4* uedge;        // (entry, its reverse entry, row start of a, d(a))
  uint8_t* flag;
  uint64_t* cnt;
};

constexpr uint32_t kTeamLoads = 4;  // 16-byte loads per lane and round

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

// Which bitmap of a shows enough misses, if nine elements in ten miss:
// (first word, words << 16 | words to read before a decision is likely), or
// words 0 when neither does.  fine_row: longest row with a usable fine one.
__device__ __forceinline__ uint2 pick_bitmap(uint32_t b0, uint32_t s, uint32_t l, uint32_t need, uint32_t fine0,
                                             uint32_t fine_row) {
  if (s < kMinRow) return make_uint2(0, 0);
  const float fs = (float)s, fl = (float)l, fn = (float)need;
  uint32_t words = coarse_words(s), at = coarse_at(b0);
#pragma unroll
  for (int fine = 0; fine < 2; ++fine) {
    if (fine) {
      if (s > fine_row) break;
      words *= 4;
      at = fine0 + at * 4;
    }
    const float bits = (float)(words * 128);
    // elements seen (1 - e^(-s/M)) M, each shown with e^(-l/M)
    const float shown =
        0.9f * bits * (1.0f - __builtin_exp2f(-1.442695f * fs / bits)) * __builtin_exp2f(-1.442695f * fl / bits);
    if (fn <= shown) {
      const uint32_t est = (uint32_t)((float)words * fn / shown) + 1;
      return make_uint2(at, (words << 16) | (est < words ? est : words));
    }
  }
  return make_uint2(0, 0);
}

// One round of a team over its row's bitmap: misses in the words
// [p, p + take) of `words`, row words at bits[at + p ..], the owner's at the
// same M from LDS word (of 16 bytes) `words` on.  Lanes past `take` load the
// last word again (every address is valid, also a resting team's).
template <uint32_t TEAM>
__device__ __forceinline__ uint32_t bitmap_round(const uint4* __restrict__ bits, uint32_t at, uint32_t words, uint32_t p,
                                                 uint32_t take, const uint4* owner) {
  const uint32_t tl = lane_id() & (TEAM - 1), last = take ? take - 1 : 0u;
  uint4 v[kTeamLoads];
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * TEAM < take)) break;
    v[j] = bits[at + p + min(j * TEAM + tl, last)];
  }
  uint32_t miss = 0;
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * TEAM < take)) break;
    const uint4 o = owner[words + p + min(j * TEAM + tl, last)];
    const uint32_t c = (uint32_t)__popc(v[j].x & ~o.x) + (uint32_t)__popc(v[j].y & ~o.y) +
                       (uint32_t)__popc(v[j].z & ~o.z) + (uint32_t)__popc(v[j].w & ~o.w);
    miss += j * TEAM + tl < take ? c : 0u;
  }
  return team_sum<TEAM>(miss);
}

// Absence bits of one hash group's seven elements in the top bits of a word,
// against a filter whose set bits are the absent elements.  An element costs
// four VALU instructions and one LDS read: address shift and mask, the word
// shifted by the element, and its low bit funnelled into the result.
__device__ __forceinline__ uint32_t group_absent(const uint4 v, const uint32_t* filt) {
  constexpr uint32_t mask = 0x1FFCu;
  const uint32_t base = (v.x & 0x1Eu) << 12;  // window (header >> 1) x 8 KB
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

// One round of a team of 16 over its row's groups: misses in [g, g + take).
__device__ __forceinline__ uint32_t group_round(uint32_t g, uint32_t take, const uint4* __restrict__ groups,
                                                const uint32_t* filt) {
  constexpr uint32_t TEAM = 16;
  const uint32_t tl = lane_id() & (TEAM - 1), last = take ? take - 1 : 0u;
  uint4 v[kTeamLoads];
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * TEAM < take)) break;
    v[j] = groups[g + min(j * TEAM + tl, last)];
  }
  uint32_t miss = 0;
#pragma unroll
  for (uint32_t j = 0; j < kTeamLoads; ++j) {
    if (j && !__ballot(j * TEAM < take)) break;
    const uint32_t bits = group_absent(v[j], filt);
    miss += (uint32_t)__popc(j * TEAM + tl < take ? bits : 0u);
  }
  return team_sum<TEAM>(miss);
}

// Ends a unit: edges of `mine` threads with !keep are rejected (flags), the
// kept ones' records move to the front of the unit's range [begin, ...), and
// *total of them are left.  part: one word per wave.  Called by every thread.
__device__ __forceinline__ void finish_unit(const FilterArgs& A, uint32_t begin, bool mine, bool keep, uint32_t entry,
                                            uint32_t reverse, uint32_t* part, uint32_t* total) {
  const uint32_t tid = threadIdx.x, lane = lane_id();
  if (mine && !keep) {
    if (entry < A.m) A.flag[entry] = kFlagN;
    if (reverse < A.m) A.flag[reverse] = kFlagN;
  }
  const uint64_t km = __ballot(keep);
  if (lane == 0) part[tid / kWave] = (uint32_t)__popcll(km);
  uint4 rec = make_uint4(0, 0, 0, 0);
  if (keep) rec = A.uedge[begin + tid];
  __syncthreads();  // also: every record that moves has been read
  uint32_t before = 0, sum = 0;
  for (uint32_t w = 0; w < blockDim.x / kWave; ++w) {
    const uint32_t c = part[w];
    before += w < tid / kWave ? c : 0u;
    sum += c;
  }
  if (keep) A.uedge[begin + before + (uint32_t)__popcll(km & lanemask_lt(lane))] = rec;
  *total = sum;
}

// Where a filter kernel's units come from and its survivors' units go: unit u
// is units[u] (step 1) or units[-u] (step -1).
struct UnitIO {
  const uint4* in;
  int in_step;
  int in_count, queue;  // counters
  uint4* next;          // large: units of the hash filter (null: to the exact kernels)
  uint4* small_exact;   // exact units of rows up to small_max_degree, from here up
  uint4* large_exact;   // the others, from here down
  uint32_t small_max_degree;
};

__device__ __forceinline__ void emit_unit(const FilterArgs& A, const UnitIO& io, const uint4 un, uint32_t total) {
  const uint4 out = make_uint4(un.x, un.x + total, un.z, un.w);
  if (io.next) {
    io.next[atomicAdd((unsigned long long*)&A.cnt[kCntHUnits], 1ull)] = out;
  } else if (un.w - un.z <= io.small_max_degree) {
    io.small_exact[atomicAdd((unsigned long long*)&A.cnt[kCntUnits1], 1ull)] = out;
  } else {
    *(io.large_exact - atomicAdd((unsigned long long*)&A.cnt[kCntUnits2], 1ull)) = out;
  }
}

// Bitmap filter of one unit at a time: an owner and up to MAXE of its edges;
// teams of 16 lanes take edges from the unit's cursor.  The owner's bitmap goes
// into LDS at the largest M needed (at LDS words [top, 2 top) of 16 bytes),
// then folded level by level ([w, 2 w) for M = 128 w).  Loading the stored
// bitmap instead of hashing the row again: R-MAT-22 shuffled, eps 0.6, large
// owners 632 -> 593 us.
template <bool LARGE>
__global__ void __launch_bounds__(LARGE ? 1024 : 256, 8) k_bitmap_units(FilterArgs A, UnitIO io) {
  stamp(A.cnt, LARGE ? kStampSim : kStampSimRest);
  constexpr uint32_t T = LARGE ? 1024 : 256, TEAM = 16;
  constexpr uint32_t MAXE = LARGE ? kLargeEdges : kSmallEdges;
  // 16-byte words of the largest M: M(46338) = 2^18 bits; 4 M(1024) = 2^14
  constexpr uint32_t TOP = LARGE ? 2048 : 128;
  constexpr uint32_t FINE = LARGE ? kWideRow - 1 : kFineRow;
  __shared__ uint4 s_own[2 * TOP];
  __shared__ uint2 e_at[MAXE];    // (first word, words << 16 | words to read first), longest first
  __shared__ uint16_t e_need[MAXE];
  __shared__ uint32_t s_surv[MAXE / 32], s_part[T / kWave], s_hist[32];
  __shared__ uint32_t s_unit, s_cursor;
  uint32_t* const own = reinterpret_cast<uint32_t*>(s_own);
  const uint32_t lane = lane_id(), tl = lane & (TEAM - 1), tid = threadIdx.x;
  const uint64_t nunits = A.cnt[io.in_count];
  unsigned long long* const queue = (unsigned long long*)&A.cnt[io.queue];
  // the first unit is the block's own, the others come from the queue, one
  // ahead
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
    const uint4 un = io.in[(int64_t)u * io.in_step];
    const uint32_t ne = un.y - un.x, bb = un.z, l = un.w - un.z;
    const bool mine = tid < ne && tid < MAXE;
    uint4 ed = make_uint4(kNone, kNone, 0, 0);  // (entry, reverse entry, row start of a, d(a))
    if (mine) ed = A.uedge[un.x + tid];
    // largest M needed: that of a row as long as the owner's, or the fine one
    // of the longest short row that may use it
    uint32_t top = coarse_words(min(l, kMaxThresholdRow));
    const uint32_t tf = 4 * coarse_words(min(l, FINE));
    top = top > tf ? top : tf;
    // that is the row's own stored bitmap, but for rows that have none
    const bool stored = LARGE ? l > kSmallRow && l <= kMaxThresholdRow : l >= kMinRow && l <= kFineRow;
    const uint4* const row = A.bits + (LARGE ? coarse_at(bb) : A.fine0 + 4 * coarse_at(bb));
    for (uint32_t t = tid; t < top; t += T) s_own[top + t] = stored ? row[t] : make_uint4(0, 0, 0, 0);
    if (tid < MAXE / 32) s_surv[tid] = 0;
    if (tid < 32) s_hist[tid] = 0;
    __syncthreads();
    if (!stored) {
      const uint32_t mask = top * 128 - 1;
      for (uint32_t t = tid; t < l; t += T) {
        const uint32_t h = vertex_hash((uint32_t)A.adj[bb + t]) & mask;
        atomicOr(&own[top * 4 + (h >> 5)], 1u << (h & 31));
      }
    }
    bool keep = false;  // survives
    uint32_t need = 0;
    uint2 at = make_uint2(0, 0);
    if (mine) {
      uint32_t cstar;
      need = misses_needed(A.eps, ed.w, l, &cstar, &keep);
      if (need) {
        at = pick_bitmap(ed.z, ed.w, l, need, A.fine0, FINE);
        keep = at.y == 0;
      }
    }
    uint32_t todo;
    const uint32_t slot = order_by_size(at.y & 0xFFFFu, s_hist, &todo);  // a barrier inside
    if (at.y) {
      e_at[slot] = at;
      e_need[slot] = (uint16_t)need;
    }
    // fold down to the shortest row that an undecided edge of b can have
    const float smin = (float)(l + 1) * (float)(A.eps * A.eps) - 2.0f;
    const uint32_t low = smin > 64.0f ? coarse_words((uint32_t)smin) : 1u;  // finer ones lie above
    for (uint32_t w = top >> 1; w >= low && w; w >>= 1) {
      for (uint32_t t = tid; t < w; t += T) {
        const uint4 x = s_own[2 * w + t], y = s_own[3 * w + t];
        s_own[w + t] = make_uint4(x.x | y.x, x.y | y.y, x.z | y.z, x.w | y.w);
      }
      __syncthreads();
    }
    __syncthreads();
    // ---- stream
    bool act = false, out = false;  // this team has an edge; the cursor is at its end
    uint32_t e = 0, a0 = 0, words = 0, p = 0, est = 0, left = 0;
    for (;;) {
      if (!act && !out) {
        uint32_t t = 0;
        if (tl == 0) t = atomicAdd(&s_cursor, 1u);
        t = (uint32_t)__shfl((int)t, (int)(lane & ~(TEAM - 1)));
        if (t < todo) {
          const uint2 q = e_at[t];
          e = t;
          a0 = q.x;
          words = q.y >> 16;
          est = q.y & 0xFFFFu;
          p = 0;
          left = e_need[t];
          act = true;
        } else {
          out = true;
        }
      }
      if (!__ballot(act)) break;
      const uint32_t want = est > p ? est - p : 1u;
      const uint32_t take = act ? min(min((want + TEAM - 1) / TEAM * TEAM, TEAM * kTeamLoads), words - p) : 0u;
      const uint32_t miss = bitmap_round<TEAM>(A.bits, a0, words, act ? p : 0u, take, s_own);
      if (act) {
        p += take;
        streamed += take;
        ++rounds;
        if (miss >= left) {
          act = false;
        } else {
          left -= miss;
          if (p >= words && a0 < A.fine0 && words <= coarse_words(FINE)) {
            a0 = A.fine0 + a0 * 4;  // once more, with the fine bitmap
            words = est = words * 4;
            p = 0;
            left = e_need[e];
          } else if (p >= words) {
            act = false;
            if (tl == 0) atomicOr(&s_surv[e >> 5], 1u << (e & 31));
          }
        }
      }
    }
    __syncthreads();
    if (at.y) keep = (s_surv[slot >> 5] >> (slot & 31)) & 1u;
    uint32_t total;
    finish_unit(A, un.x, mine, keep, ed.x, ed.y, s_part, &total);
    if (tid == 0 && total) emit_unit(A, io, un, total);
  }
  // 128 bits stand for about 22 elements
  const uint64_t elements = tl == 0 ? (uint64_t)streamed * 22 : 0ull;
  count_add<3>(A.cnt, {kCntProbes, kCntLoaded, kCntClaims}, {elements, elements, tl == 0 ? rounds : 0u});
}

// Hash filter of the large owners, unit by unit as above.  Bound by the reads
// of the groups past L2: half of the workgroups take the same time.
__global__ void __launch_bounds__(1024, 8) k_hash_units(FilterArgs A, UnitIO io) {
  stamp(A.cnt, kStampSim);
  constexpr uint32_t T = 1024, TEAM = 16, MAXE = kLargeEdges;
  constexpr uint32_t WORDS = 9 * kWindowWords16;
  __shared__ __align__(16) uint32_t filt[WORDS];
  __shared__ uint2 e_q[MAXE];  // (first group, groups << 16 | misses needed), most first
  __shared__ uint32_t s_surv[MAXE / 32], s_part[T / kWave], s_hist[32];
  __shared__ uint32_t s_unit, s_cursor;
  const uint32_t lane = lane_id(), tl = lane & (TEAM - 1), tid = threadIdx.x;
  const uint64_t nunits = A.cnt[io.in_count];
  unsigned long long* const queue = (unsigned long long*)&A.cnt[io.queue];
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
    const uint4 un = io.in[(int64_t)u * io.in_step];
    const uint32_t ne = un.y - un.x, bb = un.z, l = un.w - un.z;
    const bool mine = tid < ne && tid < MAXE;
    uint4 ed = make_uint4(kNone, kNone, 0, 0);  // (entry, reverse entry, row start of a, d(a))
    if (mine) ed = A.uedge[un.x + tid];
    // every element absent but the padding
    uint4* const f4 = reinterpret_cast<uint4*>(filt);
    for (uint32_t t = tid; t < WORDS / 4; t += T)
      f4[t] = make_uint4(~0u, ~0u, ~0u, t % (kWindowWords16 / 4) == kWindowWords16 / 4 - 1 ? 0x7FFFFFFFu : ~0u);
    if (tid < MAXE / 32) s_surv[tid] = 0;
    if (tid < 32) s_hist[tid] = 0;
    __syncthreads();
    const uint32_t bg = bb / 4, bn = row_groups(l);  // a large owner's row is wide
    for (uint32_t i = tid; i < bn; i += T) {
      const uint4 v = A.groups[bg + i];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      const uint32_t win = ((v.x & 0x1Eu) >> 1) * kWindowWords16;
#pragma unroll
      for (int q = 1; q < 8; ++q) {  // 0: the header
        const uint32_t h = q & 1 ? w[q >> 1] >> 16 : w[q >> 1] & 0xFFFFu;
        atomicAnd(&filt[win + (h >> 5)], ~(1u << (h & 31)));
        atomicAnd(&filt[h >> 5], ~(1u << (h & 31)));
      }
    }
    bool keep = false;  // survives
    uint32_t need0 = 0;
    if (mine) {
      uint32_t cstar;
      need0 = misses_needed(A.eps, ed.w, l, &cstar, &keep);
      if (need0) {
        keep = ed.w < kMinRow;  // no groups
        if (keep) need0 = 0;
      }
    }
    uint32_t todo;
    const uint32_t slot = order_by_size(need0, s_hist, &todo);
    if (need0) e_q[slot] = make_uint2(ed.z / 4, (row_groups(ed.w) << 16) | need0);
    __syncthreads();
    // ---- stream
    bool act = false, out = false;  // this team has an edge; the cursor is at its end
    uint32_t e = 0, g = bg, ge = 0, need = 0;
    for (;;) {
      if (!act && !out) {
        uint32_t t = 0;
        if (tl == 0) t = atomicAdd(&s_cursor, 1u);
        t = (uint32_t)__shfl((int)t, (int)(lane & ~(TEAM - 1)));
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
      // as many loads as reach `need` misses if an eighth of the elements
      // hit, so that little is read past the decision
      const uint32_t nl = (need + (need >> 3) + TEAM * kGroup - 1) / (TEAM * kGroup);
      const uint32_t take = act ? min(min(nl, kTeamLoads) * TEAM, ge - g) : 0u;
      const uint32_t miss = group_round(g, take, A.groups, filt);
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
    if (need0) keep = (s_surv[slot >> 5] >> (slot & 31)) & 1u;
    uint32_t total;
    finish_unit(A, un.x, mine, keep, ed.x, ed.y, s_part, &total);
    if (tid == 0 && total) emit_unit(A, io, un, total);
  }
  const uint64_t elements = tl == 0 ? (uint64_t)streamed * kGroup : 0ull;
  count_add<3>(A.cnt, {kCntProbes, kCntLoaded, kCntClaims}, {elements, elements, tl == 0 ? rounds : 0u});
}

// Owners with short rows, one wave each: the row's stored bitmap and its folds
// in LDS; 64 edges at a time, eight teams of 8 lanes.  What the bitmaps do not reject is
// counted element by element in a cuckoo hash of the owner's row (a quarter
// full at most, built when the first edge needs it), four teams of 16, so
// nothing is left to the exact kernels.  Planted communities (n = 3e5, eps
// 0.35, 2.8e7 undecided edges of rows around 185, an eighth similar): 2.7 ms,
// of which about half are the exact counts; 5.3 with binary searches in a
// sorted LDS row instead of the hash.  Waits for loads take two thirds of the
// wave cycles and the VALU is half busy: five waves a SIMD instead of six take
// 3.5 ms.  With the row hashed again for every owner, the owners dealt to the
// XCDs one by one and no owner fetched ahead: 2.85.
template <bool PIECES>
__global__ void __launch_bounds__(kBlock, 6)
    k_bitmap_wave(FilterArgs A, const uint32_t* __restrict__ wl_b, const uint32_t* __restrict__ wl_e,
                  const uint32_t* __restrict__ wl_k, const uint4* __restrict__ pieces) {
  stamp(A.cnt, kStampSimRest);
  // 16-byte words of the largest M: 4 M(256) = 2^12 bits; slots of each hash table
  constexpr uint32_t W = kBlock / kWave, TOP = 32, SLOTS = 2 * kWaveRow, SHIFT = 23;
  static_assert(SLOTS == 1u << (32 - SHIFT), "cuckoo hash shift");
  constexpr uint32_t EL = 6;  // elements per lane and round of an exact count
  __shared__ uint4 s_own[W][2 * TOP];
  __shared__ uint4 s_tab[W][2 * SLOTS / 4];
  __shared__ uint2 s_q[W][kWave];
  __shared__ uint16_t s_need[W][kWave], s_list[W][kWave];
  const uint32_t lane = lane_id(), wv = threadIdx.x / kWave;
  uint4* const own4 = s_own[wv];
  uint32_t* const own = reinterpret_cast<uint32_t*>(own4);
  uint32_t* const tab = reinterpret_cast<uint32_t*>(s_tab[wv]);
  uint2* const e_q = s_q[wv];
  uint16_t* const e_need = s_need[wv];
  uint16_t* const list = s_list[wv];
  const uint32_t owners = (uint32_t)A.cnt[kCntTiny], count = owners + (PIECES ? (uint32_t)A.cnt[kCntWPieces] : 0u);
  const uint32_t waves = gridDim.x * W;
  uint32_t streamed = 0, rounds = 0, probed = 0;
  // blocks of one XCD (every eighth) take neighbouring owners of the list,
  // whose edges share rows: its L2 then serves more of them
  const uint32_t per = gridDim.x / kXcds, vb = gridDim.x % kXcds ? blockIdx.x : blockIdx.x % kXcds * per + blockIdx.x / kXcds;
  uint32_t n_b = 0, n_e = 0, n_f = 0, n_k = 0;  // the next owner or piece, fetched one ahead
  auto fetch = [&](uint32_t i) {
    if (i < owners) {
      n_b = wl_b[i], n_e = wl_e[i], n_k = wl_k[i], n_f = 0;
    } else if (PIECES && i < count) {
      const uint4 q = pieces[i - owners];
      n_b = q.x, n_e = q.y, n_f = q.z, n_k = q.w;
    }
  };
  uint32_t idx = vb * W + wv;
  fetch(idx);
  for (; idx < count; idx += waves) {
    const uint32_t bb = __builtin_amdgcn_readfirstlane(n_b), be = __builtin_amdgcn_readfirstlane(n_e);
    const uint32_t owned = __builtin_amdgcn_readfirstlane(n_k), l = be - bb;
    const uint32_t first = PIECES ? bb + __builtin_amdgcn_readfirstlane(n_f) : bb;
    fetch(idx + waves);
    uint4 ed = make_uint4(kNone, kNone, 0, 0);  // (entry, reverse entry, row start of a, d(a))
    if (lane < owned) ed = A.uedge[first + lane];
    const uint32_t top = 4 * coarse_words(l), mask = top * 128 - 1;
    if (lane < top) own4[top + lane] = l >= kMinRow ? A.bits[A.fine0 + 4 * coarse_at(bb) + lane] : make_uint4(0, 0, 0, 0);
    wave_lds_sync();
    if (l < kMinRow) {
      if (lane < l) {
        const uint32_t h = vertex_hash((uint32_t)A.adj[bb + lane]) & mask;
        atomicOr(&own[top * 4 + (h >> 5)], 1u << (h & 31));
      }
      wave_lds_sync();
    }
    for (uint32_t w = top >> 1; w; w >>= 1) {
      if (lane < w) {
        const uint4 x = own4[2 * w + lane], y = own4[3 * w + lane];
        own4[w + lane] = make_uint4(x.x | y.x, x.y | y.y, x.z | y.z, x.w | y.w);
      }
      wave_lds_sync();
    }
    bool hashed = false, slow = false;  // the hash table is built; without it
    for (uint32_t base = 0; base < owned; base += kWave) {
      const uint32_t ne = min(owned - base, (uint32_t)kWave);
      if (base) {
        ed = make_uint4(kNone, kNone, 0, 0);
        if (lane < ne) ed = A.uedge[first + base + lane];
      }
      uint32_t cstar = 0;
      bool survive = false;
      uint2 at = make_uint2(0, 0);
      if (lane < ne) {
        const uint32_t need = misses_needed(A.eps, ed.w, l, &cstar, &survive);
        if (need) {
          at = pick_bitmap(ed.z, ed.w, l, need, A.fine0, kWaveRow);
          survive = at.y == 0;
        }
        e_need[lane] = (uint16_t)need;
      }
      const uint64_t bm = __ballot(at.y != 0);
      const uint32_t nb = (uint32_t)__popcll(bm);
      if (at.y) {
        e_q[lane] = at;
        list[(uint32_t)__popcll(bm & lanemask_lt(lane))] = (uint16_t)lane;
      }
      wave_lds_sync();
      // ---- bitmaps: teams of 8 take the edges in order
      {
        constexpr uint32_t TEAM = 8;
        const uint32_t tl = lane & (TEAM - 1);
        bool act = false;
        uint32_t e = 0, a0 = 0, words = 0, p = 0, est = 0, left = 0, next = 0;
        while (nb) {
          const uint64_t idle = __ballot(!act && tl == 0);
          if (idle && next < nb) {
            const uint32_t t = next + (uint32_t)__popcll(idle & lanemask_lt(lane & ~(TEAM - 1)));
            if (!act && t < nb) {
              e = list[t];
              const uint2 q = e_q[e];
              a0 = q.x;
              words = q.y >> 16;
              est = q.y & 0xFFFFu;
              p = 0;
              left = e_need[e];
              act = true;
            }
            next += (uint32_t)__popcll(idle);
          }
          if (!__ballot(act)) break;
          const uint32_t want = est > p ? est - p : 1u;
          const uint32_t take = act ? min(min((want + TEAM - 1) / TEAM * TEAM, TEAM * kTeamLoads), words - p) : 0u;
          const uint32_t miss = bitmap_round<TEAM>(A.bits, a0, words, act ? p : 0u, take, own4);
          if (act) {
            p += take;
            if (tl == 0) {
              streamed += take;
              ++rounds;
            }
            if (miss >= left) {
              act = false;
            } else {
              left -= miss;
              if (p >= words && a0 < A.fine0) {  // once more, with the fine bitmap
                a0 = A.fine0 + a0 * 4;
                words = est = words * 4;
                p = 0;
                left = e_need[e];
              } else if (p >= words) {
                act = false;
                if (tl == 0) e_q[e].y = kNone;  // survives
              }
            }
          }
        }
      }
      wave_lds_sync();
      if (at.y && e_q[lane].y == kNone) survive = true;
      // ---- exact counts of the survivors
      bool sim = false;
      const uint64_t sm = __ballot(survive);
      if (sm) {
        constexpr uint32_t TEAM = 16;
        const uint32_t tl = lane & (TEAM - 1);
        if (!hashed) {
          for (uint32_t t = lane; t < 2 * SLOTS / 4; t += kWave)
            s_tab[wv][t] = make_uint4(kEmptySlot, kEmptySlot, kEmptySlot, kEmptySlot);
          wave_lds_sync();
          bool ok = true;
          for (uint32_t t = lane; t < l; t += kWave)
            ok = cuckoo_insert(tab, (uint32_t)A.adj[bb + t], SLOTS, SHIFT) && ok;
          slow = __ballot(!ok) != 0;
          hashed = true;
        }
        wave_lds_sync();
        if (survive) {
          e_q[lane] = make_uint2(ed.z, (cstar << 16) | ed.w);  // d(a) <= l <= kWaveRow
          list[(uint32_t)__popcll(sm & lanemask_lt(lane))] = (uint16_t)lane;
        }
        wave_lds_sync();
        const uint32_t ns = (uint32_t)__popcll(sm);
        bool act = false;
        uint32_t e = 0, pos = 0, end = 0, hits = 0, cs = 0, next = 0;
        for (;;) {
          const uint64_t idle = __ballot(!act && tl == 0);
          if (idle && next < ns) {
            const uint32_t t = next + (uint32_t)__popcll(idle & lanemask_lt(lane & ~(TEAM - 1)));
            if (!act && t < ns) {
              e = list[t];
              const uint2 p = e_q[e];
              pos = p.x;
              end = p.x + (p.y & 0xFFFFu);
              cs = p.y >> 16;
              hits = 0;
              act = cs != 0;  // c* = 0: similar with any count
              if (!act && tl == 0) e_q[e].y = kNone;
            }
            next += (uint32_t)__popcll(idle);
          }
          if (!__ballot(act)) {
            if (next >= ns) break;
            continue;
          }
          uint32_t x[EL], v0[EL], v1[EL];
#pragma unroll
          for (uint32_t j = 0; j < EL; ++j) {
            const uint32_t k = j * TEAM + tl;
            x[j] = act && k < end - pos ? (uint32_t)A.adj[pos + k] : 0x7FFFFFFFu;  // no vertex
          }
          uint32_t h = 0;
          if (!slow) {
#pragma unroll
            for (uint32_t j = 0; j < EL; ++j) {
              v0[j] = tab[cuckoo_h0(x[j], SHIFT)];
              v1[j] = tab[SLOTS + cuckoo_h1(x[j], SHIFT)];
            }
#pragma unroll
            for (uint32_t j = 0; j < EL; ++j) h += v0[j] == x[j] || v1[j] == x[j] ? 1u : 0u;
          } else {
            for (uint32_t j = 0; j < EL; ++j) h += row_contains(A.adj, bb, be, (int32_t)x[j]) ? 1u : 0u;
          }
          h = team_sum<TEAM>(h);
          if (act) {
            const uint32_t took = min(EL * TEAM, end - pos);
            pos += took;
            hits += h;
            if (tl == 0) probed += took;
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
      wave_lds_sync();  // the lists are rewritten by the next batch
    }
  }
  const uint64_t elements = (uint64_t)streamed * 22 + probed;
  count_add<3>(A.cnt, {kCntProbes, kCntLoaded, kCntClaims}, {elements, elements, rounds});
}

// Offsets (bytes) of the copies in one allocation, and of the build's
// temporary memory.
struct PackLayout {
  size_t groups, coarse, fine, bytes;
  size_t mass, tab, narrow, wide, counts, tmp_bytes;
};

PackLayout pack_layout(uint64_t m) {
  PackLayout L;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) / 256 * 256;
    return o;
  };
  L.coarse = take((m / 16 + 2) * 16);
  L.fine = take((m / 16 + 2) * 64);
  L.groups = take((m / 4 + 2) * 16);
  L.bytes = off;
  off = 0;
  L.mass = take(kDegBuckets * 8);
  L.tab = take(kDegBuckets * sizeof(float2));
  L.narrow = take((m / kMinRow + 1) * 4);
  L.wide = take((m / kWideRow + 1) * 4);
  L.counts = take(32 * 8);
  L.tmp_bytes = off;
  return L;
}

}  // namespace

size_t packed_bytes(uint64_t m) { return pack_layout(m).bytes; }

hipError_t build_packed_rows(sgc_ctx* ctx, sgc_dgraph* g) {
  hipStream_t s = ctx->stream;
  const uint32_t n = g->n, m = g->m;
  const PackLayout L = pack_layout(m);
  char* const mem = (char*)work_memory(ctx, L.tmp_bytes);
  if (!mem) {  // every edge goes to the exact kernels
    drop_packed(g);
    return hipSuccess;
  }
  char* const out = g->packed;
  PackArgs A;
  A.n = n;
  A.rp = g->row_ptr, A.adj = g->adj, A.ndeg = g->ndeg;
  A.groups = (uint16_t*)(out + L.groups), A.coarse = (uint4*)(out + L.coarse), A.fine = (uint4*)(out + L.fine);
  A.mass = (unsigned long long*)(mem + L.mass), A.tab = (float2*)(mem + L.tab);
  A.narrow = (uint32_t*)(mem + L.narrow), A.wide = (uint32_t*)(mem + L.wide);
  A.counts = (unsigned long long*)(mem + L.counts);
  k_pack_clear<<<1, kDegBuckets, 0, s>>>(A);
  k_pack_lists<<<std::min(grid_for(n, kBlock * 8), 512u), kBlock, 0, s>>>(A);
  k_pack_table<<<1, kDegBuckets, 0, s>>>(A);
  k_pack_narrow<<<grid_for(std::min(n, m / kMinRow + 1), kBlock / kWave), kBlock, 0, s>>>(A);
  k_pack_wide<<<grid_for(std::min(n, m / kWideRow + 1), 1), kBlock, 0, s>>>(A);
  return hipGetLastError();
}

bool filter_stage(const sgc_dgraph* g, ScanParams p) {
  return g->packed && g->mirror && !p.prune && !p.count_all && g->tuning.hash_tables != 0;
}

void launch_plan_filter(const sgc_dgraph* g, const PassBuffers& b, hipStream_t s) {
  // the lists share arrays that the core pass initialises later
  k_plan_filter<<<grid_for(g->n, kBlock), kBlock, 0, s>>>(g->n, g->row_begin, g->row_end, b.cnt_u, b.work_u, b.units,
                                                          b.ucap / 2, b.ucap, (uint32_t*)b.label, (uint32_t*)b.parent,
                                                          (uint32_t*)b.lo, g->m < kPieceEntries, b.cnt);
}

bool filter_leaves_units(const sgc_dgraph* g) { return g->max_degree > std::min(kWaveRow, kWaveEdges); }

void launch_filter(const sgc_dgraph* g, const PassBuffers& b, ScanParams p, int cu_count, hipStream_t s) {
  const uint32_t cus = (uint32_t)(cu_count > 0 ? cu_count : 256);
  const PackLayout L = pack_layout(g->m);
  const char* const mem = (const char*)g->packed;
  const FilterArgs A{g->m,     p.eps,
                     g->adj,   (const uint4*)(mem + L.groups),
                     (const uint4*)(mem + L.coarse), (uint32_t)((L.fine - L.coarse) / 16),
                     b.uedge,  b.flag,
                     b.cnt};
  // Units of owners above kWaveRow entries: a unit has at least 32 edges unless
  // it is its owner's last, m / 2 edges are owned and an owner has more than 256
  // entries, so there are at most m / 64 + m / 257 of each kind and each of the
  // four lists has room in an eighth of the array (m / 16).
  const uint32_t fcap = b.ucap / 2;
  UnitIO io;
  io.small_exact = b.units + fcap;
  io.large_exact = b.units + b.ucap - 1;
  io.small_max_degree = g->tuning.small_max_degree;
  uint4* const hash_units = b.units + fcap / 4;
  const bool coarse = p.eps >= kCoarseEps;
  io.in = b.units + fcap - 1, io.in_step = -1, io.in_count = kCntFUnits2, io.queue = kCntFQueue2;
  const bool hashes = p.eps >= kHashEps;
  io.next = hashes ? hash_units : nullptr;
  // kernels whose owners the graph cannot have are not launched (an owner
  // with more than kWaveEdges edges has a longer row than that)
  const bool has_large = g->max_degree > kSmallRow, has_small = g->max_degree > std::min(kWaveRow, kWaveEdges);
  if ((coarse || !hashes) && has_large) {
    k_bitmap_units<true><<<cus * 2, 1024, 0, s>>>(A, io);
    io.in = hash_units, io.in_step = 1, io.in_count = kCntHUnits, io.queue = kCntHQueue;
  }
  io.next = nullptr;
  if (hashes && has_large) k_hash_units<<<cus * 2, 1024, 0, s>>>(A, io);
  io.in = b.units, io.in_step = 1, io.in_count = kCntFUnits1, io.queue = kCntFQueue1;
  if (has_small) k_bitmap_units<false><<<cus * 8, 256, 0, s>>>(A, io);
  const bool cut = g->m < kPieceEntries;
  const uint64_t want = ((uint64_t)g->n * (cut ? 2 : 1) + kBlock / kWave - 1) / (kBlock / kWave), cap = (uint64_t)cus * 6;
  const uint32_t grid = (uint32_t)(want < cap ? want : cap);
  const uint32_t *const wl_b = (const uint32_t*)b.label, *const wl_e = (const uint32_t*)b.parent,
                 *const wl_k = (const uint32_t*)b.lo;
  if (cut)
    k_bitmap_wave<true><<<grid, kBlock, 0, s>>>(A, wl_b, wl_e, wl_k, wave_pieces(b.units, fcap));
  else
    k_bitmap_wave<false><<<grid, kBlock, 0, s>>>(A, wl_b, wl_e, wl_k, nullptr);
}

}  // namespace sgc
