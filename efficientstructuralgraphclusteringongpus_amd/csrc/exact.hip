// Exact common-neighbour counts for units (an owner b and some of its
// undecided edges (a, b)) whose owner's row fits LDS as one table: rows of up
// to 1024 entries as a cuckoo hash or, on graphs of few ids, a bit set over
// all of them; longer rows as a bit set, on graphs of up to 2^20 ids.  What is
// left (long rows over more ids, the pruned core check's deferrals, graphs
// tuned to hash_tables = 0) goes to k_sim_units.
//
// Teams of 16 lanes take (edge, segment of the short row) pairs, 96 elements
// to a round.  k_sim_units gives an edge a whole wave: most short rows are
// shorter than a wave's load, and the LDS bookkeeping of a claim, the same for
// 20 elements as for 1000, came to more than the counting.  A long short row
// is cut into segments of kSegment so that no team is left alone with one; the
// segments' (hits, consumed) add up in one 64-bit LDS word, read as a snapshot
// for the early exit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.h"
#include "device_util.h"

namespace sgc {

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kTeam = 16;
constexpr uint32_t kSegment = 1536;                  // a bucket edge of order_by_size
constexpr uint32_t kSmallKeys = 1024;                // longest row in a cuckoo hash
constexpr uint32_t kBitmapIds = 1u << 20;            // most ids of a bit set (128 KB)

// PER: elements per lane and round.  Six where several blocks share a CU; one
// block of 16 waves, beside a bit set of over 56 KB, needs sixteen loads in
// flight: R-MAT-20, all common neighbours counted, 6 / 8 / 12 / 16 a lane
// 6.0 / 5.6 / 5.1 / 5.1 ms (k_sim_units 6.7; R-MAT-18 1.72 -> 1.16, R-MAT-16
// 0.73 -> 0.52).  What bounds it there is the latency of the short rows' loads,
// from L2 and beyond.  Units are units[u] (small) or units[ucap - 1 - u] (LARGE), as the planner
// lays them out; at most 256 / 768 edges each.  `tab`: the bit set's
// ceil(n / 32) words, or 4 * 1024 slots.
template <bool LARGE, bool BITMAP, uint32_t PER, int WAVES>
__global__ void __launch_bounds__(LARGE ? 1024 : 256, WAVES)
    k_exact_units(uint32_t n, uint32_t m, const uint32_t* __restrict__ src, const int32_t* __restrict__ adj,
                  bool mirrored, double eps, uint8_t* __restrict__ flag, uint32_t* __restrict__ cn_out,
                  const uint4* __restrict__ uedge, const uint4* __restrict__ units, uint32_t ucap,
                  uint64_t* __restrict__ cnt, int units_slot, int queue_slot) {
  stamp(cnt, LARGE ? kStampExactLarge : kStampExactSmall);
  constexpr uint32_t T = LARGE ? 1024 : 256, MAXE = LARGE ? 768 : 256, ROUND = kTeam * PER;
  extern __shared__ __align__(16) uint32_t tab[];
  __shared__ unsigned long long e_state[MAXE];  // hits << 32 | consumed
  __shared__ __align__(16) uint4 e_q[MAXE];     // (row start, d(a), c*), longest rows first
  __shared__ uint32_t s_hist[32];
  __shared__ uint32_t s_unit, s_cursor, s_fail, s_long, s_most;
  const uint32_t tid = threadIdx.x, lane = lane_id(), tl = lane & (kTeam - 1);
  const uint64_t nunits = cnt[units_slot];
  uint32_t streamed = 0, rounds = 0, nxt = blockIdx.x;
  for (;;) {
    if (tid == 0) {
      s_unit = nxt;
      s_cursor = s_fail = s_long = s_most = 0;
      if (nxt < nunits)
        nxt = nunits > gridDim.x ? gridDim.x + (uint32_t)atomicAdd((unsigned long long*)&cnt[queue_slot], 1ull) : kNone;
    }
    if (tid < 32) s_hist[tid] = 0;
    __syncthreads();
    const uint32_t u = s_unit;
    if (u >= nunits) break;
    const uint4 un = units[LARGE ? ucap - 1 - u : u];  // (begin, end) in uedge, the owner's row [bb, be)
    const uint32_t ne = min(un.y - un.x, MAXE), bb = un.z, be = un.w, l = be - bb;
    uint4 ed = make_uint4(kNone, kNone, 0, 0);  // (entry, reverse entry, row start of a, d(a))
    if (tid < ne) ed = uedge[un.x + tid];
    // ---- the owner's row
    uint32_t shift = 0, second = 0;
    if constexpr (BITMAP) {
      const uint32_t words = (n + 31) / 32;
      for (uint32_t t = tid * 4; t < words; t += T * 4)  // the allocation is a multiple of 16 bytes
        *reinterpret_cast<uint4*>(tab + t) = make_uint4(0, 0, 0, 0);
      __syncthreads();
      for (uint32_t t = bb + tid; t < be; t += T) {
        const uint32_t x = (uint32_t)adj[t];
        atomicOr(&tab[x >> 5], 1u << (x & 31));
      }
    } else {
      // two tables of 2^bits >= 2 l slots
      const uint32_t bits = l > 32 ? 33 - __clz(l - 1) : 6u;
      second = 1u << bits;
      shift = 32 - bits;
      for (uint32_t t = tid; t < second / 2; t += T)
        reinterpret_cast<uint4*>(tab)[t] = make_uint4(kEmptySlot, kEmptySlot, kEmptySlot, kEmptySlot);
      __syncthreads();
      bool ok = true;
      for (uint32_t t = tid; t < l; t += T) ok = cuckoo_insert(tab, (uint32_t)adj[bb + t], second, shift) && ok;
      if (!ok) s_fail = 1;
    }
    // ---- the edges
    const uint32_t s = ed.w;
    uint32_t cstar = 0;
    double rhs = 0;
    if (ed.x < m) {
      rhs = predicate_rhs(eps, s, l);
      cstar = s <= kMaxThresholdRow && !cn_out ? min_common_threshold(rhs, s) : kNone;
    }
    const bool stream = ed.x < m && cstar != 0 && (cstar == kNone || cstar <= s);
    uint32_t todo;
    const uint32_t slot = order_by_size(stream ? min(s, 65535u) : 0u, s_hist, &todo);  // a barrier inside
    if (stream) {
      e_state[slot] = 0;
      e_q[slot] = make_uint4(ed.z, s, cstar, 0);
      if (s >= kSegment) {
        atomicAdd(&s_long, 1u);
        atomicMax(&s_most, s);
      }
    }
    __syncthreads();
    const bool slow = !BITMAP && s_fail;  // no table after all: search the row
    const uint32_t nlong = s_long, segments = (s_most + kSegment - 1) / kSegment;
    // ---- stream
    bool act = false, out = false;  // this team has an edge; the cursor is at its end
    uint32_t e = 0, pos = 0, end = 0, h0 = 0, rest = 0, hits = 0, used = 0, cs = 0;
    for (;;) {
      if (!act && !out) {
        uint32_t t = 0;
        if (tl == 0) t = atomicAdd(&s_cursor, 1u);
        t = (uint32_t)__shfl((int)t, (int)(lane & ~(kTeam - 1)));
        uint32_t seg = 0;
        if (t >= todo) {  // every first segment is taken: the others of the long rows
          t -= todo;
          seg = nlong ? 1 + t / nlong : segments;
          t = nlong ? t % nlong : 0u;
          out = seg >= segments;
        }
        if (!out) {
          const uint4 q = e_q[t];
          if (seg * kSegment < q.y) {
            const unsigned long long st = e_state[t];
            e = t;
            pos = q.x + seg * kSegment;
            end = q.x + min(q.y, (seg + 1) * kSegment);
            cs = q.z;
            h0 = (uint32_t)(st >> 32);
            rest = q.y - (uint32_t)st;  // elements not consumed when the segment starts
            hits = used = 0;
            act = !seg || cs == kNone || (h0 < cs && h0 + rest >= cs);
          }
        }
      }
      if (!__ballot(act)) {
        if (!__ballot(!out)) break;
        continue;
      }
      const uint32_t left = act ? end - pos : 0u;
      uint32_t x[PER], h = 0;
#pragma unroll
      for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t k = j * kTeam + tl;
        x[j] = k < left ? (uint32_t)adj[pos + k] : (BITMAP ? 0u : 0x7FFFFFFFu);  // the latter is no vertex
      }
      if constexpr (BITMAP) {
        uint32_t v[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) v[j] = tab[x[j] >> 5];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) h += j * kTeam + tl < left ? (v[j] >> (x[j] & 31)) & 1u : 0u;
      } else if (!slow) {
        uint32_t v0[PER], v1[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
          v0[j] = tab[cuckoo_h0(x[j], shift)];
          v1[j] = tab[second + cuckoo_h1(x[j], shift)];
        }
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) h += v0[j] == x[j] || v1[j] == x[j] ? 1u : 0u;
      } else {
        for (uint32_t j = 0; j < PER; ++j) h += row_contains(adj, bb, be, (int32_t)x[j]) ? 1u : 0u;
      }
      h = team_sum<kTeam>(h);
      if (act) {
        const uint32_t took = min(left, ROUND);
        pos += took;
        used += took;
        hits += h;
        if (tl == 0) {
          streamed += took;
          ++rounds;
        }
        // other segments only add to what the snapshot knew
        if (pos >= end || (cs != kNone && (h0 + hits >= cs || h0 + hits + (rest - used) < cs))) {
          if (tl == 0) atomicAdd(&e_state[e], ((unsigned long long)hits << 32) | used);
          act = false;
        }
      }
    }
    __syncthreads();
    // ---- both directed entries of every edge
    if (ed.x < m) {
      const uint32_t got = stream ? (uint32_t)(e_state[slot] >> 32) : 0u;
      uint32_t rev = ed.y;
      if (rev == kNone && !mirrored) {
        const uint32_t b = src[bb];
        uint32_t lo = ed.z, hi = ed.z + s;
        while (lo < hi) {
          const uint32_t mid = lo + ((hi - lo) >> 1);
          if (adj[mid] < (int32_t)b)
            lo = mid + 1;
          else
            hi = mid;
        }
        rev = lo < ed.z + s && adj[lo] == (int32_t)b ? lo : kNone;
      }
      if (cn_out) {
        cn_out[ed.x] = got;
        if (rev < m) cn_out[rev] = got;
      } else {
        const uint8_t f = (cstar != kNone ? got >= cstar : predicate_exact(got, rhs)) ? kFlagY : kFlagN;
        flag[ed.x] = f;
        if (rev < m) flag[rev] = f;
      }
    }
    __syncthreads();  // the state is reset by the next unit
  }
  const uint64_t el = tl == 0 ? streamed : 0u;
  count_add<3>(cnt, {kCntProbes, kCntLoaded, kCntClaims}, {el, el, tl == 0 ? rounds : 0u});
}

}  // namespace

bool exact_units_cover(uint32_t n, bool large) { return !large || n <= kBitmapIds; }

void launch_exact_units(const sgc_dgraph* g, const PassBuffers& b, const uint4* units, uint32_t ucap, ScanParams p,
                        int cu_count, hipStream_t s, bool large, uint32_t* cn_out) {
  const uint32_t cus = (uint32_t)(cu_count > 0 ? cu_count : 256);
  const size_t bits = ((size_t)g->n + 127) / 128 * 16;
  if (large) {
    // a bit set of less than half the LDS leaves room for a second block
    if (bits <= 56u << 10)
      k_exact_units<true, true, 6, 8><<<cus * 2, 1024, bits, s>>>(g->n, g->m, g->src, g->adj, g->mirror != nullptr,
                                                                  p.eps, b.flag, cn_out, b.uedge, units, ucap, b.cnt,
                                                                  kCntUnits2, kCntQueue2);
    else
      k_exact_units<true, true, 16, 4><<<cus, 1024, bits, s>>>(g->n, g->m, g->src, g->adj, g->mirror != nullptr, p.eps,
                                                               b.flag, cn_out, b.uedge, units, ucap, b.cnt, kCntUnits2,
                                                               kCntQueue2);
  } else if (bits <= 16 * kSmallKeys) {
    k_exact_units<false, true, 6, 6><<<cus * 6, 256, bits, s>>>(g->n, g->m, g->src, g->adj, g->mirror != nullptr, p.eps,
                                                          b.flag, cn_out, b.uedge, units, ucap, b.cnt, kCntUnits1,
                                                          kCntQueue1);
  } else {
    k_exact_units<false, false, 6, 6><<<cus * 6, 256, 16 * kSmallKeys, s>>>(
        g->n, g->m, g->src, g->adj, g->mirror != nullptr, p.eps, b.flag, cn_out, b.uedge, units, ucap, b.cnt,
        kCntUnits1, kCntQueue1);
  }
}

}  // namespace sgc
