// Device helpers used by the generated per-rule join kernels.
//
// Execution model of a generated kernel (see srd_pipeline.h for the launch
// protocol): a wave64 owns one slice, a contiguous range of the flattened
// level-1 items (possibly spanning keys).  Items are processed 64 at a time,
// one per lane.  If the rule has a second nested level, the lanes that
// produced a binding publish it in LDS and the wave walks the concatenation
// of their level-2 iteration spaces 64 items at a time (each position's
// owner found from per-batch start flags, a ballot and a popcount), so a
// lane with a huge level-2 range does not serialize the wave.  Every emitted
// tuple is one lane's result for one item; ballot + mbcnt give its position,
// so emission never diverges.
//
// Counterparts in the reference: the warp-cooperative WCOJ body emitted by
// src/srdatalog/codegen/jit/pipeline.py:360 / root.py / instructions.py over
// the search primitives of runtime/generalized_datalog/gpu/search.h and
// IntersectView (gpu/device_sorted_array_index.ipp:1284-1487).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "srd_device.h"
#include "srd_pipeline.h"

namespace srdj {

using srd::IndexView;
using srd::Rng;

__device__ __forceinline__ const uint32_t* colp(const IndexView& v, int c) {
  return v.cols + uint64_t(c) * v.stride;
}

// find_slot, find_slot_from: srd_device.h
using srd::find_slot;
using srd::find_slot_from;

// Equal range of the value at driver position pos inside [b,e) of column
// col (values within [b,e) sorted); `last` = column is the index's last.
__device__ __forceinline__ Rng run_at(const uint32_t* __restrict__ col, uint32_t pos, uint32_t e,
                                      uint32_t v, bool last) {
  if (last) return Rng{pos, pos + 1};
  return Rng{pos, srd::upper_bound_la(col, pos + 1, e, v)};
}

// Persistent-wave slice dispenser.  Every lane executes the atomic (lane 0
// adds 1, the others 0) and the wave takes lane 0's result with v_readlane,
// a scalar.  There must be no lane-dependent branch around the atomic: with
// `if (lane == 0) s = atomicAdd(...)` the compiler threads the lanes that
// skip the branch (whose s is the constant 0) straight back to the
// broadcast, forming a second loop in which lanes 1..63 re-read lane 0's
// stale register and never fetch a new slice.
// Slices [slice_lo, n_slices) are split into SRD_XCDS ranges; a wave takes
// the next slice of its own XCD's range, then of the following ranges in
// turn; it returns n_slices when every range is exhausted.  The first
// slices of a range belong to its waves by position (`first`: the wave has
// taken none yet), and only those beyond come from the counter: a launch with no
// more slices than waves touches no counter.  With every slice drawn, the
// 8,192 waves of a small launch queued on the eight counters, at the end eight
// times each: 33 us for the load of 5,000 pairs, 21 us with this.
__device__ __forceinline__ uint64_t next_slice(const SrdLaunchArgs& A, uint64_t n, bool first) {
  const uint64_t lo = A.slice_lo;
  if (n <= lo) return n;
  const uint64_t span = n - lo;
  const uint32_t nr = A.n_ranges ? A.n_ranges : 1u;
  const uint32_t home = blockIdx.x % nr;
  const uint32_t wpb = blockDim.x / 64u;
  if (first) {
    const uint64_t s = lo + span * home / nr + uint64_t(blockIdx.x / nr) * wpb +
                       __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
    if (s < lo + span * (home + 1) / nr) return s;
  }
  for (uint32_t k = 0; k < nr; ++k) {
    const uint32_t x = (home + k) % nr;
    // slices of range x beyond its waves' own
    const uint64_t own = gridDim.x > x ? uint64_t((gridDim.x - x + nr - 1) / nr) * wpb : 0;
    const uint64_t b = lo + span * x / nr + own, e = lo + span * (x + 1) / nr;
    if (b >= e) continue;
    const uint32_t t = atomicAdd(A.work_ctr + x * SRD_CTR_STRIDE, srd::lane_id() == 0 ? 1u : 0u);
    const uint64_t s = b + __builtin_amdgcn_readlane(t, 0);
    if (s < e) return s;
  }
  return n;
}

// Mark mode: note that the key's block of 2^18 keys holds a set bit.  A byte
// per block, stored plainly: the bytes of a whole bitmap fill a few lines,
// and a bit set with an atomic per newly marked key serialised every wave of
// the launch on those lines (the load of 260,000 R-MAT pairs: 254 us with
// 64 waves in flight and 1,744 us with 4,096; 70 us with stores).
__device__ __forceinline__ void mark_block(const SrdLaunchArgs& A, uint64_t key) {
  __hip_atomic_store(A.mark_sum + (key >> 18), uint8_t(1), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// ---- products in the mark mode ----
// A product A x B whose tuples are (row a, last column b) sets, for every a
// of A, the same set of bits in a's row of the bitmap.  B is sorted, so its
// bits are first folded into (word, mask) pairs, 64 bits to a word, and each
// pair is then tested against and OR-ed into every row: |A| * words(B) word
// operations instead of |A| * |B| bit operations, and neighbouring lanes
// touch neighbouring words.  Points-to sets of thousands of objects put 10
// to 60 of them into a word (Andersen at 1/10 of its full size: the four
// marking traversals 562 -> 169 ms of kernel time a fixpoint).

// Wave steps of a product of nr rows and the sorted values [b, e) of col: the
// pairs are at most the values, and at most the words their span covers.
// Lanes hold pairs and the rows are walked, or, when that takes fewer
// steps, lanes hold rows and the pairs are walked.
__device__ __forceinline__ uint64_t prod_steps(const uint32_t* __restrict__ col, uint32_t b,
                                               uint32_t e, uint32_t nr) {
  const uint32_t nm = e - b;
  uint32_t nw = nm;
  if (nm > 64u) nw = min(nm, (col[e - 1] >> 6) - (col[b] >> 6) + 1u);
  const uint64_t by_row = uint64_t((nw + 63u) / 64u) * nr;
  const uint64_t by_pair = uint64_t((nr + 63u) / 64u) * nw;
  return min(by_row, by_pair) + 2u * uint64_t((nm + 63u) / 64u) + 1u;
}

// OR the n (<= 64) pairs of lw / lm into rows [r0, r1) of cr.
__device__ __forceinline__ void prod_flush(const SrdLaunchArgs& A, uint64_t kb, uint32_t rshift,
                                           const uint32_t* __restrict__ cr, uint32_t r0, uint32_t r1,
                                           uint32_t n, const uint32_t* lw, const uint64_t* lm) {
  const uint32_t lane = srd::lane_id();
  uint64_t* bits = reinterpret_cast<uint64_t*>(A.mark_bits);
  const uint32_t nr = r1 - r0;
  constexpr uint32_t U = 4;  // words loaded before the first is tested
  if (uint64_t(nr) <= uint64_t((nr + 63u) / 64u) * n) {
    const uint32_t w = lane < n ? lw[lane] : 0u;
    const uint64_t m = lane < n ? lm[lane] : 0;
    for (uint32_t t = r0; t < r1; t += 64) {
      const uint32_t cnt = min(64u, r1 - t);
      const uint32_t ra = lane < cnt ? cr[t + lane] : 0u;
      for (uint32_t i = 0; i < cnt; i += U) {
        uint64_t at[U], cur[U];
#pragma unroll
        for (uint32_t q = 0; q < U; ++q) {
          // past the last row: the last row again (its bits are set by then)
          const uint32_t a = __builtin_amdgcn_readlane(ra, min(i + q, cnt - 1));
          at[q] = ((kb + (uint64_t(a) << rshift)) >> 6) + w;
          cur[q] = m ? bits[at[q]] : ~uint64_t(0);
        }
#pragma unroll
        for (uint32_t q = 0; q < U; ++q)
          if (m & ~cur[q]) {
            atomicOr(reinterpret_cast<unsigned long long*>(bits + at[q]), (unsigned long long)m);
            mark_block(A, at[q] << 6);
          }
      }
    }
    return;
  }
  for (uint32_t t = r0; t < r1; t += 64) {
    const bool in = t + lane < r1;
    const uint64_t row = (kb + (uint64_t(in ? cr[t + lane] : 0u) << rshift)) >> 6;
    for (uint32_t j = 0; j < n; j += U) {
      uint64_t at[U], cur[U], m[U];
#pragma unroll
      for (uint32_t q = 0; q < U; ++q) {
        const uint32_t p = min(j + q, n - 1);
        m[q] = lm[p];
        at[q] = row + lw[p];
        cur[q] = in ? bits[at[q]] : ~uint64_t(0);
      }
#pragma unroll
      for (uint32_t q = 0; q < U; ++q)
        if (m[q] & ~cur[q]) {
          atomicOr(reinterpret_cast<unsigned long long*>(bits + at[q]), (unsigned long long)m[q]);
          mark_block(A, at[q] << 6);
        }
    }
  }
}

// Fold the sorted values [mb, me) of cm into (word, mask) pairs and hand them
// to flush(n), n <= 64 at a time, in lw / lm: 128 LDS words of the calling
// wave, lm all zero on entry and left so.  Wave-uniform arguments, all 64 lanes.
template <class F>
__device__ __forceinline__ void fold_pairs(const uint32_t* __restrict__ cm, uint32_t mb, uint32_t me,
                                           uint32_t* lw, uint64_t* lm, F&& flush) {
  const uint32_t lane = srd::lane_id();
  uint32_t n = 0, prev = ~0u;
  constexpr uint32_t L = 4;  // values loaded ahead, in 64s
  uint32_t ahead[L];
  for (uint32_t pos = mb, q = 0; pos < me; pos += 64, q = (q + 1) % L) {
    if (q == 0) {
#pragma unroll
      for (uint32_t i = 0; i < L; ++i)
        ahead[i] = pos + 64u * i + lane < me ? cm[pos + 64u * i + lane] : 0u;
    }
    const uint32_t v = q == 0 ? ahead[0] : (q == 1 ? ahead[1] : (q == 2 ? ahead[2] : ahead[3]));
    const uint32_t cnt = min(64u, me - pos);
    const bool in = lane < cnt;
    const uint32_t w = in ? v >> 6 : ~0u;
    uint32_t up = __shfl_up(w, 1, 64);
    if (lane == 0) up = prev;
    const bool head = in && w != up;
    const uint64_t hm = srd::ballot(head);
    // the pair of this value's word: the last one opened at or below it
    const uint32_t slot = n + srd::popc_below(hm) + (head ? 1u : 0u) - 1u;
    if (in) {
      atomicOr(reinterpret_cast<unsigned long long*>(lm + slot), 1ull << (v & 63u));
      if (head) lw[slot] = w;
    }
    n += uint32_t(__popcll(hm));
    prev = __builtin_amdgcn_readlane(w, cnt - 1);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (n > 64) {  // 64 complete pairs; the last one may still grow
      flush(64u);
      n -= 64;
      const uint32_t w2 = lw[64 + lane];
      const uint64_t m2 = lm[64 + lane];
      __builtin_amdgcn_wave_barrier();
      lw[lane] = w2;
      lm[lane] = m2;
      lm[64 + lane] = 0;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  }
  if (n) flush(n);
  __builtin_amdgcn_wave_barrier();
  lm[lane] = 0;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// Mark rows [r0, r1) of cr times the sorted values [mb, me) of cm: bit
// kb + (row << rshift) + value (lw, lm: fold_pairs).
__device__ __forceinline__ void prod_mark(const SrdLaunchArgs& A, uint64_t kb, uint32_t rshift,
                                          const uint32_t* __restrict__ cm, uint32_t mb, uint32_t me,
                                          const uint32_t* __restrict__ cr, uint32_t r0, uint32_t r1,
                                          uint32_t* lw, uint64_t* lm) {
  if (r1 <= r0) return;
  fold_pairs(cm, mb, me, lw, lm,
             [&](uint32_t n) { prod_flush(A, kb, rshift, cr, r0, r1, n, lw, lm); });
}

// Mark the sorted values [b, e) of col in the one row at bit kb (a multiple of
// 64).  Thousands of items mark the row of a popular root key, from every
// XCD: the words are read at device scope, past caches that would show them
// clear, and set 64 bits at a time (bit by bit behind plain loads, the atomics
// of one such row took 8 ms).
__device__ __forceinline__ void run_mark(const SrdLaunchArgs& A, uint64_t kb,
                                         const uint32_t* __restrict__ col, uint32_t b, uint32_t e,
                                         uint32_t* lw, uint64_t* lm) {
  const uint32_t lane = srd::lane_id();
  uint64_t* row = reinterpret_cast<uint64_t*>(A.mark_bits) + (kb >> 6);
  fold_pairs(col, b, e, lw, lm, [&](uint32_t n) {
    if (lane < n) {
      const uint32_t w = lw[lane];
      const uint64_t m = lm[lane];
      const uint64_t cur = __hip_atomic_load(row + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (m & ~cur) {
        atomicOr(reinterpret_cast<unsigned long long*>(row + w), (unsigned long long)m);
        mark_block(A, kb + (uint64_t(w) << 6));
      }
    }
  });
}

// The same for the ranges of the lanes `mine`, all of one row, through their
// keys' bitmaps (view v, lane's slot hb, first and last value of its range):
// the bitmaps are OR-ed together 64 words at a time and the row is updated
// once for all of them, one load per 64 words of a range of thousands.
__device__ __forceinline__ void run_mark_bits(const SrdLaunchArgs& A, uint64_t kb, const IndexView& v,
                                              uint64_t mine, uint32_t hb, uint32_t first, uint32_t last) {
  const uint32_t lane = srd::lane_id();
  const bool in = (mine >> lane) & 1u;
  const uint32_t hi = srd::wave_max(in ? last >> 6 : 0u);
  const uint32_t lo = ~srd::wave_max(in ? ~(first >> 6) : 0u);
  uint64_t* row = reinterpret_cast<uint64_t*>(A.mark_bits) + (kb >> 6);
  const uint64_t* bm = reinterpret_cast<const uint64_t*>(v.bm);
  const uint64_t bw = v.bm_words >> 1;
  constexpr uint32_t U = 4;
  for (uint32_t w0 = lo; w0 <= hi; w0 += 64) {
    const uint32_t w = w0 + lane;
    const bool on = w <= hi && w < bw;
    uint64_t acc = 0;
    for (uint64_t m = mine; m;) {
      uint64_t x[U];
#pragma unroll
      for (uint32_t q = 0; q < U; ++q) {
        // past the last range: the one before again
        const uint32_t o = uint32_t(__builtin_ctzll(m));
        x[q] = on ? bm[uint64_t(__builtin_amdgcn_readlane(hb, o)) * bw + w] : 0;
        const uint64_t rest = m & (m - 1);
        if (q + 1 < U && rest) m = rest;
      }
      m &= m - 1;
#pragma unroll
      for (uint32_t q = 0; q < U; ++q) acc |= x[q];
    }
    if (acc) {
      const uint64_t cur = __hip_atomic_load(row + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (acc & ~cur) {
        atomicOr(reinterpret_cast<unsigned long long*>(row + w), (unsigned long long)acc);
        mark_block(A, kb + (uint64_t(w) << 6));
      }
    }
  }
}

// Row r of nr at the part num/den of a product's cost: cuts at equal costs
// of two neighbouring slices give equal rows, so the parts tile the rows.
__device__ __forceinline__ uint32_t prod_cut(uint32_t nr, uint64_t num, uint64_t den) {
  return uint32_t(uint64_t(nr) * num / den);
}

// Fused mode: open a staging segment of SRD_SEG rows for the wave (all lanes
// take part; lane 0's bump is broadcast with v_readlane).  Returns ~0 when
// staging is exhausted (the overflow flag is raised; the slice keeps
// counting, and the host then re-runs the write pass).
__device__ __forceinline__ uint64_t seg_open(const SrdLaunchArgs& A) {
  const unsigned long long r =
      atomicAdd(A.stage_ctr, srd::lane_id() == 0 ? (unsigned long long)SRD_SEG : 0ull);
  const uint64_t s = srd::read_lane_u64(r, 0);
  const bool ovf = s + SRD_SEG > A.stage_cap;  // wave-uniform
  if (ovf) atomicOr(A.overflow, srd::lane_id() == 0 ? 1u : 0u);
  return ovf ? ~uint64_t(0) : s;
}

// Fused mode: log segment [start, start+used) as rows local..local+used of
// `slice`'s output.
__device__ __forceinline__ void seg_close(const SrdLaunchArgs& A, uint64_t slice, uint64_t start,
                                          uint32_t used, uint32_t local) {
  if (start == ~uint64_t(0) || used == 0) return;
  const uint32_t r = atomicAdd(A.rec_ctr, srd::lane_id() == 0 ? 1u : 0u);
  const uint32_t idx = __builtin_amdgcn_readlane(r, 0);
  const bool ovf = idx >= A.rec_cap;  // wave-uniform
  if (ovf) atomicOr(A.overflow, srd::lane_id() == 0 ? 1u : 0u);
  if (!ovf && srd::lane_id() == 0) {
    A.recs[3ull * idx] = slice;
    A.recs[3ull * idx + 1] = start;
    A.recs[3ull * idx + 2] = (uint64_t(local) << 32) | used;
  }
}

// Cooperative lower bound: for every lane with `on`, the first position p in
// [b, e) of col with col[p] >= v (e if none).  Consecutive `on` lanes with the
// same `seg` form a run; the lanes of a run must share [b, e) and hold
// non-decreasing v (a run is one owner's candidates, read in column order).
// The first lane of each run searches lower_bound(v_first) and the last one
// upper_bound(v_last) over the whole range; every other lane of the run then
// searches only the window between those two positions, where its answer
// lies.  A divergent full-range search costs one cache-line lookup per lane
// and step; the window searches of one run touch a few shared lines instead.
// Must be called with all 64 lanes active (wave-uniform control flow).
__device__ __forceinline__ uint32_t seg_lower_bound(const uint32_t* __restrict__ col, uint32_t b,
                                                    uint32_t e, uint32_t v, bool on, uint32_t seg) {
  const uint32_t lane = srd::lane_id();
  const uint64_t onm = srd::ballot(on);
  const uint32_t seg_p = __shfl_up(seg, 1, 64);
  const uint32_t seg_n = __shfl_down(seg, 1, 64);
  const bool on_p = lane > 0 && ((onm >> (lane - 1)) & 1ull);
  const bool on_n = lane < 63 && ((onm >> (lane + 1)) & 1ull);
  const bool first = on && !(on_p && seg_p == seg);
  const bool last = on && !(on_n && seg_n == seg);
  // run ends: first lanes lower_bound(v), last-only lanes upper_bound(v)
  const bool upper = last && !first;
  uint32_t lo = b;
  uint32_t n = (first || last) ? e - b : 0u;
  while (n > 0) {
    const uint32_t half = n >> 1;
    const uint32_t mid = lo + half;
    const uint32_t x = col[mid];
    if (upper ? x <= v : x < v) {
      lo = mid + 1;
      n -= half + 1;
    } else {
      n = half;
    }
  }
  const uint64_t fm = srd::ballot(first);
  const uint64_t lm = srd::ballot(last);
  const uint64_t le = lane == 63 ? ~0ull : ((2ull << lane) - 1);
  const uint64_t below = fm & le;
  const uint32_t src_f = below ? 63u - uint32_t(__clzll((long long)below)) : lane;
  const uint64_t above = lm >> lane;
  const uint32_t src_l = above ? lane + uint32_t(__ffsll((unsigned long long)above)) - 1u : lane;
  const uint32_t w_lo = __shfl(lo, int(src_f), 64);
  const uint32_t w_hi = __shfl(lo, int(src_l), 64);
  if (!on || first) return lo;
  // w_lo <= answer <= w_hi for every lane strictly inside or at the end of a run
  uint32_t l2 = w_lo;
  uint32_t n2 = w_hi - w_lo;
  while (n2 > 0) {
    const uint32_t half = n2 >> 1;
    const uint32_t mid = l2 + half;
    if (col[mid] < v) {
      l2 = mid + 1;
      n2 -= half + 1;
    } else {
      n2 = half;
    }
  }
  return l2;
}

// Whether index view v holds a row whose first sizeof...(key) columns equal
// key (negated atoms: the rule's binding survives only when this is false).
template <class... T>
__device__ __forceinline__ bool has_prefix(const IndexView& v, T... key) {
  constexpr int n = int(sizeof...(T));
  const uint32_t k[n] = {uint32_t(key)...};
  if (v.n == 0) return false;
  Rng r = srd::root_find(v, k[0]);
#pragma unroll
  for (int d = 1; d < n; ++d) {
    if (r.e <= r.b) return false;
    r = srd::child_find(v, d, r, k[d], d == int(v.arity) - 1);
  }
  return r.e > r.b;
}

// Bitmap slot of the heavy key whose depth-1 range of view v starts at row
// b, or ~0u when that key has no bitmap.
__device__ __forceinline__ uint32_t heavy_slot(const IndexView& v, uint32_t b) {
  if (v.n_hv == 0) return ~0u;
  const uint32_t p = srd::lower_bound(v.hv_start, 0, v.n_hv, b);
  return (p < v.n_hv && v.hv_start[p] == b) ? p : ~0u;
}

// Whether value x is in the range whose bitmap is `slot` of view v.
__device__ __forceinline__ bool heavy_has(const IndexView& v, uint32_t slot, uint32_t x) {
  const uint32_t w = x >> 5;
  return w < v.bm_words && ((v.bm[uint64_t(slot) * v.bm_words + w] >> (x & 31u)) & 1u);
}

// Wave-uniform copy of a 64-bit value held by `lane`.
__device__ __forceinline__ uint64_t uniform_from(uint64_t v, int lane) {
  uint32_t lo = __builtin_amdgcn_readlane(uint32_t(v), lane);
  uint32_t hi = __builtin_amdgcn_readlane(uint32_t(v >> 32), lane);
  return (uint64_t(hi) << 32) | lo;
}

}  // namespace srdj
