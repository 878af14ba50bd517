// svdb_cand.h — the first passes' candidate lists (internal, device code).
//
// A list belongs to one lane of a scan and one of its queries: up to
// kLowpLC (ordering key, slot) entries in global memory, in no order, and a
// header {entries, bound}: every row the list covers and does not hold is
// keyed at or above the bound.  (Lists from nothing, in registers: see
// cand_store_sorted.)  With a starting threshold most subtiles bring
// a lane nothing and a query's lists together take a few hundred rows of a
// million, so an entry is one 8-byte store at the lane's own count — no list
// in registers (eight sorted entries per fragment had taken 64 of a wavefront's
// 256 registers at four fragments, and an insertion some 50 instructions for
// every lane of the wavefront).  A full list drops its largest entry for a
// smaller key, reading itself back: the bound is then its largest key.
// Scan time against the sorted register lists, with thresholds that let a
// quarter as many rows pass (lowp_enqueue): 500k × 128, 64 cosine queries
// 107 → 66 µs; 200k × 200, 101 queries of three metrics, k = 100 181 → 56;
// 1M × 128, 700 queries, k = 100 1,169 → 430; 150k × 768 FP8, 4,096 queries,
// k = 100 1,267 → 905; 2M × 128, 16,384 queries, k = 10 7,150 → 6,890.
#pragma once

#include "svdb_lowp.h"

namespace svdb {

// The scans' forms: only the smallest key of each list (the sample
// pre-pass), lists from nothing (kept sorted in registers), lists below a
// starting threshold (stored as they come).
enum ScanForm { kFormMin = 0, kFormSorted = 1, kFormAppend = 2 };

// Wait states from an MFMA to another unit's use of its result: passes + 4,
// v_mfma_f32_16x16x32_bf16 taking 4 passes and FP8's
// v_mfma_scale_f32_16x16x128_f8f6f4 8.
constexpr int kBf16States = 8, kFp8States = 12;

// The compiler, which inserts those states, does not always see a read behind a
// branch that the scans nearly always fall through (the rare insertion): at
// 1,536 columns accumulators were copied four states after their last MFMA,
// three too early, and rows were lost.  The scans therefore read a subtile's
// accumulators behind the next subtile's first MFMAs, which fences hold in
// front, and let the last subtile's settle here, once per tile; where those
// MFMAs are too few for the form's states (FP8 with one fragment) the rest is
// waited for here too.  What the compiler makes of it is followed through every
// branch of the built kernels by tests/test_mfma_waits_cpu.py.
template <int STATES, int QF>
__device__ __forceinline__ void settle_mfma(float __attribute__((ext_vector_type(4))) (&acc)[QF]) {
  static_assert(STATES >= 1 && STATES <= 16, "one s_nop");
  static_assert(QF == 1 || QF == 2 || QF == 4, "every accumulator is named");
  if constexpr (QF == 1)
    asm volatile("s_nop %1" : "+v"(acc[0]) : "n"(STATES - 1));
  else if constexpr (QF == 2)
    asm volatile("s_nop %2" : "+v"(acc[0]), "+v"(acc[1]) : "n"(STATES - 1));
  else
    asm volatile("s_nop %4"
                 : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
                 : "n"(STATES - 1));
}

__device__ __forceinline__ size_t cand_list(const LowpScanArgs& a, uint32_t q, uint32_t list) {
  return (size_t)q * a.NL + list;
}

// A lane's last entry waits here for the start of the next tile (or for the
// lane's next entry): a tile ends with a wait for its successor's loads, which
// counts stores too, and one issued late in the tile would hold up the block
// (2M × 128, 16,384 cosine queries: 7.5 ms with stores at once, 6.9 deferred).
// Entries count from the block's first list: its lists stay below 2^32 entries.
struct CandPending {
  uint32_t at = ~0u;  // entry index (~0: none)
  uint32_t key, slot;
};

__device__ __forceinline__ void cand_flush(uint2* ent, CandPending& p) {
  if (p.at != ~0u) ent[p.at] = make_uint2(p.key, p.slot);
  p.at = ~0u;
}

// The four rows of a lane's accumulator: those keyed below tau enter list
// `list` holding `cnt` entries, the smallest first.  A wavefront seldom has
// more than one such row, so a pass takes each lane's smallest and the loop
// ends with the wavefront's last.  A test and a store for each of the four
// rows spent the time in branches over nothing, and sixteen copies of that code
// made a kernel of 74 KB, past the 64 KB instruction cache (1M × 256, 8,192
// queries: 5.1 ms, so 3.9).  Called by a whole wavefront; `ent` is the entries
// of the block's first list.
__device__ __forceinline__ void cand_append4(uint2* ent, CandPending& p, uint32_t list,
                                             uint32_t& cnt, float& tau, float (&k4)[4],
                                             uint32_t srow) {
  const uint32_t e0 = list * kLowpLC;
  do {
    const float k = fminf(fminf(k4[0], k4[1]), fminf(k4[2], k4[3]));
    if (k < tau) {
      const uint32_t r = k4[0] == k ? 0 : k4[1] == k ? 1 : k4[2] == k ? 2 : 3;
      const uint32_t at = cnt;
      if (at < (uint32_t)kLowpLC) {
        cand_flush(ent, p);
        p.at = e0 + at;
        p.key = __float_as_uint(k);
        p.slot = srow + r;
        cnt = at + 1;
      }
      if (__builtin_expect(cnt == (uint32_t)kLowpLC, 0)) {
        // full: from here on tau is the largest key held, whose place a
        // smaller one takes
        cand_flush(ent, p);
        uint2* e = ent + e0;
        float m1 = -INFINITY, m2 = -INFINITY;  // the largest two keys held
        uint32_t big = 0;
#pragma unroll 2
        for (int i = 0; i < kLowpLC; i += 2) {
          const uint4 v = *reinterpret_cast<const uint4*>(e + i);
          const float x = __uint_as_float(v.x), y = __uint_as_float(v.z);
          m2 = fmaxf(m2, fminf(m1, x));
          big = x > m1 ? i : big;
          m1 = fmaxf(m1, x);
          m2 = fmaxf(m2, fminf(m1, y));
          big = y > m1 ? i + 1 : big;
          m1 = fmaxf(m1, y);
        }
        tau = m1;
        if (at == (uint32_t)kLowpLC) {
          e[big] = make_uint2(__float_as_uint(k), srow + r);
          tau = fmaxf(m2, k);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) k4[i] = r == (uint32_t)i ? INFINITY : k4[i];
    }
  } while (__ballot(fminf(fminf(k4[0], k4[1]), fminf(k4[2], k4[3])) < tau));
}

// A sorted register list to its place: kLowpLP entries, unused ones with slot ~0
// behind the others and keyed with the bound, which is the last entry's key.
__device__ __forceinline__ void cand_store_sorted(const LowpScanArgs& a, size_t list,
                                                  const float (&lk)[kLowpLP],
                                                  const uint32_t (&ls)[kLowpLP]) {
  // (a branch an entry: with plain stores the compiler keeps the lists elsewhere
  // during the scan; FP8, 31k × 768, 1,848 cosine queries: 432 µs, 409 so)
  uint2* e = a.ent + list * kLowpLP;
#pragma unroll
  for (int j = 0; j < kLowpLP; j++)
    if (ls[j] != ~0u) e[j] = make_uint2(__float_as_uint(lk[j]), ls[j]);
    else e[j] = make_uint2(__float_as_uint(lk[kLowpLP - 1]), ~0u);
}

}  // namespace svdb
