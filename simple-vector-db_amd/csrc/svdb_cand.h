// svdb_cand.h — the first passes' candidate lists (internal, device code).
//
// A list belongs to one lane of a scan and one of its queries: up to
// kLowpLC (ordering key, slot) entries in global memory, in no order, and a
// header {entries, bound}: every row the list covers and does not hold is
// keyed at or above the bound.  With a starting threshold most subtiles bring
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

// An MFMA's result must not be read by another unit for some wait states after
// it issued, and the compiler, which inserts them, does not see a read behind a
// branch that the scans nearly always fall through (the rare insertion): at
// 1,536 columns accumulators were copied four states after their last MFMA,
// three too early, and rows were lost.  The scans therefore read a subtile's
// accumulators behind the next subtile's first MFMAs, which fences hold in
// front, and let the last subtile's settle here, once per tile.
__device__ __forceinline__ void settle_mfma(float __attribute__((ext_vector_type(4))) & acc) {
  asm volatile("s_nop 7" : "+v"(acc));
}

__device__ __forceinline__ size_t cand_list(const LowpScanArgs& a, uint32_t q, uint32_t list) {
  return (size_t)q * a.NL + list;
}

// The four rows of a lane's accumulator, at least one keyed below tau: those
// below it enter the list at `e` holding `cnt` entries.  Straight-line stores
// (a lane seldom has more than one, but its wavefront's lanes have theirs at
// different rows); a list that is or has become full takes the loop.
__device__ __forceinline__ void cand_append4(uint2* __restrict__ e, uint32_t& cnt, float& tau,
                                             float (&k4)[4], uint32_t srow) {
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (k4[r] < tau && cnt < (uint32_t)kLowpLC) {
      e[cnt++] = make_uint2(__float_as_uint(k4[r]), srow + r);
      k4[r] = INFINITY;
    }
  if (__builtin_expect(cnt < (uint32_t)kLowpLC, 1)) return;
  for (int r = 0; r < 4;) {
    float m1 = -INFINITY, m2 = -INFINITY;  // the largest two keys held
    uint32_t at = 0;
#pragma unroll 2
    for (int i = 0; i < kLowpLC; i += 2) {
      const uint4 v = *reinterpret_cast<const uint4*>(e + i);
      const float x = __uint_as_float(v.x), y = __uint_as_float(v.z);
      m2 = fmaxf(m2, fminf(m1, x));
      at = x > m1 ? i : at;
      m1 = fmaxf(m1, x);
      m2 = fmaxf(m2, fminf(m1, y));
      at = y > m1 ? i + 1 : at;
      m1 = fmaxf(m1, y);
    }
    tau = m1;
    // the next row keyed below the largest entry takes its place
    for (; r < 4; r++) {
      const float k = r == 0 ? k4[0] : r == 1 ? k4[1] : r == 2 ? k4[2] : k4[3];
      if (!(k < tau)) continue;
      e[at] = make_uint2(__float_as_uint(k), srow + r);
      tau = fmaxf(m2, k);
      r++;
      break;
    }
  }
}

// A sorted register list (unused entries: slot ~0) to its place.
__device__ __forceinline__ void cand_store_sorted(const LowpScanArgs& a, size_t list,
                                                  const float (&lk)[kLowpLP],
                                                  const uint32_t (&ls)[kLowpLP]) {
  uint2* e = a.ent + list * kLowpLC;
  uint32_t n = 0;
#pragma unroll
  for (int j = 0; j < kLowpLP; j++)
    if (ls[j] != ~0u) {
      e[j] = make_uint2(__float_as_uint(lk[j]), ls[j]);
      n++;
    }
  a.hdr[list] = make_uint2(n, __float_as_uint(lk[kLowpLP - 1]));
}

}  // namespace svdb
