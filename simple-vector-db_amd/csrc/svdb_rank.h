// svdb_rank.h — FP64 rank keys, their order, and slots (internal, device code).
#pragma once

#include "svdb_kernels.h"

namespace svdb {

// A rank key as a uint64 that orders like the doubles (-0 folded to +0, NaN
// above +inf), and back.
__device__ __forceinline__ uint64_t rank_bits(double v) {
  v = v + 0.0;  // -0 → +0 (not folded: strict FP)
  uint64_t u = (uint64_t)__double_as_longlong(v);
  if (v != v) u = 0x7FF8000000000000ull;
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

__device__ __forceinline__ double rank_value(uint64_t u) {
  uint64_t b = (u >> 63) ? (u & 0x7FFFFFFFFFFFFFFFull) : ~u;
  return __longlong_as_double((long long)b);
}

__device__ __forceinline__ bool lex_lt(uint64_t ka, uint32_t sa, uint64_t kb, uint32_t sb) {
  return (ka < kb) | ((ka == kb) & (sa < sb));
}

// A wavefront's common value, in scalar registers.
__device__ __forceinline__ uint64_t uni64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ bool slot_alive(const uint64_t* alive, uint32_t r) {
  return (alive[r >> 6] >> (r & 63)) & 1ull;
}

__device__ __forceinline__ uint64_t logical_id(const StoreView& st, uint32_t slot) {
  if (!st.has_deletes) return slot;
  uint32_t w = slot >> 6;
  uint64_t below = st.alive[w] & ((1ull << (slot & 63)) - 1ull);
  return (uint64_t)st.rank_base[w] + (uint64_t)__popcll(below);
}

}  // namespace svdb
