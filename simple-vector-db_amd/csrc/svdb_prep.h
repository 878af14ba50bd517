// svdb_prep.h — the part of the query prep that BF16 and FP8 share
// (internal, device code).
//
// One wavefront per query slot.  The row is staged in LDS by coalesced loads
// (four per lane in flight); the canonical ‖q‖² chain then
// reads it back 16 columns at a time at wave-uniform addresses (broadcast
// reads, no conflicts), every lane carrying the same chain, and the
// quantization works on columns spread over the lanes.  The chain's d
// dependent FP64 fmas bound it.  A thread per query had one global load
// latency per column on that chain and quantized serially between its steps:
// 35 µs at 128 columns and 485 µs at 1,536 for any batch too small to hide
// it (now 5 and 20 µs), 48 µs for 16,384 queries of 128 columns (now 23),
// 354 µs for 4,096 FP8 queries of 768 (now 26).
#pragma once

#include "svdb_lowp.h"

namespace svdb {

constexpr int kPrepWaves = 4;  // query slots per block

struct PrepSlot {
  int range;      // -1: padding slot
  uint32_t row;   // row of Q
};

__device__ __forceinline__ PrepSlot prep_slot(const QueryPrepArgs& a, uint32_t slot, int& metric) {
  int r = 0;
  while (r + 1 < a.nr && slot >= a.soff[r + 1]) r++;
  metric = a.metric[r];
  const uint32_t i = slot - a.soff[r];
  return i < a.n[r] ? PrepSlot{r, a.qoff[r] + i} : PrepSlot{-1, 0};
}

// Stages row q (d columns, zeros up to `cols`; copied to qd unless that is
// null) and returns its canonical
// Σ fma(v, v, ·) (the zeros beyond d leave a chain's bits as they are),
// max |v| and whether every element is finite, the same in every lane.
__device__ __forceinline__ double prep_stage(const double* __restrict__ q,
                                             double* __restrict__ qd, uint32_t d, uint32_t cols,
                                             double* row, int lane, double& maxabs, bool& finite) {
  double mx = 0.0;
  bool fin = true;
  for (uint32_t c0 = 0; c0 < cols; c0 += 256) {
    double v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t c = c0 + j * 64 + lane;
      v[j] = c < d ? q[c] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t c = c0 + j * 64 + lane;
      if (c < cols) row[c] = v[j];
      if (qd && c < d) qd[c] = v[j];
      fin = fin && isfinite(v[j]);
      mx = fmax(mx, fabs(v[j]));
    }
  }
  for (int o = 32; o >= 1; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  maxabs = mx;
  finite = __all(fin);
  __builtin_amdgcn_wave_barrier();
  double acc = 0.0;
  for (uint32_t c = 0; c < cols; c += 16) {
    double x[16];
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
      const double2 t = *reinterpret_cast<const double2*>(row + c + j);
      x[j] = t.x;
      x[j + 1] = t.y;
    }
#pragma unroll
    for (int j = 0; j < 16; j++) acc = fma(x[j], x[j], acc);
  }
  return acc;
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

}  // namespace svdb
