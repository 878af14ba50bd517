// svdb_scan_f64.hip — the FP64 exhaustive scan on the matrix cores, and the
// selection of its results (gfx950).  Built with -ffp-contract=off; every fma
// below is explicit.
//
// v_mfma_f64_16x16x4f64 adds the four products of a k-step onto each
// accumulator one after the other, each as one correctly rounded fused
// multiply-add (the same bits as sequential fma chains, subnormal, infinite
// and NaN operands included), so chained over the k-steps in column order it
// computes exactly the canonical dot key s = Σ_i fma(q_i, x_i, s); cosine
// divides it.  Euclidean keys, Σ fma(t, t, s) with t = x_i − q_i, have no
// matrix form: the dot product gives a = (xx + qq) − 2·dot (xx, qq the
// canonical squared norms), within E = c·(‖x‖ + ‖q‖)² + e of the canonical key
// (l2_bound), and only a pair whose lower bound a − E could still be among its
// query's nearest computes the canonical key (exact_chain); every other pair is
// provably out.
//
// Block: 4 wavefronts, 16 queries each (64 per block), sharing the rows of
// one slice, which stream through LDS in stages of 64 rows × SC columns
// (global_load_lds_dwordx4, double-buffered, so the next stage's loads run
// under this stage's MFMAs).  A row step (64 rows, all columns) is an even
// number of stages, so each of the two buffers, which the compiler has to know
// apart, has its own place in the loop and the step's epilogue is there once.
// Up to 64 columns (SC = 32) and up to 128 (SC = 64) a row step is two stages
// and a wavefront's queries stay in registers (QRES); wider rows take
// 32-column stages and load each stage's query values one stage ahead.
// Any width: rows are zero up to a multiple of 8 columns, query values past D
// are zero, and the stages stop at D's last k-step, so the columns added to a
// chain are 0 · 0, which leave it as it is.
// 16-byte units are XOR-swizzled by row so the operand reads of 16 rows hit
// distinct banks.  Lane l, g = l / 16, j = l % 16; k-step s of a stage covers
// its columns 4s..4s+3:
//   A (queries)  lane l holds Q[qw + j][col0 + 4s + g]   (global loads)
//   B (rows)     lane l holds X[row0 + 16t + j][col0 + 4s + g]  (LDS)
//   accumulator  tile t, register r of lane l: query qw + g + 4r, row
//                row0 + 16t + j
//
// The bound a list starts from comes from a sample (MINS): the same products
// over 1/16 of the rows, each lane keeping the smallest of its rows' keys
// (Euclidean: of their upper bounds a + E).  The lanes' rows are disjoint, so
// the k-th smallest of those minima is at or above the k-th key of the store;
// about 16·k rows of a query lie below it.
//
// Results: each (query, slice) has an unsorted list in global memory.  A row
// enters when its key is at most the query's global bound gtk — the smallest
// k-th key any of its lists has reached, atomic min — and ranks before the
// list's own k-th.  A list that cannot take a row is cut to its k best
// (f64_compact), which gives it that k-th and lowers gtk, and the row is tried
// again.  A test per (query, row) is one comparison of doubles; all else happens
// in branches that a row step seldom takes.  (Sorted lists spread over a wavefront's registers
// had taken 48 of them at k <= 64 and 96 above, and every insertion a chain of
// lane shuffles.  500k × 128, 1,024 queries, dot, k = 10: 3.54 → 2.53 ms for the
// call, 37 → 52 TF/s; 300k × 100, 77 queries, Euclidean, k = 100, on the VALU
// before: 3.74 → 0.32 ms; 1M × 128, 16 queries, dot, k = 100: 3.59 → 0.36 ms.)
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "svdb_bins.h"
#include "svdb_f64_lists.h"
#include "svdb_kernels.h"
#include "svdb_rank.h"

namespace svdb {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

// Hides a lane's value at the end of a loop over whole wavefronts: where the
// compiler sees what a lane that has nothing left does in the next turn, it may
// send it there by a way of its own, and the cross-lane steps on the way are
// then taken without it (such lanes had held the counts by which full lists are
// found: they were not cut).
__device__ __forceinline__ void whole_wave(uint32_t& v) { asm volatile("" : "+v"(v)); }

// Byte offset in a stage of SC columns of 16-byte unit u (columns 2u, 2u+1)
// of row r.
template <int SC>
__device__ __forceinline__ int f64_unit(int r, int u) {
  return (r * (SC / 2) + (u ^ (r & 15))) * 16;
}

// The stage of rows row0.. (clamped to the store) and columns col0.. (those
// below the row stride): direct-to-LDS instructions of 64 × 16 bytes.
template <int SC>
__device__ __forceinline__ void f64_issue_stage(const StoreView& st, unsigned char* buf,
                                                uint32_t row0, uint32_t col0, int wave,
                                                int lane) {
  constexpr int UPR = SC / 2;  // units per row
#pragma unroll
  for (int i = 0; i < kF64StageRows * UPR / (64 * kWavesPerBlock); i++) {
    const int p0 = (wave + kWavesPerBlock * i) * 64;  // first unit slot of this instruction
    const int p = p0 + lane;
    const int r = p / UPR, u = (p % UPR) ^ (r & 15);
    const uint32_t row = min(row0 + (uint32_t)r, st.nrows - 1);
    const uint32_t col = col0 + 2 * u;
    if (col < st.ldx)
      __builtin_amdgcn_global_load_lds(st.X + (size_t)row * st.ldx + col,
                                       (lds_void_t*)(buf + p0 * 16), 16, 0, 0);
  }
}

// The canonical chain of row x and query q over D columns (x 16-byte aligned,
// zero past D): Euclidean Σ_i fma(t, t, s), t = x_i − q_i, else Σ_i fma(q_i, x_i, s).
template <bool L2>
__device__ __forceinline__ double exact_chain(const double* __restrict__ x,
                                              const double* __restrict__ q, uint32_t D) {
  double s = 0.0;
  for (uint32_t c = 0; c < D; c += 8) {
    double xv[8], qv[8];
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const double2 v = *reinterpret_cast<const double2*>(x + c + i);
      xv[i] = v.x;
      xv[i + 1] = v.y;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) qv[i] = c + i < D ? q[c + i] : 0.0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const double t = xv[i] - qv[i];
      s = L2 ? fma(t, t, s) : fma(qv[i], xv[i], s);
    }
  }
  return s;
}

// Bound on |a − s*| for a = fl(fl(xx + qq) − 2·dot) and the canonical key
// s*, with xx, qq, dot and s* the canonical fma chains over D columns and
// u = 2^-53.  Each chain is within γ_D = D·u/(1 − D·u) of its exact value
// relative to its sum of |terms| (xx: ‖x‖², qq: ‖q‖², dot: ‖q‖‖x‖), the two
// roundings of a add at most 2u(1 + γ_D)·S with S = (‖x‖ + ‖q‖)², and the
// rounded differences t_i change ‖x − q‖² ≤ S by at most 2u + u², so
// |a − s*| ≤ (2γ_D + 4u + O(u²))·S, and the final a ∓ E rounds by at most
// 2u·S more.  E = (4D + 128)·u·sn² with sn = fl(sqrt(xx)) + fl(sqrt(qq))
// (≥ (‖x‖ + ‖q‖)(1 − γ_D − 3u)) is more than twice that for any D the
// store allows, and e = (8D + 64)·2^-1074 covers the absolute error of
// subnormal results (at most one 2^-1074 per rounding, 5D + 4 of them).
// A non-finite operand gives a non-finite bound: the pair takes the
// exact path.
template <bool UPPER>
__device__ __forceinline__ double l2_bound(double xx, double qq, double dot, double xs,
                                          double qs, double crel, double eabs) {
  const double ap = (xx + qq) - 2.0 * dot;
  const double sn = xs + qs;
  const double E = crel * (sn * sn) + eabs;
  return UPPER ? ap + E : ap - E;
}

// A wavefront's list state, in LDS: per query its entries, the k-th (key, slot)
// of its last cut and the global bound as last read.
struct F64Wave {
  uint32_t cnt[kScanTQ];
  uint32_t own_slot[kScanTQ];
  uint64_t own_key[kScanTQ];
  uint64_t gk[kScanTQ];
  uint32_t queue[128];  // pairs awaiting their key
};

// Cuts a list of n entries to its k best by (key, slot), one wavefront.  Up to 64
// entries find their places by comparing with each other (28 entries: 0.5 µs);
// of more, the k-th key is found by bisecting the key's bits with counts over the
// wavefront, the slot among equal keys likewise, and what remains is packed (3 µs).
__device__ __attribute__((noinline)) void f64_compact(uint64_t* key, uint32_t* slot, uint32_t n,
                                                      uint32_t k, uint64_t* own_key,
                                                      uint32_t* own_slot, uint64_t* gtk) {
  constexpr int R = kF64MaxCap / 64;
  const int lane = threadIdx.x & 63;
  __threadfence_block();  // entries other lanes have stored
  if (n <= 64) {
    const bool in = (uint32_t)lane < n;
    const uint64_t kl = in ? key[lane] : ~0ull;
    const uint32_t sl = in ? slot[lane] : ~0u;
    uint32_t place = 0;
    for (uint32_t t = 0; t < n; t++) {
      const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)kl, t);
      const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(kl >> 32), t);
      place += lex_lt(((uint64_t)hi << 32) | lo, __builtin_amdgcn_readlane(sl, t), kl, sl);
    }
    if (in && place < k) {
      key[place] = kl;
      slot[place] = sl;
    }
    if (in && place == k - 1) {
      *own_key = kl;
      *own_slot = sl;
      __hip_atomic_fetch_min(gtk, kl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }
  uint64_t kv[R];
  uint32_t sv[R];
  uint64_t kmin = ~0ull, kmax = 0;
#pragma unroll
  for (int i = 0; i < R; i++) {
    const uint32_t e = i * 64 + lane;
    kv[i] = e < n ? key[e] : ~0ull;
    sv[i] = e < n ? slot[e] : ~0u;
    kmin = min(kmin, kv[i]);
    if (e < n) kmax = max(kmax, kv[i]);
  }
  for (int o = 32; o >= 1; o >>= 1) {
    kmin = min(kmin, (uint64_t)__shfl_xor((long long)kmin, o));
    kmax = max(kmax, (uint64_t)__shfl_xor((long long)kmax, o));
  }
  uint64_t lo = uni64(kmin), hi = uni64(kmax);
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < R; i++) c += __popcll(__ballot(kv[i] <= mid));
    if (c >= k) hi = mid;
    else lo = mid + 1;
  }
  const uint64_t K = lo;
  uint32_t lt = 0;
#pragma unroll
  for (int i = 0; i < R; i++) lt += __popcll(__ballot(kv[i] < K));
  uint32_t slo = 0, shi = ~0u - 1;  // the (k - lt)-th slot among the keys equal to K
  while (slo < shi) {
    const uint32_t mid = slo + (shi - slo) / 2;
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < R; i++) c += __popcll(__ballot(kv[i] == K && sv[i] <= mid));
    if (c >= k - lt) shi = mid;
    else slo = mid + 1;
  }
  uint32_t base = 0;
#pragma unroll
  for (int i = 0; i < R; i++) {
    const bool keep = kv[i] < K || (kv[i] == K && sv[i] <= slo);
    const uint64_t m = __ballot(keep);
    if (keep) {
      const uint32_t pos = base + __popcll(m & ((1ull << lane) - 1ull));
      key[pos] = kv[i];
      slot[pos] = sv[i];
    }
    base += __popcll(m);
  }
  if (lane == 0) {
    *own_key = K;
    *own_slot = slo;
    __hip_atomic_fetch_min(gtk, K, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// A wavefront's way into its lists.
template <int METRIC>
struct F64Lane {
  const ScanF64Args& a;
  F64Wave& ws;
  size_t list0, list_q;  // query qw's list; from one query's to the next's
  uint32_t qw, r_begin;
  int lane;

  // Row `row` with rank key `kk` enters query j's list if it is to (lanes with
  // c set); true where the list is full, to be tried again once it is cut.
  __device__ __forceinline__ bool append(bool c, uint64_t kk, uint32_t row, int j) {
    if (!(c && kk <= ws.gk[j] && lex_lt(kk, row, ws.own_key[j], ws.own_slot[j]))) return false;
    const uint32_t pos = atomicAdd(&ws.cnt[j], 1u);
    if (pos >= a.kstride) return true;
    // (the list's place is worked out here: kept for each of a lane's four queries
    // it was spilled, and read back ahead of every entry)
    asm volatile("" : "+v"(j));
    const size_t o = list0 + (size_t)(uint32_t)j * list_q + pos;
    a.part_key[o] = kk;
    a.part_slot[o] = row;
    return false;
  }

  // Lists that could not take a row are cut.
  __device__ __forceinline__ void cut_lists() {
    const uint32_t n = lane < kScanTQ ? __hip_atomic_load(&ws.cnt[lane], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_WORKGROUP)
                                      : 0u;
    uint64_t m = __ballot(n > a.kstride);
    while (m) {
      const int j = __ffsll((long long)m) - 1;
      m &= m - 1;
      const uint32_t kj = (uint32_t)a.k[qw + j];
      const size_t o = list0 + (size_t)j * list_q;
      f64_compact(a.part_key + o, a.part_slot + o, a.kstride, kj, &ws.own_key[j],
                  &ws.own_slot[j], a.gtk + qw + j);
      if (lane == 0) ws.cnt[j] = kj;
    }
    __builtin_amdgcn_wave_barrier();
  }

  // n queued pairs, one per lane, get their canonical keys and enter their lists.
  __device__ __forceinline__ void run_batch(uint32_t n) {
    uint32_t v = (uint32_t)lane < n;
    const uint32_t e = v ? ws.queue[lane] : 0u;
    const uint32_t row = r_begin + (e >> 4);
    const int j = (int)(e & 15u);
    uint64_t kk = ~0ull;
    if (v) {
      const uint32_t q = qw + (uint32_t)j;
      double s = exact_chain<METRIC == kL2>(a.st.X + (size_t)row * a.st.ldx,
                                            a.Q + (size_t)q * a.ldq, a.D);
      if (METRIC == kDot) s = -s;
      if (METRIC == kCos) s = -(s / (a.qn[q] * a.st.xn[row]));
      kk = rank_bits(s);
    }
    for (;;) {
      v = append(v != 0, kk, row, j);
      if (__builtin_expect(__ballot(v) == 0, 1)) break;
      cut_lists();
      whole_wave(v);
    }
  }

  // The pairs of the row step at base in `hits` (bit 4t + r) join the queue, qcount
  // long; full batches of 64 are run.
  __device__ __forceinline__ void queue_pairs(uint32_t hits, uint32_t base, uint32_t& qcount) {
    const int g = lane >> 4, jr = lane & 15;
    uint64_t any;
    while ((any = __ballot(hits != 0)) != 0) {
      if (hits) {
        const int b = __ffs((int)hits) - 1;
        hits &= hits - 1;
        const uint32_t row = base + 16 * (b >> 2) + jr;
        ws.queue[qcount + __popcll(any & ((1ull << lane) - 1ull))] =
            ((row - r_begin) << 4) | (uint32_t)(g + 4 * (b & 3));
      }
      qcount += __popcll(any);
      __builtin_amdgcn_wave_barrier();
      if (qcount >= 64) {
        run_batch(64);
        qcount -= 64;
        const uint32_t rest = (uint32_t)lane < qcount ? ws.queue[64 + lane] : 0u;
        __builtin_amdgcn_wave_barrier();
        if ((uint32_t)lane < qcount) ws.queue[lane] = rest;
        __builtin_amdgcn_wave_barrier();
      }
      whole_wave(hits);
    }
  }
};

// The pairs of a row step whose lists were full: their keys are computed again
// (in line, with the keys kept, the accumulators would be live across the cuts
// and the loop over the rows would spill).
template <int METRIC>
__device__ __attribute__((noinline)) void f64_again(const ScanF64Args* a, F64Wave* ws,
                                                    size_t list0, uint32_t qw, uint32_t r_begin,
                                                    uint32_t again, uint32_t base) {
  F64Lane<METRIC> in{*a, *ws, list0, (size_t)a->P * a->kstride, qw, r_begin,
                     (int)(threadIdx.x & 63)};
  uint32_t n = 0;
  in.cut_lists();
  in.queue_pairs(again, base, n);
  if (n) in.run_batch(n);
}

// MINS: the sample; mins[(query · slices + slice) · 16 + lane % 16] gets the
// upper 32 bits of the smallest key (all ones: none).
template <int METRIC, int SC, bool QRES, bool MINS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
k_scan_f64_mfma(ScanF64Args a) {
  constexpr int NT = kF64StageRows / 16;
  constexpr int KS = SC / 4;
  __shared__ __attribute__((aligned(16))) unsigned char buf0[kF64StageRows * SC * 8];
  __shared__ __attribute__((aligned(16))) unsigned char buf1[kF64StageRows * SC * 8];
  // Per-row values of a row step (‖x‖, Σx², the alive words), staged
  // through LDS with the stage loads one row step ahead (two row steps in
  // flight, by parity), so the epilogue reads them from LDS instead of
  // waiting on global memory
  __shared__ __attribute__((aligned(16))) double rowv[2][2][kF64StageRows];
  __shared__ __attribute__((aligned(16))) uint32_t alivew[2][2];
  __shared__ F64Wave wst[kWavesPerBlock];
  const int lane = threadIdx.x & 63;
  // (dot and cosine: in a scalar register, so that nothing spills with 64-column
  // stages; the Euclidean form is faster as it is, 500k × 128: 2,760 µs and 2,840)
  const int wave = METRIC == kL2 ? (int)(threadIdx.x >> 6)
                                 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, jr = lane & 15;
  F64Wave& ws = wst[wave];
  constexpr uint32_t QB = kScanTQ * kWavesPerBlock;
  const uint32_t ngroups = (a.nq + QB - 1) / QB;
  // XCD-aware block order (block ids ≡ x mod 8 run on XCD x): whole slices,
  // with all their query groups one after the other, per XCD, when there are
  // slices for all eight.
  uint32_t group, slice;
  if (a.P % 8 == 0) {
    const uint32_t xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    group = local % ngroups;
    slice = (local / ngroups) * 8 + xcd;
  } else {
    group = blockIdx.x % ngroups;
    slice = blockIdx.x / ngroups;
  }
  const uint32_t qw = group * QB + wave * kScanTQ;  // this wave's first query
  const uint32_t r_begin = slice * a.slice_stride;  // a multiple of 64
  const uint32_t r_end = min(r_begin + a.rows_per_slice, a.st.nrows);
  const uint32_t nsteps =
      r_end > r_begin ? (r_end - r_begin + kF64StageRows - 1) / kF64StageRows : 0;
  const uint32_t npairs = QRES ? 1 : (a.D + 2 * SC - 1) / (2 * SC);  // stage pairs a row step
  const uint32_t qlast = a.nq - 1;
  const bool active = qw < a.nq;  // wave-uniform: a wave past nq only helps load
  const double* __restrict__ qp = a.Q + (size_t)min(qw + jr, qlast) * a.ldq;
  const size_t list0 = ((size_t)min(qw, qlast) * a.P + slice) * a.kstride;  // query qw's list
  const size_t list_q = (size_t)a.P * a.kstride;  // from one query's list to the next's

  if (lane < kScanTQ) {
    ws.cnt[lane] = 0;
    ws.own_key[lane] = ~0ull;
    ws.own_slot[lane] = ~0u;
    ws.gk[lane] = ~0ull;
  }
  double qn4[4], qq4[4];
  bool qv4[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const uint32_t q = min(qw + g + 4 * r, qlast);
    qn4[r] = METRIC != kDot ? a.qn[q] : 0.0;
    qq4[r] = METRIC == kL2 ? a.qq[q] : 0.0;
    qv4[r] = qw + g + 4 * r < a.nq;
  }
  // Euclidean: the constants of l2_bound
  const double crel = (4.0 * a.D + 128.0) * 0x1p-53;
  const double eabs = (8.0 * a.D + 64.0) * 0x1p-1074;
  // lane j: query qw + j's global bound, read once per row step
  uint64_t gk_next = ~0ull;

  f64x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = (f64x4){0.0, 0.0, 0.0, 0.0};
  // query values: the first and second chunk's (QRES), or this stage's and
  // the next one's
  double qa[KS], qb[KS];
  // (whole stages without a test per value, which the compiler turns into a
  // branch each)
  auto load_q = [&](double (&v)[KS], uint32_t col0) __attribute__((always_inline)) {
    if (!QRES && col0 + SC <= a.D) {
      const double* __restrict__ q = qp + col0 + g;
#pragma unroll
      for (int s = 0; s < KS; s++) v[s] = q[4 * s];
      return;
    }
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const uint32_t c = col0 + 4 * s + g;
      v[s] = c < a.D ? qp[c] : 0.0;
    }
  };

  F64Lane<METRIC> in{a, ws, list0, list_q, qw, r_begin, lane};
  uint32_t qcount = 0;  // Euclidean: queued pairs

  // The per-row values of the row step at base into rowv / alivew[par]:
  // wave 0 the norms, wave 1 the squared norms (4-byte direct-to-LDS loads,
  // lane l: dword l&1 of row 32i + l/2, rows clamped to the store), wave 2
  // the alive word (row steps start at a multiple of 64).
  auto issue_rowvals = [&](int par, uint32_t base) __attribute__((always_inline)) {
    const uint32_t last = a.st.nrows - 1;
    if ((wave == 0 && METRIC != kDot) || (wave == 1 && METRIC == kL2)) {
      const double* src = wave == 0 ? a.st.xn : a.st.nx2;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const uint32_t row = min(base + 32 * i + (lane >> 1), last);
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(src + row) + (lane & 1),
                                         (lds_void_t*)&rowv[par][wave][32 * i], 4, 0, 0);
      }
    } else if (wave == 2 && lane < 2) {
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const uint32_t*>(a.st.alive + (base >> 6)) + lane,
          (lds_void_t*)&alivew[par][0], 4, 0, 0);
    }
  };

  // Per-row-step epilogue: which of the step's pairs may enter a list.
  double mins[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
  auto epilogue = [&](uint32_t base, int par) __attribute__((always_inline)) {
    if constexpr (MINS) {
      const uint64_t word = ((uint64_t)alivew[par][1] << 32) | alivew[par][0];
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const bool rv = base + 16 * t + jr < r_end && ((word >> (16 * t + jr)) & 1ull);
        const double xn = METRIC != kDot ? rowv[par][0][16 * t + jr] : 0.0;
        const double xx = METRIC == kL2 ? rowv[par][1][16 * t + jr] : 0.0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          double v;
          if constexpr (METRIC == kDot) v = -acc[t][r];
          else if constexpr (METRIC == kCos) v = -(acc[t][r] / (qn4[r] * xn));
          else v = l2_bound<true>(xx, qq4[r], acc[t][r], xn, qn4[r], crel, eabs);
          if (rv) mins[r] = fmin(mins[r], v);  // (a NaN leaves the minimum)
        }
      }
      return;
    }
    if (lane < kScanTQ) ws.gk[lane] = gk_next;
    __builtin_amdgcn_wave_barrier();
    // each query's bound as a double (NaN while there is none: every
    // comparison below then lets the row through)
    double thr[4];
#pragma unroll
    for (int r = 0; r < 4; r++)
      thr[r] = rank_value(min(ws.gk[g + 4 * r], ws.own_key[g + 4 * r]));
    const uint64_t word = ((uint64_t)alivew[par][1] << 32) | alivew[par][0];
    uint32_t hits = 0;  // bit 4t + r
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const uint32_t row = base + 16 * t + jr;
      const bool rv = row < r_end && ((word >> (16 * t + jr)) & 1ull);
      const double xn = METRIC != kDot ? rowv[par][0][16 * t + jr] : 0.0;
      const double xx = METRIC == kL2 ? rowv[par][1][16 * t + jr] : 0.0;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        bool out;  // surely ranks after the bound
        if constexpr (METRIC == kDot) {
          out = -acc[t][r] > thr[r];
        } else if constexpr (METRIC == kCos) {
          // The key is fl(−dot / w): a quotient above the bound by more than
          // 2^-48 of the bound's magnitude is above it after rounding too (w and
          // thr·w well inside the range of normal numbers).
          const double w = qn4[r] * xn;
          const double m = thr[r] * w, am = fabs(m);
          out = -acc[t][r] > m + 0x1p-48 * am && am > 0x1p-900 && w > 0x1p-900 && w < 0x1p900;
        } else {
          // (an overflowed bound says nothing about its key)
          const double lb = l2_bound<false>(xx, qq4[r], acc[t][r], xn, qn4[r], crel, eabs);
          out = lb > thr[r] && lb < INFINITY;
        }
        hits |= (rv && qv4[r] && !out) ? 1u << (4 * t + r) : 0u;
      }
    }
    if (__builtin_expect(__ballot(hits != 0) == 0, 1)) return;
    if constexpr (METRIC == kL2) {
      in.queue_pairs(hits, base, qcount);
    } else {
      uint32_t again = 0;
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const bool c = (hits >> (4 * t + r)) & 1u;
          if (__ballot(c) == 0) continue;
          const double xn = METRIC == kCos ? rowv[par][0][16 * t + jr] : 0.0;
          const double sc = METRIC == kCos ? -(acc[t][r] / (qn4[r] * xn)) : -acc[t][r];
          if (in.append(c, rank_bits(sc), base + 16 * t + jr, g + 4 * r))
            again |= 1u << (4 * t + r);
        }
      if (__builtin_expect(__ballot(again != 0) != 0, 0))
        // (the arguments where the kernel got them: a pointer to `a` would have
        // every wavefront copy it to its stack)
        f64_again<METRIC>((const ScanF64Args*)__builtin_amdgcn_kernarg_segment_ptr(), &ws, list0,
                          qw, r_begin, again, base);
    }
  };

  if (nsteps > 0) {
    f64_issue_stage<SC>(a.st, buf0, r_begin, 0, wave, lane);
    issue_rowvals(0, r_begin);
    load_q(qa, 0);
    if (QRES) load_q(qb, SC);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  // Whole stages and others have a form each, chosen for both stages of a pair: chosen
  // a stage at a time, the sums were copied once a stage to where the other form
  // keeps them (1M × 768, 1,024 queries, dot: 32.6 → 29.3 ms, 300k × 40, Euclidean:
  // 830 → 773 µs), but with 64-column stages two forms of a pair spill (500k × 100,
  // cosine: 2,444 µs a stage at a time, 2,570 a pair).
  constexpr bool BYSTAGE = SC == 64;
  // One stage's MFMAs: columns col0.. of the rows in `cur`, with query values
  // qv; W: a whole stage.
  auto products = [&](const unsigned char* cur, const double (&qv)[KS], uint32_t col0, auto W)
                      __attribute__((always_inline)) {
    auto kstep = [&](int s) __attribute__((always_inline)) {
      // B operand of tile t: row 16t + j, column 4s + g = unit 2s + g/2, half g&1
      double b[NT];
#pragma unroll
      for (int t = 0; t < NT; t++)
        b[t] = *reinterpret_cast<const double*>(
            cur + f64_unit<SC>(16 * t + jr, 2 * s + (g >> 1)) + (g & 1) * 8);
#pragma unroll
      for (int t = 0; t < NT; t++)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(qv[s], b[t], acc[t], 0, 0, 0);
    };
    if (W || (BYSTAGE && col0 + SC <= a.D)) {
#pragma unroll
      for (int s = 0; s < KS; s++) kstep(s);
    } else {
#pragma unroll
      for (int s = 0; s < KS; s++)
        if (col0 + 4 * s < a.D) kstep(s);
    }
  };
  // A row step's two stages from column col0 on, the last of the step's or not; W:
  // both whole.
  auto pair = [&](uint32_t step, uint32_t base, uint32_t col0, bool last, auto W)
                  __attribute__((always_inline)) {
    // (qa has arrived, but by way of branches that hide it from the compiler:
    // waiting for it at its first use, it would wait for the loads issued next)
    if (!QRES) {
#pragma unroll
      for (int s = 0; s < KS; s++) asm volatile("" : "+v"(qa[s]));
    }
    // first stage: the second one's loads, the MFMAs, then the wait for the
    // loads and for every wave to be done with the buffer
    if (W || col0 + SC < a.D) {
      f64_issue_stage<SC>(a.st, buf1, base, col0 + SC, wave, lane);
      if (!QRES) load_q(qb, col0 + SC);
    }
    if (active) products(buf0, qa, col0, W);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // second stage, with the next pair's or row step's first loads
    if (!last) {
      f64_issue_stage<SC>(a.st, buf0, base, col0 + 2 * SC, wave, lane);
      load_q(qa, col0 + 2 * SC);
    } else if (step + 1 < nsteps) {
      f64_issue_stage<SC>(a.st, buf0, base + kF64StageRows, 0, wave, lane);
      issue_rowvals((step + 1) & 1, base + kF64StageRows);
      if (!QRES) load_q(qa, 0);
    }
    if (active && (W || col0 + SC < a.D)) products(buf1, qb, col0 + SC, W);
    if (!last) {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  };
  const uint32_t nwhole = BYSTAGE ? 0 : a.D / (2 * SC);
  for (uint32_t step = 0; step < nsteps; step++) {
    const uint32_t base = r_begin + step * kF64StageRows;
    // the global bounds for this row step's epilogue, read at its first
    // stage so the load's latency runs under the step's MFMAs
    if (!MINS && lane < kScanTQ)
      gk_next = __hip_atomic_load(a.gtk + min(qw + lane, qlast), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t pr = 0; pr < nwhole; pr++)
      pair(step, base, pr * 2 * SC, pr + 1 == npairs, std::true_type{});
    if (nwhole < npairs) pair(step, base, nwhole * 2 * SC, true, std::false_type{});
    if (active) {
      epilogue(base, step & 1);
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = (f64x4){0.0, 0.0, 0.0, 0.0};
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (!active) return;
  if constexpr (MINS) {
    uint32_t* out = reinterpret_cast<uint32_t*>(a.part_key);
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (qv4[r])
        out[((size_t)(qw + g + 4 * r) * a.P + slice) * 16 + jr] =
            mins[r] < INFINITY ? (uint32_t)(rank_bits(mins[r]) >> 32) : ~0u;
    return;
  }
  if (METRIC == kL2 && qcount) in.run_batch(qcount);
  __builtin_amdgcn_wave_barrier();
  if (lane < kScanTQ && qw + lane < a.nq)
    a.part_cnt[(size_t)(qw + lane) * a.P + slice] = ws.cnt[lane];
}

// Every column compared, rows in whole 16-byte loads and zero past D;
// Euclidean needs the squared row norms, which cover every column: a column
// prefix (kd-tree dimension below the row width) stays on the VALU scan.
bool scan_f64_uses_mfma(int metric, uint32_t D, const StoreView& st) {
  return D > 0 && st.ldx % 8 == 0 && D <= st.ldx && D + 8 > st.ldx &&
         ((uintptr_t)st.X & 15) == 0 && st.nx2 != nullptr && metric >= 0;
}

// gtk[q] = a rank key at or above the k-th of the n sample minima of query q
// (their upper 32 bits, the lower ones set); all ones when there are fewer.
// One wavefront per query bisects the bits with counts over the wavefront.
constexpr uint32_t kMinsPerLane = 16;

__global__ __launch_bounds__(256) void k_bound_f64(const uint32_t* __restrict__ mins, uint32_t n,
                                                   uint32_t nq, const int* __restrict__ k,
                                                   uint64_t* __restrict__ gtk) {
  const int lane = threadIdx.x & 63;
  const uint32_t q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= nq) return;
  const uint32_t kk = (uint32_t)k[q];
  uint32_t u[kMinsPerLane];
  uint32_t lo = ~0u;
#pragma unroll
  for (uint32_t i = 0; i < kMinsPerLane; i++) {
    const uint32_t c = i * 64 + lane;
    u[i] = c < n ? mins[(size_t)q * n + c] : ~0u;
    lo = min(lo, u[i]);
  }
  for (int o = 32; o >= 1; o >>= 1) lo = min(lo, (uint32_t)__shfl_xor((int)lo, o));
  uint32_t hi = ~0u;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    uint32_t c = 0;
#pragma unroll
    for (uint32_t i = 0; i < kMinsPerLane; i++) c += __popcll(__ballot(u[i] <= mid));
    if (c >= kk) hi = mid;
    else lo = mid + 1;
  }
  if (lane == 0) gtk[q] = ((uint64_t)lo << 32) | 0xFFFFFFFFull;
}

template <int METRIC, bool MINS>
static hipError_t scan_f64_mfma_t(const ScanF64Args& a, hipStream_t s) {
  constexpr uint32_t QB = kScanTQ * kWavesPerBlock;
  const dim3 grid(((a.nq + QB - 1) / QB) * a.P);
  if (a.D <= 64)
    hipLaunchKernelGGL((k_scan_f64_mfma<METRIC, 32, true, MINS>), grid, dim3(256), 0, s, a);
  else if (a.D <= 128)
    hipLaunchKernelGGL((k_scan_f64_mfma<METRIC, 64, true, MINS>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_scan_f64_mfma<METRIC, 32, false, MINS>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

template <bool MINS>
static hipError_t scan_f64_mfma_m(const ScanF64Args& a, int metric, hipStream_t s) {
  switch (metric) {
    case kL2: return scan_f64_mfma_t<kL2, MINS>(a, s);
    case kCos: return scan_f64_mfma_t<kCos, MINS>(a, s);
    case kDot: return scan_f64_mfma_t<kDot, MINS>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_scan_f64_mfma(const ScanF64Args& a, int metric, int kmax, hipStream_t s) {
  if (a.nq == 0 || a.P == 0) return hipSuccess;
  if (!scan_f64_uses_mfma(metric, a.D, a.st) || !a.gtk || !a.part_cnt ||
      a.kstride > kF64MaxCap || (metric == kL2 && !a.qq))
    return hipErrorInvalidValue;
  const uint32_t rows = f64_slice_rows(a.st.nrows, a.P);
  if (a.kstride <= (uint32_t)kmax && a.kstride < rows) return hipErrorInvalidValue;
  ScanF64Args m = a;
  hipError_t e;
  // The sample; the minima lie where the lists will.
  const uint32_t S =
      f64_sample_runs(a.st.nrows, kmax, a.D, (size_t)a.P * a.kstride / 8);
  if (S) {
    m.P = S;
    m.slice_stride = a.st.nrows / S / 64 * 64;
    m.rows_per_slice = std::max<uint32_t>(64, a.st.nrows / f64_share(a.D) / S / 64 * 64);
    if ((e = scan_f64_mfma_m<true>(m, metric, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_bound_f64, dim3((a.nq + 3) / 4), dim3(256), 0, s,
                       reinterpret_cast<const uint32_t*>(a.part_key), 16 * S, a.nq, a.k, a.gtk);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  } else {
    e = launch_fill_i32(reinterpret_cast<int*>(a.gtk), 2 * a.nq, -1, s);
    if (e != hipSuccess) return e;
  }
  m.P = a.P;
  m.rows_per_slice = m.slice_stride = rows;
  return scan_f64_mfma_m<false>(m, metric, s);
}

// ---------------------------------------------------------- selection
//
// One block per query: of the lists' entries with keys at most gtk (a bound on
// the k-th), packed into LDS, each finds its place by counting the entries
// before it.  More than kCountMax are first counted into 256 bins of the key
// range that holds the k-th until at most kCountMax lie at or below its bin;
// where equal keys prevent that, they are cut by slot the same way to exactly
// k.  Entries past the LDS capacity are read again from the lists.  16 lanes
// take a list, four lists in flight.  Ids and scores are written in rank order.
// 77 queries at k = 100 15 µs, 1,024 at k = 10 27 µs (a wavefront per query
// merging sorted lists: 1,000 and 29).
constexpr uint32_t kF64SelCap = 2048;
constexpr uint32_t kCountMax = 512;

template <int T>
struct F64Sel {
  uint64_t key[kF64SelCap];
  uint32_t slot[kF64SelCap];
  uint64_t fkey[kCountMax];
  uint32_t fslot[kCountMax];
  uint32_t hist[256];
  unsigned long long lo, hi;
  uint32_t n, rank, le, nf;
};

template <int T>
__global__ __launch_bounds__(T) void k_select_f64(MergeArgs a, const uint32_t* __restrict__ cnt,
                                                  const uint64_t* __restrict__ gtk, int metric) {
  __shared__ F64Sel<T> sm;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t q = blockIdx.x;
  const uint32_t kk = (uint32_t)a.k[q];
  const uint64_t bound = gtk[q];
  const uint64_t* __restrict__ pkey = a.part_key + (size_t)q * a.P * a.kstride;
  const uint32_t* __restrict__ pslot = a.part_slot + (size_t)q * a.P * a.kstride;
  const uint32_t* __restrict__ pc = cnt + (size_t)q * a.P;
  if (tid == 0) {
    sm.n = 0;
    sm.nf = 0;
    sm.lo = ~0ull;
    sm.hi = 0;
  }
  __syncthreads();
  // f(key, slot) for every entry at or below the bound, in the lists (four
  // lists' counts, then their first entries, in flight together)
  auto lists = [&](auto&& f) __attribute__((always_inline)) {
    constexpr uint32_t G = T / 16, U = 4;
    for (uint32_t l0 = tid >> 4; l0 < a.P; l0 += G * U) {
      uint32_t m[U];
      uint64_t k0[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) m[u] = l0 + u * G < a.P ? pc[l0 + u * G] : 0u;
#pragma unroll
      for (uint32_t u = 0; u < U; u++)
        k0[u] = (uint32_t)(tid & 15) < m[u] ? pkey[(size_t)(l0 + u * G) * a.kstride + (tid & 15)]
                                            : ~0ull;
#pragma unroll
      for (uint32_t u = 0; u < U; u++)
        for (uint32_t e = tid & 15; e < m[u]; e += 16) {
          const size_t o = (size_t)(l0 + u * G) * a.kstride + e;
          const uint64_t k = e < 16 ? k0[u] : pkey[o];
          if (k <= bound) f(k, pslot[o]);
        }
    }
  };
  uint64_t lo = ~0ull, hi = 0;
  lists([&](uint64_t k, uint32_t s) {
    lo = min(lo, k);
    hi = max(hi, k);
    const uint32_t pos = atomicAdd(&sm.n, 1u);
    if (pos < kF64SelCap) {
      sm.key[pos] = k;
      sm.slot[pos] = s;
    }
  });
  for (int o = 32; o >= 1; o >>= 1) {
    lo = min(lo, (uint64_t)__shfl_xor((long long)lo, o));
    hi = max(hi, (uint64_t)__shfl_xor((long long)hi, o));
  }
  if (lane == 0) {
    atomicMin(&sm.lo, (unsigned long long)lo);
    atomicMax(&sm.hi, (unsigned long long)hi);
  }
  __syncthreads();
  const uint32_t n = sm.n;
  auto each = [&](auto&& f) __attribute__((always_inline)) {
    if (n <= kF64SelCap) {
      for (uint32_t c = tid; c < n; c += T) f(sm.key[c], sm.slot[c]);
    } else {
      lists(f);
    }
  };
  auto put = [&](uint64_t k, uint32_t s, uint32_t place) __attribute__((always_inline)) {
    const double v = rank_value(k);
    double sc = __longlong_as_double(0x7FF8000000000000ll);
    // NaN keys come back as the one canonical quiet NaN (its sign is
    // not meaningful); a zero dot/cos rank key is a +0 score.
    if (v == v) sc = metric == kL2 ? sqrt(v) : (v == 0.0 ? 0.0 : -v);
    a.ids[(size_t)q * a.ostride + place] = logical_id(a.st, s);
    a.scores[(size_t)q * a.ostride + place] = sc;
  };
  auto place_all = [&](const uint64_t* key, const uint32_t* slot, uint32_t m)
                       __attribute__((always_inline)) {
    for (uint32_t c = tid; c < m; c += T) {
      const uint64_t k = key[c];
      const uint32_t s = slot[c];
      uint32_t place = 0;
      for (uint32_t t = 0; t < m; t++) place += lex_lt(key[t], slot[t], k, s);
      if (place < kk) put(k, s, place);
    }
  };
  for (uint32_t e = n + tid; e < kk; e += T) {
    a.ids[(size_t)q * a.ostride + e] = ~0ull;
    a.scores[(size_t)q * a.ostride + e] = __longlong_as_double(0x7FF8000000000000ll);
  }
  if (n <= kCountMax) {
    place_all(sm.key, sm.slot, n);
    return;
  }
  // Narrows [sm.lo, sm.hi] to the bin of the values that holds the sm.rank-th
  // smallest of those `in` counts (the values below sm.lo, sm.le with those in
  // the range, are taken), until few enough lie at or below it or it holds one
  // value.
  auto narrow = [&](auto&& value, auto&& in) {
    for (;;) {
      const uint64_t l = sm.lo, h = sm.hi;
      if (l == h || sm.le <= kCountMax) break;
      const int shift = bin_shift(h - l);
      for (int b = tid; b < 256; b += T) sm.hist[b] = 0;
      __syncthreads();
      each([&](uint64_t k, uint32_t s) {
        const uint64_t v = value(k, s);
        if (in(k, s) && v >= l && v <= h) atomicAdd(&sm.hist[(v - l) >> shift], 1u);
      });
      __syncthreads();
      if (wave == 0) {
        const uint32_t hs[4] = {sm.hist[4 * lane], sm.hist[4 * lane + 1], sm.hist[4 * lane + 2],
                                sm.hist[4 * lane + 3]};
        const uint32_t sum = hs[0] + hs[1] + hs[2] + hs[3];
        uint32_t inc = sum;
        for (int off = 1; off < 64; off <<= 1) {
          const uint32_t v = __shfl_up(inc, off);
          if (lane >= off) inc += v;
        }
        const uint32_t total = __shfl(inc, 63);  // of [l, h]
        const uint32_t exc = inc - sum, r = sm.rank;
        if (exc < r && r <= inc) {
          uint32_t cum = exc, here = 0, bin = 4 * lane;
#pragma unroll
          for (int b = 0; b < 4; b++)
            if (bin == 4u * lane + b) {
              here = hs[b];
              if (cum + hs[b] < r) {
                cum += hs[b];
                bin++;
              }
            }
          sm.le = sm.le - total + cum + here;
          sm.rank = r - cum;
          sm.lo = l + ((uint64_t)bin << shift);
          sm.hi = bin_last(l, h, bin, shift);
        }
      }
      __syncthreads();
    }
  };
  if (tid == 0) {
    sm.rank = kk;
    sm.le = n;
  }
  __syncthreads();
  narrow([](uint64_t k, uint32_t) { return k; }, [](uint64_t, uint32_t) { return true; });
  const uint64_t K = sm.hi;
  uint64_t S = ~0ull;
  if (sm.le > kCountMax) {
    // more than kCountMax keys up to the k-th: of those equal to it, the
    // lowest slots
    const uint32_t rank = sm.rank;
    __syncthreads();
    if (tid == 0) {
      sm.lo = 0;
      sm.hi = 0xFFFFFFFFull;
      sm.rank = rank;
    }
    __syncthreads();
    narrow([](uint64_t, uint32_t s) { return (uint64_t)s; },
           [&](uint64_t k, uint32_t) { return k == K; });
    S = sm.hi;
  }
  each([&](uint64_t k, uint32_t s) {
    if (k < K || (k == K && s <= S)) {
      const uint32_t pos = atomicAdd(&sm.nf, 1u);
      sm.fkey[pos] = k;
      sm.fslot[pos] = s;
    }
  });
  __syncthreads();
  place_all(sm.fkey, sm.fslot, sm.nf);
}

hipError_t launch_select_f64(const MergeArgs& m, const uint32_t* cnt, const uint64_t* gtk,
                             int metric, hipStream_t s) {
  if (m.nq == 0) return hipSuccess;
  if (m.nq <= 256)
    hipLaunchKernelGGL(k_select_f64<1024>, dim3(m.nq), dim3(1024), 0, s, m, cnt, gtk, metric);
  else
    hipLaunchKernelGGL(k_select_f64<256>, dim3(m.nq), dim3(256), 0, s, m, cnt, gtk, metric);
  return hipGetLastError();
}

}  // namespace svdb
