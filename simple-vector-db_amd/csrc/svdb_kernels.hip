// svdb_kernels.hip — gfx950 kernels of the similarity / nearest-vector path.
//
// Built with -ffp-contract=off: every a*b+c below that is not an explicit
// fma() is a rounded multiply then a rounded add; the explicit fma() calls
// are the canonical FP64 steps (correctly rounded v_fma_f64).  sqrt and '/'
// on doubles lower to the correctly rounded sequences (v_rsq_f64 + Newton
// steps + fixup; v_div_scale/v_div_fmas/v_div_fixup).
//
// Canonical FP64 arithmetic (matches oracle/svdb_oracle.c bit for bit):
//   L2 key  s = Σ_i fma(t, t, s), t = x_i - q_i, i = 0..D-1 in order
//   dot key s = Σ_i fma(q_i, x_i, s)
//   cosine  dot / (sqrt(Σ fma(q,q)) * sqrt(Σ fma(x,x)))
// Ranking: ascending "rank key" (L2: s; dot/cos: -score) mapped to a uint64
// that orders like the doubles (-0 folded to +0, NaN above +inf), then the
// slot (physical row), which orders like the logical index.
#include "svdb_kernels.h"

#include <math.h>

#include <algorithm>

#include "svdb_rank.h"

namespace svdb {

// ----------------------------------------------------------------- helpers

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t uniform32(uint32_t v) {
  return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ uint64_t read_lane64(uint64_t v, int l) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, l);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), l);
  return ((uint64_t)hi << 32) | lo;
}

// A sorted list of (key, slot) spread over a wavefront: entry e lives in
// lane e % 64, register e / 64.  Unused entries hold the sentinel
// (UINT64_MAX, UINT32_MAX), which is above every real entry (slots are
// < UINT32_MAX).
template <int KPL>
struct WList {
  uint64_t k[KPL];
  uint32_t s[KPL];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int p = 0; p < KPL; p++) {
      k[p] = ~0ull;
      s[p] = ~0u;
    }
  }
  // Entry kk-1 (the current k-th best), wave-uniform.
  __device__ __forceinline__ void kth(int kk, uint64_t& tk, uint32_t& ts) const {
    int e = kk - 1, p = e >> 6, ln = e & 63;
    uint64_t a = k[0];
    uint32_t b = s[0];
#pragma unroll
    for (int q = 1; q < KPL; q++)
      if (p == q) {
        a = k[q];
        b = s[q];
      }
    tk = uniform64(__shfl(a, ln));
    ts = uniform32(__shfl(b, ln));
  }
  // Insert (K, S) (wave-uniform) keeping the first kk entries the kk best.
  __device__ __forceinline__ void insert(uint64_t K, uint32_t S, int kk, int lane) {
    int pos = 0;
#pragma unroll
    for (int p = 0; p < KPL; p++) pos += __popcll(__ballot(lex_lt(k[p], s[p], K, S)));
    if (pos >= kk) return;
    uint64_t pk[KPL];
    uint32_t ps[KPL];
#pragma unroll
    for (int p = 0; p < KPL; p++) {
      pk[p] = __shfl_up(k[p], 1);
      ps[p] = __shfl_up(s[p], 1);
    }
#pragma unroll
    for (int p = 1; p < KPL; p++) {
      uint64_t ck = __shfl(k[p - 1], 63);
      uint32_t cs = __shfl(s[p - 1], 63);
      if (lane == 0) {
        pk[p] = ck;
        ps[p] = cs;
      }
    }
#pragma unroll
    for (int p = 0; p < KPL; p++) {
      int e = p * 64 + lane;
      if (e > pos) {
        k[p] = pk[p];
        s[p] = ps[p];
      } else if (e == pos) {
        k[p] = K;
        s[p] = S;
      }
    }
  }
};

// ------------------------------------------------------------ store writes

// ‖·‖ and its square (the sequential fma chain) of n rows of D columns, stored
// rows or queries.  One wavefront per row: coalesced loads into LDS, 512
// columns at a time, then the chain over broadcast reads, 16 columns per step.
// A thread per row had a load latency per column on the chain: 77 rows of 100
// columns 14 µs, now 3; 500k of 128 columns 770 µs, now 260.
__global__ __launch_bounds__(256) void k_row_norms(const double* __restrict__ Q, size_t ldq,
                                                     uint32_t nq, uint32_t D,
                                                     double* __restrict__ qn,
                                                     double* __restrict__ qq) {
  constexpr int CH = 512;
  __shared__ __attribute__((aligned(16))) double row[4][CH];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t i = blockIdx.x * 4 + wave;
  if (i >= nq) return;
  const double* q = Q + (size_t)i * ldq;
  double acc = 0.0;
  for (uint32_t c0 = 0; c0 < D; c0 += CH) {
    const uint32_t m = min((uint32_t)CH, (D - c0 + 15) & ~15u);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < CH / 64; j++) {
      const uint32_t c = j * 64 + lane;
      if (c < m) row[wave][c] = c0 + c < D ? q[c0 + c] : 0.0;
    }
    __builtin_amdgcn_wave_barrier();
    // (the zeros past D leave the chain as it is)
    for (uint32_t c = 0; c < m; c += 16) {
      double x[16];
#pragma unroll
      for (int j = 0; j < 16; j++) x[j] = row[wave][c + j];
#pragma unroll
      for (int j = 0; j < 16; j++) acc = fma(x[j], x[j], acc);
    }
  }
  if (lane == 0) {
    qn[i] = sqrt(acc);
    if (qq) qq[i] = acc;
  }
}

hipError_t launch_query_norms(const double* Q, size_t ldq, uint32_t nq, uint32_t D, double* qn,
                              double* qq, hipStream_t s) {
  if (nq == 0) return hipSuccess;
  hipLaunchKernelGGL(k_row_norms, dim3((nq + 3) / 4), dim3(256), 0, s, Q, ldq, nq, D, qn, qq);
  return hipGetLastError();
}

hipError_t launch_row_norms(const double* X, size_t ldx, uint32_t first, uint32_t n, uint32_t d,
                            double* nx2, double* xn, hipStream_t s) {
  return launch_query_norms(X + (size_t)first * ldx, ldx, n, d, xn + first, nx2 + first, s);
}

// Plain device copy, 16 bytes per lane, grid-stride (also the known-traffic
// reference for hardware byte counters: it reads and writes `bytes` once).
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n16) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n16;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

__global__ void k_copy1(const unsigned char* __restrict__ src, unsigned char* __restrict__ dst,
                        size_t n) {
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

hipError_t launch_copy(const void* src, void* dst, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const bool aligned = ((uintptr_t)src % 16 == 0) && ((uintptr_t)dst % 16 == 0);
  const size_t n16 = aligned ? bytes / 16 : 0;
  if (n16) {
    const size_t blocks = std::min<size_t>((n16 + 255) / 256, 256 * 32);
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, s, (const uint4*)src,
                       (uint4*)dst, n16);
  }
  const size_t rest = bytes - n16 * 16;
  if (rest)
    hipLaunchKernelGGL(k_copy1, dim3((unsigned)((rest + 255) / 256)), dim3(256), 0, s,
                       (const unsigned char*)src + n16 * 16, (unsigned char*)dst + n16 * 16, rest);
  return hipGetLastError();
}

__global__ void k_fill_i32(int* __restrict__ p, uint32_t n, int v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

hipError_t launch_fill_i32(int* p, uint32_t n, int v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_i32, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

// ------------------------------------- FP64 scan of a column prefix, Euclidean
//
// kdtree_nearest and svdb_search over fewer columns than the rows have (every
// column: the matrix-core scan, svdb_scan_f64.hip).
//
// Grid (query groups of kScanTQ, row slices); 4 wavefronts per block share
// the block's queries and take interleaved 128-row steps of the slice.  Each
// lane owns two rows per step (row base+lane and base+64+lane) and keeps the
// kScanTQ×2 FP64 accumulators; query values are wave-uniform loads.  After
// a step every (query, row) key is tested against that query's current k-th
// best (wave-uniform); hits are inserted into the query's wave-distributed
// sorted list.  Each wavefront writes its lists as one partial list per
// query.

__device__ __forceinline__ void accum8(double (&acc)[kScanTQ][2], const double (&x0)[8],
                                       const double (&x1)[8], const double* __restrict__ Qg,
                                       size_t ldq, uint32_t c) {
  // Queries in groups of G: a group's 8·G values are scalar loads, and the
  // next group's loads are issued (into the other of two register sets)
  // before this group's fmas, with scheduling barriers keeping it that way —
  // left to itself the compiler hoists all 16 queries' loads to the top
  // (256 scalar registers) and spills most of them.  A group's 2·G
  // (query, row) chains interleave; every chain advances in element order.
  constexpr int G = 2;
  constexpr int NG = kScanTQ / G;
  double qv[2][G][8];
#pragma unroll
  for (int jj = 0; jj < G; jj++)
#pragma unroll
    for (int i = 0; i < 8; i++) qv[0][jj][i] = Qg[(size_t)jj * ldq + c + i];
#pragma unroll
  for (int g = 0; g < NG; g++) {
    if (g + 1 < NG) {
#pragma unroll
      for (int jj = 0; jj < G; jj++)
#pragma unroll
        for (int i = 0; i < 8; i++)
          qv[(g + 1) & 1][jj][i] = Qg[(size_t)((g + 1) * G + jj) * ldq + c + i];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; i++) {
#pragma unroll
      for (int jj = 0; jj < G; jj++) {
        const int j = g * G + jj;
        const double q = qv[g & 1][jj][i];
        double t0 = x0[i] - q, t1 = x1[i] - q;
        acc[j][0] = fma(t0, t0, acc[j][0]);
        acc[j][1] = fma(t1, t1, acc[j][1]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int KPL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KPL == 1 ? 3 : 2))) void
k_scan_f64(ScanF64Args a) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // XCD-aware block order: block ids ≡ x (mod 8) run on XCD x, which gets
  // whole slices (slice ≡ x mod 8) with all their query groups one after
  // the other; the groups of a slice then stream its rows through that
  // XCD's L2 in near lockstep instead of each from HBM.
  const uint32_t ngroups = (a.nq + kScanTQ - 1) / kScanTQ;
  const uint32_t xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  const uint32_t q0 = (local % ngroups) * kScanTQ;
  const uint32_t slice = (local / ngroups) * 8 + xcd;
  const uint32_t r_begin = slice * a.rows_per_slice;
  const uint32_t r_end = min(r_begin + a.rows_per_slice, a.st.nrows);
  // Queries past nq reuse the last query's row (their lists are not written).
  const uint32_t qlast = a.nq - 1;
  const double* __restrict__ Qg = a.Q + (size_t)min(q0, qlast) * a.ldq;
  const bool full_group = q0 + kScanTQ <= a.nq;

  WList<KPL> L[kScanTQ];
  // Per-query state, lane j holding query j's: the current k-th best
  // (key, slot) and k.  Kept in vector registers and read
  // into scalars one query at a time in the epilogue: as arrays of
  // wave-uniform values they needed about 100 scalar registers and the
  // kernel spilled scalars throughout its main loop.
  uint64_t tk_l = ~0ull;
  uint32_t ts_l = ~0u;
  int kq_l = 0;
  if (lane < kScanTQ) kq_l = a.k[min(q0 + lane, qlast)];
#pragma unroll
  for (int j = 0; j < kScanTQ; j++) L[j].init();

  for (uint32_t base = r_begin + wave * kScanRows; base < r_end;
       base += kWavesPerBlock * kScanRows) {
    const uint32_t r0 = base + lane, r1 = base + 64 + lane;
    const uint32_t c0 = min(r0, a.st.nrows - 1), c1 = min(r1, a.st.nrows - 1);
    const double* __restrict__ x0p = a.st.X + (size_t)c0 * a.st.ldx;
    const double* __restrict__ x1p = a.st.X + (size_t)c1 * a.st.ldx;
    double acc[kScanTQ][2];
#pragma unroll
    for (int j = 0; j < kScanTQ; j++) acc[j][0] = acc[j][1] = 0.0;

    uint32_t c = 0;
    if (full_group) {
      for (; c + 8 <= a.D; c += 8) {
        double x0[8], x1[8];
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          double2 v0 = *reinterpret_cast<const double2*>(x0p + c + i);
          double2 v1 = *reinterpret_cast<const double2*>(x1p + c + i);
          x0[i] = v0.x; x0[i + 1] = v0.y;
          x1[i] = v1.x; x1[i + 1] = v1.y;
        }
        accum8(acc, x0, x1, Qg, a.ldq, c);
      }
    }
    for (; c < a.D; c++) {
      double xa = x0p[c], xb = x1p[c];
#pragma unroll
      for (int j = 0; j < kScanTQ; j++) {
        double q = a.Q[(size_t)min(q0 + j, qlast) * a.ldq + c];
        double t0 = xa - q, t1 = xb - q;
        acc[j][0] = fma(t0, t0, acc[j][0]);
        acc[j][1] = fma(t1, t1, acc[j][1]);
      }
    }

    const bool v0 = r0 < r_end && slot_alive(a.st.alive, c0);
    const bool v1 = r1 < r_end && slot_alive(a.st.alive, c1);
    // lane j: query q0 + j's global bound (the smallest k-th key any list
    // of the query has published; rows with keys above it are out)
    uint64_t gk_l = ~0ull;
    if (a.gtk && lane < kScanTQ)
      gk_l = __hip_atomic_load(a.gtk + min(q0 + lane, qlast), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 0; j < kScanTQ; j++) {
      uint64_t tkj = read_lane64(tk_l, j);
      uint32_t tsj = __builtin_amdgcn_readlane(ts_l, j);
      const int kqj = __builtin_amdgcn_readlane(kq_l, j);
      const uint64_t gkj = read_lane64(gk_l, j);
      const uint64_t k0 = rank_bits(acc[j][0]), k1 = rank_bits(acc[j][1]);
      // slots past nq (a partial group) keep no list
      const bool jv = q0 + j < a.nq;
      uint64_t m0 = __ballot(jv && v0 && k0 <= gkj && lex_lt(k0, r0, tkj, tsj));
      uint64_t m1 = __ballot(jv && v1 && k1 <= gkj && lex_lt(k1, r1, tkj, tsj));
      // After each insertion the k-th entry may have moved: lanes that no
      // longer beat it drop out (their insertion would change nothing).
      const bool moved = (m0 | m1) != 0;
      while (m0) {
        int src = __ffsll((long long)m0) - 1;
        m0 &= m0 - 1;
        L[j].insert(uniform64(__shfl(k0, src)), base + src, kqj, lane);
        L[j].kth(kqj, tkj, tsj);
        m0 &= __ballot(lex_lt(k0, r0, tkj, tsj));
      }
      m1 &= __ballot(lex_lt(k1, r1, tkj, tsj));
      while (m1) {
        int src = __ffsll((long long)m1) - 1;
        m1 &= m1 - 1;
        L[j].insert(uniform64(__shfl(k1, src)), base + 64 + src, kqj, lane);
        L[j].kth(kqj, tkj, tsj);
        m1 &= __ballot(lex_lt(k1, r1, tkj, tsj));
      }
      if (moved && lane == j) {
        tk_l = tkj;
        ts_l = tsj;
        // a full list publishes its k-th key
        if (a.gtk && tkj != ~0ull && tkj < gk_l)
          __hip_atomic_fetch_min(a.gtk + q0 + j, tkj, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }

  const uint32_t list = slice * kWavesPerBlock + wave;
#pragma unroll
  for (int j = 0; j < kScanTQ; j++) {
    if (q0 + j >= a.nq) break;
    const int kqj = __builtin_amdgcn_readlane(kq_l, j);
    size_t o = ((size_t)(q0 + j) * a.P + list) * a.kstride;
#pragma unroll
    for (int p = 0; p < KPL; p++) {
      int e = p * 64 + lane;
      if (e < kqj) {
        a.part_key[o + e] = L[j].k[p];
        a.part_slot[o + e] = L[j].s[p];
      }
    }
  }
}

hipError_t launch_scan_f64(const ScanF64Args& a, int kmax, uint32_t nslices, hipStream_t s) {
  if (a.nq == 0) return hipSuccess;
  // nslices is a multiple of 8 (one set of slices per XCD); 1-D grid
  if (nslices % 8 || a.P != nslices * kWavesPerBlock) return hipErrorInvalidValue;
  const dim3 grid(((a.nq + kScanTQ - 1) / kScanTQ) * nslices);
  if (kmax > 64) hipLaunchKernelGGL(k_scan_f64<2>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_scan_f64<1>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

// ------------------------------------------------ one query, nearest row
//
// kdtree_nearest called once per request (the reference's handlers do) on a
// store small enough to scan in microseconds: the launch, not the scan, is
// the cost, so the whole answer is one kernel — no query upload (the query
// travels in the kernel arguments), no merge launch, no result copy (the
// last block writes the id to host memory).  The blocks' results meet
// through a ticket: every block publishes its (key, slot) and takes a
// ticket (release/acquire at agent scope); the block holding the last
// ticket reads them all.

__device__ __forceinline__ void min_pair(uint64_t& bk, uint32_t& bs, uint64_t k, uint32_t s) {
  if (lex_lt(k, s, bk, bs)) {
    bk = k;
    bs = s;
  }
}

__global__ __launch_bounds__(256) void k_nearest1(const Nearest1Args a) {
  __shared__ uint64_t wk[4];
  __shared__ uint32_t ws[4];
  __shared__ int last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t bk = ~0ull;
  uint32_t bs = ~0u;
  for (uint32_t r = blockIdx.x * 256 + threadIdx.x; r < a.st.nrows; r += gridDim.x * 256) {
    if (!slot_alive(a.st.alive, r)) continue;
    const double* __restrict__ x = a.st.X + (size_t)r * a.st.ldx;
    double s = 0.0;
    for (uint32_t i = 0; i < a.D; i++) {
      const double t = x[i] - a.q[i];
      s = fma(t, t, s);
    }
    min_pair(bk, bs, rank_bits(s), r);
  }
  auto block_min = [&]() {
    for (int off = 32; off >= 1; off >>= 1) {
      const uint64_t ok = (uint64_t)__shfl_xor((long long)bk, off);
      const uint32_t os = (uint32_t)__shfl_xor((int)bs, off);
      min_pair(bk, bs, ok, os);
    }
    if (lane == 0) {
      wk[wave] = bk;
      ws[wave] = bs;
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < 4; w++) min_pair(bk, bs, wk[w], ws[w]);
  };
  block_min();
  if (threadIdx.x == 0) {
    __hip_atomic_store(a.part_key + blockIdx.x, bk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(a.part_slot + blockIdx.x, bs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t t =
        __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    last = t == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  bk = ~0ull;
  bs = ~0u;
  for (uint32_t b = threadIdx.x; b < gridDim.x; b += 256)
    min_pair(bk, bs, __hip_atomic_load(a.part_key + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
             __hip_atomic_load(a.part_slot + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  __syncthreads();  // wk / ws are reused
  block_min();
  if (threadIdx.x == 0) {
    __hip_atomic_store(a.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    a.out_id[0] = bs == ~0u ? ~0ull : logical_id(a.st, bs);
    __threadfence_system();
    __hip_atomic_store(a.out_id + 1, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

hipError_t launch_nearest1(const Nearest1Args& a, hipStream_t s) {
  if (a.D == 0 || a.D > kNearestMaxD || a.st.nrows == 0) return hipErrorInvalidValue;
  const uint32_t blocks =
      std::min<uint32_t>(kNearestMaxBlocks, (a.st.nrows + 255) / 256);
  hipLaunchKernelGGL(k_nearest1, dim3(blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------- list merge
//
// One wavefront per query merges the query's P sorted partial lists into
// its final top-k, then writes logical ids and FP64 scores.  A partial list
// whose first entry does not beat the current k-th best is skipped whole.

template <int KPL>
__global__ __launch_bounds__(256) void k_merge(MergeArgs a) {
  const int lane = threadIdx.x & 63;
  const uint32_t q = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (q >= a.nq) return;
  const int kk = a.k[q];
  WList<KPL> L;
  L.init();
  uint64_t tk = ~0ull;
  uint32_t ts = ~0u;
  for (uint32_t p = 0; p < a.P; p++) {
    const size_t o = ((size_t)q * a.P + p) * a.kstride;
    const uint64_t e0k = uniform64(a.part_key[o]);
    const uint32_t e0s = uniform32(a.part_slot[o]);
    if (!lex_lt(e0k, e0s, tk, ts)) continue;
#pragma unroll
    for (int pp = 0; pp < KPL; pp++) {
      const int e = pp * 64 + lane;
      uint64_t ck = ~0ull;
      uint32_t cs = ~0u;
      if (e < kk) {
        ck = a.part_key[o + e];
        cs = a.part_slot[o + e];
      }
      uint64_t m = __ballot(lex_lt(ck, cs, tk, ts));
      while (m) {
        int src = __ffsll((long long)m) - 1;
        m &= m - 1;
        L.insert(uniform64(__shfl(ck, src)), uniform32(__shfl(cs, src)), kk, lane);
        L.kth(kk, tk, ts);
        m &= __ballot(lex_lt(ck, cs, tk, ts));
      }
    }
    L.kth(kk, tk, ts);
  }
#pragma unroll
  for (int pp = 0; pp < KPL; pp++) {
    const int e = pp * 64 + lane;
    if (e < kk) {
      uint64_t id = ~0ull;
      double sc = __longlong_as_double(0x7FF8000000000000ll);
      if (L.s[pp] != ~0u) {
        double v = rank_value(L.k[pp]);
        // NaN keys come back as the one canonical quiet NaN (its sign is
        // not meaningful)
        if (v == v) sc = sqrt(v);
        id = logical_id(a.st, L.s[pp]);
      }
      a.ids[(size_t)q * a.ostride + e] = id;
      a.scores[(size_t)q * a.ostride + e] = sc;
    }
  }
}

hipError_t launch_merge(const MergeArgs& a, int kmax, hipStream_t s) {
  if (a.nq == 0) return hipSuccess;
  const dim3 grid((a.nq + kWavesPerBlock - 1) / kWavesPerBlock);
  if (kmax > 64) hipLaunchKernelGGL(k_merge<2>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_merge<1>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------- pair metrics
//
// FP64: one wavefront per pair, coalesced loads; lane l accumulates the
// elements i ≡ l (mod 64) in increasing order with fma, then six xor
// butterfly steps (offsets 32..1).  Every lane ends with the same sum.
//
// The slots are read from, and the metrics written to, pinned host memory by
// whole blocks, 4·ppw pairs at a time: no copies before or after, and the bus
// works beside the rows' gather.  Bound by that gather: a wavefront has four
// pairs' loads in flight, and the last four butterfly steps are DPP rotations
// (within a row of 16 whose lanes already agree modulo 2n, a rotation by n
// brings the value that xor n would) rather than LDS permutes.
// 1M pairs of 128 columns, cosine: the kernel 430 µs with a pair per wavefront,
// 450 so with the bus traffic in it; the call, with the host side, 1.77 → 0.98 ms.

template <int N>
__device__ __forceinline__ double row_ror_add(double x) {
  const int2 v = __builtin_bit_cast(int2, x);
  const int2 r = make_int2(__builtin_amdgcn_mov_dpp(v.x, 0x120 + N, 0xf, 0xf, true),
                           __builtin_amdgcn_mov_dpp(v.y, 0x120 + N, 0xf, 0xf, true));
  return x + __builtin_bit_cast(double, r);
}

__device__ __forceinline__ double wave_sum_f64(double x) {
  x = x + __shfl_xor(x, 32);
  x = x + __shfl_xor(x, 16);
  x = row_ror_add<8>(x);
  x = row_ror_add<4>(x);
  x = row_ror_add<2>(x);
  return row_ror_add<1>(x);
}

constexpr uint32_t kPairsPerWave = 16;

template <int METRIC>
__global__ __launch_bounds__(256) void k_pair_f64(const double* __restrict__ X, size_t ldx,
                                                  const uint32_t* __restrict__ slots, uint32_t np,
                                                  uint32_t D, uint32_t ppw,
                                                  double* __restrict__ out) {
  __shared__ uint32_t s_a[kWavesPerBlock * kPairsPerWave], s_b[kWavesPerBlock * kPairsPerWave];
  __shared__ double s_out[kWavesPerBlock * kPairsPerWave];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t p0 = blockIdx.x * kWavesPerBlock * ppw;
  const uint32_t m = min(kWavesPerBlock * ppw, np - p0);
  if (tid < m) s_a[tid] = slots[p0 + tid];
  if (tid >= 128 && tid - 128 < m) s_b[tid - 128] = slots[np + p0 + tid - 128];
  __syncthreads();
  for (uint32_t j0 = wave * ppw; j0 < min(m, (wave + 1) * ppw); j0 += 4) {
    const double *A[4], *B[4];
    double d[4], na[4], nb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t j = min(j0 + u, m - 1);
      A[u] = X + (size_t)__builtin_amdgcn_readfirstlane(s_a[j]) * ldx;
      B[u] = X + (size_t)__builtin_amdgcn_readfirstlane(s_b[j]) * ldx;
      d[u] = na[u] = nb[u] = 0.0;
    }
#pragma unroll 2
    for (uint32_t i = lane; i < D; i += 64) {
      double x[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        x[u] = A[u][i];
        y[u] = B[u][i];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (METRIC == kL2) {
          const double t = x[u] - y[u];
          d[u] = fma(t, t, d[u]);
        } else {
          d[u] = fma(x[u], y[u], d[u]);
          if (METRIC == kCos) {
            na[u] = fma(x[u], x[u], na[u]);
            nb[u] = fma(y[u], y[u], nb[u]);
          }
        }
      }
    }
    double rd = 0.0, ra = 0.0, rb = 0.0;  // lane u: pair j0 + u
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const double sd = wave_sum_f64(d[u]);
      rd = lane == (uint32_t)u ? sd : rd;
      if (METRIC == kCos) {
        const double sx = wave_sum_f64(na[u]), sy = wave_sum_f64(nb[u]);
        ra = lane == (uint32_t)u ? sx : ra;
        rb = lane == (uint32_t)u ? sy : rb;
      }
    }
    if (lane < 4 && j0 + lane < m) {
      double r = rd;
      if (METRIC == kL2) r = sqrt(rd);
      else if (METRIC == kCos) r = rd / (sqrt(ra) * sqrt(rb));
      s_out[j0 + lane] = r;
    }
  }
  __syncthreads();
  if (tid < m) out[p0 + tid] = s_out[tid];
}

hipError_t launch_pair_f64(const double* X, size_t ldx, const uint32_t* slots, uint32_t np,
                           uint32_t D, int metric, double* out, hipStream_t s) {
  if (np == 0) return hipSuccess;
  // (up to 16,384 pairs a turn of four per wavefront: 1,024 blocks)
  const uint32_t ppw = np <= 16384 ? 4 : kPairsPerWave, pb = kWavesPerBlock * ppw;
  dim3 grid((np + pb - 1) / pb), block(256);
  switch (metric) {
    case kL2: hipLaunchKernelGGL(k_pair_f64<kL2>, grid, block, 0, s, X, ldx, slots, np, D, ppw, out); break;
    case kCos: hipLaunchKernelGGL(k_pair_f64<kCos>, grid, block, 0, s, X, ldx, slots, np, D, ppw, out); break;
    case kDot: hipLaunchKernelGGL(k_pair_f64<kDot>, grid, block, 0, s, X, ldx, slots, np, D, ppw, out); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The reference's float metrics (vector_database.c:301-352), bit-identical to
// it: FP64 products added into float accumulators (acc = (float)((double)acc +
// a*b)); Euclidean squares the float-rounded difference in float; sqrt and the
// cosine division in double.  One wavefront: every product first, a column per
// lane, into LDS, then the serial chains (cosine: its three in lanes 0..2, one
// instruction stream).  Bound by those chains, some 24 cycles a column, with the
// elements read beforehand: a single thread that also read them and multiplied
// took 14.2 µs at 128 columns, 4.5 so.
constexpr uint32_t kRefCols = 256;

__device__ __forceinline__ float ref32_wave(const double* __restrict__ A,
                                            const double* __restrict__ B, uint32_t n, int metric,
                                            double (&P)[3][kRefCols]) {
  const uint32_t lane = threadIdx.x;
  const double* mine = P[lane < 3 && metric == kCos ? lane : 0];
  float acc = 0.0f;
  for (uint32_t c0 = 0; c0 < n; c0 += kRefCols) {
    const uint32_t m = min(kRefCols, n - c0);
    for (uint32_t i = lane; i < m; i += 64) {
      const double u = A[c0 + i], v = B[c0 + i];
      if (metric == kL2) {
        const float diff = (float)(u - v);
        P[0][i] = (double)(diff * diff);
      } else {
        P[0][i] = u * v;
        if (metric == kCos) {
          P[1][i] = u * u;
          P[2][i] = v * v;
        }
      }
    }
    __syncthreads();
    uint32_t i = 0;
    if (metric == kL2) {
      for (; i + 8 <= m; i += 8) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = (float)mine[i + j];
#pragma unroll
        for (int j = 0; j < 8; j++) acc = acc + t[j];
      }
      for (; i < m; i++) acc = acc + (float)mine[i];
    } else {
      for (; i + 8 <= m; i += 8) {
        double t[8];
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = mine[i + j];
#pragma unroll
        for (int j = 0; j < 8; j++) acc = (float)((double)acc + t[j]);
      }
      for (; i < m; i++) acc = (float)((double)acc + mine[i]);
    }
    __syncthreads();
  }
  if (metric == kCos) {
    const float na = __shfl(acc, 1), nb = __shfl(acc, 2);
    return (float)((double)acc / (sqrt((double)na) * sqrt((double)nb)));
  }
  return metric == kL2 ? (float)sqrt((double)acc) : acc;
}

// One pair of device rows.
__global__ __launch_bounds__(64) void k_pair_ref32(const double* __restrict__ A,
                                                   const double* __restrict__ B, uint32_t n,
                                                   int metric, float* __restrict__ out) {
  __shared__ double P[3][kRefCols];
  const float r = ref32_wave(A, B, n, metric, P);
  if (threadIdx.x == 0) out[0] = r;
}

// One pair from the kernel arguments (the drop-in per-call functions): the
// result, then seq once it is visible, into host memory the caller polls.
__global__ __launch_bounds__(64) void k_pair_ref32_args(const PairRef32Args a) {
  __shared__ double P[3][kRefCols];
  const float r = ref32_wave(a.ab, a.ab + a.n, a.n, a.metric, P);
  if (threadIdx.x != 0) return;
  a.out[0] = (uint64_t)__float_as_uint(r);
  __threadfence_system();
  __hip_atomic_store(a.out + 1, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

hipError_t launch_pair_ref32_args(const PairRef32Args& a, hipStream_t s) {
  if (a.n > kRef32ArgsMax) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pair_ref32_args, dim3(1), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_pair_ref32(const double* A, const double* B, uint32_t n, int metric, float* out,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_pair_ref32, dim3(1), dim3(64), 0, s, A, B, n, metric, out);
  return hipGetLastError();
}

}  // namespace svdb
