// svdb_lowp.hip — BF16 MFMA first pass, shortlist, FP64 rerank with
// certification (gfx950).  See svdb_lowp.h for the shadow layout and the
// error bound.  Built with -ffp-contract=off like the FP64 kernels.
#include "svdb_lowp.h"

#include <math.h>

#include "svdb_bins.h"
#include "svdb_prep.h"
#include "svdb_rank.h"

namespace svdb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------- helpers

__device__ __forceinline__ uint16_t bf16_of(double x) {
  float f = __double2float_rn(x);
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u) return (u & 0x007FFFFFu) ? (uint16_t)0x7FC0 : (uint16_t)(u >> 16);
  u += 0x7FFFu + ((u >> 16) & 1u);
  uint16_t b = (uint16_t)(u >> 16);
  if ((b & 0x7F80u) == 0) b &= 0x8000u;  // no bf16 subnormals: flush to zero
  return b;
}

__device__ __forceinline__ double bf16_val(uint16_t b) {
  return (double)__uint_as_float((uint32_t)b << 16);
}

__device__ __forceinline__ uint32_t rank_bits32(float v) {
  uint32_t u = __float_as_uint(v + 0.0f);
  if (v != v) u = 0x7FC00000u;
  return (u >> 31) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ uint32_t uni32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Wave-distributed sorted list (entry e in lane e%64, register e/64).
template <int KPL>
struct WL {
  uint64_t k[KPL];
  uint32_t s[KPL];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int p = 0; p < KPL; p++) {
      k[p] = ~0ull;
      s[p] = ~0u;
    }
  }
  __device__ __forceinline__ void at(int e, uint64_t& tk, uint32_t& ts) const {
    int p = e >> 6, ln = e & 63;
    uint64_t a = k[0];
    uint32_t b = s[0];
#pragma unroll
    for (int q = 1; q < KPL; q++)
      if (p == q) {
        a = k[q];
        b = s[q];
      }
    tk = uni64(__shfl(a, ln));
    ts = uni32(__shfl(b, ln));
  }
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

// ------------------------------------------------------------- shadow rows

__global__ void k_shadow_init(Shadow sh, uint32_t first, uint32_t n) {
  uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  uint32_t slot = first + r;
  sh.nx[slot] = INFINITY;
  sh.xn[slot] = -INFINITY;
  sh.inv[slot] = 0.0f;
  sh.pen[slot] = INFINITY;
}

hipError_t launch_shadow_init(const Shadow& sh, uint32_t first, uint32_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_shadow_init, dim3((n + 255) / 256), dim3(256), 0, s, sh, first, n);
  return hipGetLastError();
}

__device__ void kill_shadow_row(const Shadow& sh, uint32_t slot) {
  uint16_t* xb = sh.Xb + (size_t)slot * sh.dp;
  for (size_t i = 0; i < sh.dp; i++) xb[i] = 0;
  sh.nx[slot] = INFINITY;
  sh.xn[slot] = -INFINITY;
  sh.inv[slot] = 0.0f;
  sh.pen[slot] = INFINITY;
}

// One wavefront per row (after k_row_norms has written nx2 / xn), two columns
// a lane; bound by the row's read and write.  The error sum is in no fixed
// order: (1 + 2^-40) covers its rounding for d <= 2^11 as it does for a
// sequential one.  (A thread per row read a column at a time: one row of 128
// 25 µs, now 4; 500k rows 1.6 ms, now 0.25.)
__global__ __launch_bounds__(256) void k_quantize_rows(Shadow sh, const double* __restrict__ X,
                                                       size_t ldx, const double* __restrict__ nx2,
                                                       const double* __restrict__ xnorm,
                                                       const uint32_t* __restrict__ slots,
                                                       uint32_t first, uint32_t n, uint32_t d) {
  const int lane = threadIdx.x & 63;
  const uint32_t r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  const uint32_t slot = slots ? slots[r] : first + r;
  const double* x = X + (size_t)slot * ldx;
  uint32_t* xb = reinterpret_cast<uint32_t*>(sh.Xb + (size_t)slot * sh.dp);
  const double norm = xnorm[slot];
  double esq = 0.0, maxabs = 0.0;
  bool finite = true;
  for (uint32_t c = 2 * lane; c < sh.dp; c += 128) {
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const double v = c + j < d ? x[c + j] : 0.0;
      finite = finite && isfinite(v);
      maxabs = fmax(maxabs, fabs(v));
      const uint16_t b = bf16_of(v);
      const double e = bf16_val(b) - v;
      esq = fma(e, e, esq);
      word |= (uint32_t)b << (16 * j);
    }
    xb[c >> 1] = word;
  }
  for (int o = 32; o >= 1; o >>= 1) {
    maxabs = fmax(maxabs, __shfl_xor(maxabs, o));
    esq += __shfl_xor(esq, o);
  }
  finite = __all(finite);
  const double lim = 1152921504606846976.0;  // 2^60
  const bool degenerate = !finite || !(norm >= 1.0 / lim) || !(norm <= lim) || !(maxabs <= lim);
  if (degenerate)
    for (uint32_t c = 2 * lane; c < sh.dp; c += 128) xb[c >> 1] = 0;
  if (lane != 0) return;
  if (degenerate) {
    sh.nx[slot] = INFINITY;
    sh.xn[slot] = -INFINITY;
    sh.inv[slot] = 0.0f;
    sh.pen[slot] = INFINITY;
    uint32_t cnt = atomicAdd(sh.degen_count, 0u);
    bool present = false;
    for (uint32_t j = 0; j < cnt && j < (uint32_t)kDegenCap; j++) present |= sh.degen[j] == slot;
    if (!present) {
      uint32_t idx = atomicAdd(sh.degen_count, 1u);
      if (idx < (uint32_t)kDegenCap) sh.degen[idx] = slot;
    }
    return;
  }
  sh.nx[slot] = __double2float_rd(nx2[slot]);
  sh.xn[slot] = __double2float_ru(norm);
  sh.inv[slot] = __double2float_rn(1.0 / norm);
  sh.pen[slot] = 0.0f;
  const double up = 1.0 + 0x1p-40;
  const double ratio = (sqrt(esq) * up) / norm * up;
  // (rho only grows: a row below the value read need not be counted in)
  const uint32_t rb = __float_as_uint(__double2float_ru(ratio));
  if (rb > __hip_atomic_load(sh.rho_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(sh.rho_bits, rb);
}

hipError_t launch_quantize_rows(const Shadow& sh, const double* X, size_t ldx, const double* nx2,
                                const double* xn, const uint32_t* slots, uint32_t first,
                                uint32_t n, uint32_t d, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_quantize_rows, dim3((n + 3) / 4), dim3(256), 0, s, sh, X, ldx, nx2, xn,
                     slots, first, n, d);
  return hipGetLastError();
}

__global__ void k_kill_rows(Shadow sh, const uint32_t* __restrict__ slots, uint32_t n) {
  uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) kill_shadow_row(sh, slots[r]);
}

hipError_t launch_kill_rows(const Shadow& sh, const uint32_t* slots, uint32_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_kill_rows, dim3((n + 63) / 64), dim3(64), 0, s, sh, slots, n);
  return hipGetLastError();
}

// ------------------------------------------------------------- query prep
//
// Per query: FP64 ‖q‖ (the canonical chain), bf16 q̂ scaled by -2 (Euclidean)
// or -1 (dot, cosine) — exact power-of-two scalings — and the per-query
// bound constants.  The error sums are in no fixed order; (1 + 2^-40) covers
// their rounding in any order.

__global__ __launch_bounds__(64 * kPrepWaves) void k_query_prep(QueryPrepArgs a) {
  extern __shared__ __attribute__((aligned(16))) double prep_rows[];
  const int lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x < (uint32_t)a.nr) a.fail_count[threadIdx.x] = 0u;
  const uint32_t i = blockIdx.x * kPrepWaves + (threadIdx.x >> 6);
  if (i >= a.nslots) return;
  int metric;
  const PrepSlot ps = prep_slot(a, i, metric);
  const uint32_t d = a.d, cols = (d + 15) & ~15u;
  uint32_t* qb = reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(a.Qb) + (size_t)i * a.dp);
  QParams* qp = a.qp;
  QParams p{};
  p.metric = metric;
  if (ps.range < 0) {
    for (uint32_t c = 2 * lane; c < a.dp; c += 128) qb[c >> 1] = 0;
    p.flags = 1;
    if (lane == 0) qp[i] = p;
    return;
  }
  double* row = prep_rows + (threadIdx.x >> 6) * cols;
  double maxabs;
  bool finite;
  const double nq2 = prep_stage(a.Q + (size_t)ps.row * a.ldq,
                                a.Qd ? a.Qd + (size_t)ps.row * a.ldq : nullptr, d, cols, row,
                                lane, maxabs, finite);
  const double sc = metric == kL2 ? -2.0 : -1.0;
  double esq = 0.0, hsq = 0.0;
  for (uint32_t c = 2 * lane; c < a.dp; c += 128) {
    uint32_t word = 0;
    if (c < cols) {
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const double v = row[c + j];
        const double h = bf16_val(bf16_of(v));
        const double e = h - v;
        esq = fma(e, e, esq);
        hsq = fma(h, h, hsq);
        word |= (uint32_t)bf16_of(h * sc) << (16 * j);
      }
    }
    if (c + 1 >= d) word &= c < d ? 0xFFFFu : 0u;  // (0 · sc is -0)
    qb[c >> 1] = word;
  }
  esq = wave_sum(esq);
  hsq = wave_sum(hsq);
  const double rho = (double)__uint_as_float(*a.rho_bits);
  const double qn = sqrt(nq2);
  const double lim = 1152921504606846976.0;  // 2^60
  const double up = 1.0 + 0x1p-40;
  const double gam = (double)(d + 32) * 0x1p-24;
  const double qh = sqrt(hsq) * up, eq = sqrt(esq) * up;
  const double qh1 = qh * (1.0 + rho) * (1.0 + gam) * up;  // >= |s| / ‖x‖
  const double delta = (double)d * 0x1p-124;
  const double c = (gam * qh * (1.0 + rho) + eq + rho * qh * (1.0 + gam) +
                    (double)(d + 8) * 0x1p-52 * qn) * up;
  p.qn = qn;
  p.nq2 = nq2;
  p.flags = (!finite || !(qn >= 1.0 / lim) || !(qn <= lim) || !(maxabs <= lim)) ? 1 : 0;
  if (metric == kL2) {
    const double a = 1.0 - c / qn - 0x1p-24 * (1.0 + qh1 / qn) - 0x1p-30;
    p.P = __double2float_rd(a);
    p.scale = 1.0;
    p.off = nq2 - qn * (c + 0x1p-24 * qh1) - 2.0 * delta;
    if (!(a > 0.0)) p.flags = 1;
  } else if (metric == kDot) {
    const double cp = (c + 0x1p-23 * (qh1 + c) * 1.01) * up;
    p.P = __double2float_rd(-cp);
    p.scale = 1.0;
    p.off = -delta;
  } else {
    p.P = 0.0f;
    p.scale = 1.0 / qn;
    p.off = -(c + 0x1p-23 * qh1 * 1.01 + delta * lim) / qn - (double)(d + 16) * 0x1p-52;
  }
  if (lane == 0) qp[i] = p;
}

hipError_t launch_query_prep(const QueryPrepArgs& a, hipStream_t s) {
  if (a.nslots == 0) return hipSuccess;
  const uint32_t cols = (a.d + 15) & ~15u;
  hipLaunchKernelGGL(k_query_prep, dim3((a.nslots + kPrepWaves - 1) / kPrepWaves),
                     dim3(64 * kPrepWaves), kPrepWaves * cols * sizeof(double), s, a);
  return hipGetLastError();
}

// ------------------------------------------------------------- shortlist
//
// One block per query: the L smallest ordering keys of the query's NL candidate
// lists (svdb_cand.h), unordered (the rerank orders them), and the bound
// beta = min(every list's bound, L-th key): no row outside the shortlist has
// a smaller ordering key.  The headers are read first, all together; then four
// threads take a list, four entries each, and each thread has four such loads
// in flight, so the time goes with neither the lists' number nor their length
// but with both.  The entries are packed into LDS as order-preserving bits and the L-th smallest is found by
// counting them into 256 bins of the range that still holds it, until a bin is
// one key wide (2 or 3 counts for keys of one magnitude).  More entries than
// the LDS holds (the widening retries over full lists) are read again from the
// lists instead. 
// Against a wavefront per query with a sorted list (L <= 64) and radix passes
// over every list slot (wider): 1 query over 1M rows 108 → 9 µs, 16,384 over
// 2M rows 310 → 66, 1,400 queries at L = 256 over 1M rows 137 → 95, 4,096 FP8
// queries at L = 128 270 → 87, at 1,024 310 → 87.
// LDS capacity: the lists of a 64-wide shortlist hold some 400 entries (FP8
// 1,600), wider ones' up to about 3,500; 4,096 for all had 4 blocks per CU
// where 2,048 has 8 (16,384 queries, L = 64: 106 against 66 µs; 4,096 FP8
// queries, L = 128: 87 against 524, most of them read again).
constexpr uint32_t kSelLists = 2048;

template <int T, uint32_t CAP>
struct SelShared {
  uint32_t key[CAP], slot[CAP];
  uint8_t cnt[kSelLists];
  uint32_t hist[256];
  uint32_t n, lo, hi, rank, lt, eq;
  uint32_t wlo[T / 64], whi[T / 64];
  float wmin[T / 64];
};

__device__ __forceinline__ float rank_float32(uint32_t u) {
  return __uint_as_float((u >> 31) ? (u & 0x7FFFFFFFu) : ~u);
}

// This lane's first place of `m` in a block-wide counter: the wavefront's
// lanes are counted together and reserved with one atomic.
__device__ __forceinline__ uint32_t wave_reserve(uint32_t* counter, uint32_t m, int lane) {
  uint32_t inc = m;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t v = __shfl_up(inc, off);
    if (lane >= off) inc += v;
  }
  uint32_t base = 0;
  if (lane == 63 && inc) base = atomicAdd(counter, inc);
  return __shfl(base, 63) + inc - m;
}

template <int T, uint32_t CAP>
__device__ __forceinline__ void shortlist_body(const ShortlistArgs& a, uint32_t i,
                                               SelShared<T, CAP>& sm) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t q = a.qidx ? a.qidx[i] : i;  // candidate lists of query q -> output row i
  const bool sorted = !a.hdr;
  const uint2* __restrict__ hdr = a.hdr + (sorted ? 0 : (size_t)q * a.NL);
  const uint32_t LC = sorted ? kLowpLP : kLowpLC;
  const uint2* __restrict__ ent = a.ent + (size_t)q * a.NL * LC;
  if (tid == 0) {
    sm.n = 0;
    sm.lt = 0;
    sm.eq = 0;
  }
  __syncthreads();
  // every entry below the LDS capacity, their number, range and the bounds
  float bmin = INFINITY;
  uint32_t lo = ~0u, hi = 0u;
  for (uint32_t l = tid; l < a.NL; l += T) {
    if (sorted) {
      uint32_t m = 0;
#pragma unroll
      for (int e = 0; e < kLowpLP; e += 2) {
        const uint4 v = *reinterpret_cast<const uint4*>(ent + (size_t)l * kLowpLP + e);
        m += (v.y != ~0u) + (v.w != ~0u);
        if (e == kLowpLP - 2) bmin = fminf(bmin, __uint_as_float(v.z));
      }
      sm.cnt[l] = (uint8_t)m;
      continue;
    }
    const uint2 h = hdr[l];
    sm.cnt[l] = (uint8_t)h.x;
    bmin = fminf(bmin, __uint_as_float(h.y));
  }
  __syncthreads();
  constexpr int U = 4;
  const int qs = sorted ? 1 : 2;  // log2 of a list's groups of four entries
  static_assert(kLowpLP == 8 && kLowpLC == 16, "qs");
  const uint32_t quads = a.NL << qs;
  for (uint32_t t0 = 0; t0 < quads; t0 += U * T) {
    uint32_t m[U], sum = 0;
    uint4 v[U][2];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t t = t0 + u * T + tid, e0 = (t & ((1u << qs) - 1)) * 4;
      const uint32_t c = t < quads ? sm.cnt[t >> qs] : 0u;
      m[u] = c > e0 ? min(4u, c - e0) : 0u;
      sum += m[u];
      if (m[u]) {
        const uint4* src = reinterpret_cast<const uint4*>(ent + (size_t)t * 4);
        v[u][0] = src[0];
        v[u][1] = src[1];
      }
    }
    uint32_t pos = wave_reserve(&sm.n, sum, lane);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t ks[4] = {v[u][0].x, v[u][0].z, v[u][1].x, v[u][1].z};
      const uint32_t ss[4] = {v[u][0].y, v[u][0].w, v[u][1].y, v[u][1].w};
#pragma unroll
      for (int j = 0; j < 4; j++)
        if ((uint32_t)j < m[u]) {
          const uint32_t kb = rank_bits32(__uint_as_float(ks[j]));
          lo = min(lo, kb);
          hi = max(hi, kb);
          if (pos < CAP) {
            sm.key[pos] = kb;
            sm.slot[pos] = ss[j];
          }
          pos++;
        }
    }
  }
  for (int off = 32; off >= 1; off >>= 1) {
    bmin = fminf(bmin, __shfl_xor(bmin, off));
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, off));
    hi = max(hi, (uint32_t)__shfl_xor((int)hi, off));
  }
  if (lane == 0) {
    sm.wmin[wave] = bmin;
    sm.wlo[wave] = lo;
    sm.whi[wave] = hi;
  }
  __syncthreads();
  const uint32_t n = sm.n;
  if (tid == 0) {
    for (int w = 1; w < T / 64; w++) {
      lo = min(lo, sm.wlo[w]);
      hi = max(hi, sm.whi[w]);
      bmin = fminf(bmin, sm.wmin[w]);
    }
    sm.lo = lo;
    sm.hi = hi;
    sm.rank = a.L;
  }
  // f(key bits, slot) for every entry
  auto each = [&](auto&& f) __attribute__((always_inline)) {
    if (n <= CAP) {
      for (uint32_t c = tid; c < n; c += T) f(sm.key[c], sm.slot[c]);
      return;
    }
    for (uint32_t l = tid; l < a.NL; l += T) {
      const uint32_t m = sm.cnt[l];
      for (uint32_t e = 0; e < m; e++) {
        const uint2 v = ent[(size_t)l * LC + e];
        f(rank_bits32(__uint_as_float(v.x)), v.y);
      }
    }
  };
  __syncthreads();
  if (n > a.L) {
    for (;;) {
      // the L-th smallest key is the sm.rank-th of those in [l, h]
      const uint32_t l = sm.lo, h = sm.hi;
      if (l == h) break;
      const int shift = bin_shift(h - l);
      for (int b = tid; b < 256; b += T) sm.hist[b] = 0;
      __syncthreads();
      each([&](uint32_t k, uint32_t) {
        if (k >= l && k <= h) atomicAdd(&sm.hist[(k - l) >> shift], 1u);
      });
      __syncthreads();
      if (wave == 0) {
        // lane b holds bins 4b..4b+3; an inclusive scan over lanes finds
        // the bin where the running count reaches the target rank
        const uint32_t hs[4] = {sm.hist[4 * lane], sm.hist[4 * lane + 1], sm.hist[4 * lane + 2],
                                sm.hist[4 * lane + 3]};
        const uint32_t sum = hs[0] + hs[1] + hs[2] + hs[3];
        uint32_t inc = sum;
        for (int off = 1; off < 64; off <<= 1) {
          const uint32_t v = __shfl_up(inc, off);
          if (lane >= off) inc += v;
        }
        const uint32_t exc = inc - sum, rank = sm.rank;
        if (exc < rank && rank <= inc) {
          uint32_t cum = exc, bin = 4 * lane;
#pragma unroll
          for (int b = 0; b < 3; b++)
            if (bin == 4u * lane + b && cum + hs[b] < rank) {
              cum += hs[b];
              bin++;
            }
          sm.rank = rank - cum;
          sm.lo = l + (bin << shift);
          sm.hi = bin_last(l, h, bin, shift);
        }
      }
      __syncthreads();
    }
  }
  // entries below the L-th key: all of them; equal to it: the first that
  // come, as many as are needed
  const bool all = n <= a.L;
  const uint32_t kstar = all ? ~0u : sm.lo;
  const uint32_t need_eq = all ? 0u : sm.rank;
  const uint32_t n_lt = all ? 0u : a.L - need_eq;
  each([&](uint32_t k, uint32_t slot) {
    uint32_t pos = ~0u;
    if (all || k < kstar) {
      pos = atomicAdd(&sm.lt, 1u);
    } else if (k == kstar) {
      const uint32_t e = atomicAdd(&sm.eq, 1u);
      if (e < need_eq) pos = n_lt + e;
    }
    if (pos != ~0u) {
      a.short_slot[(size_t)i * a.L + pos] = slot;
      a.short_key[(size_t)i * a.L + pos] = rank_float32(k);
    }
  });
  // unused tail (fewer than L entries)
  for (uint32_t e = n + tid; e < a.L; e += T) {
    a.short_slot[(size_t)i * a.L + e] = ~0u;
    a.short_key[(size_t)i * a.L + e] = INFINITY;
  }
  if (tid == 0) a.beta[i] = n >= a.L ? fminf(bmin, rank_float32(all ? hi : kstar)) : bmin;
}

// Several ranges' shortlists (or reranks) in one launch: range r takes
// blocks first[r] .. first[r+1]-1 (a launch per range costs its latency
// once per range, and small ranges leave most of the GPU idle).
template <typename A>
struct RangeBatch {
  A r[kMaxLaunchRanges];
  int metric[kMaxLaunchRanges];
  uint32_t first[kMaxLaunchRanges + 1];
  int n;
};

template <typename A>
__device__ __forceinline__ int range_of(const RangeBatch<A>& b, uint32_t blk) {
  int i = 0;
  while (i + 1 < b.n && blk >= b.first[i + 1]) i++;
  return i;
}

template <int T, uint32_t CAP>
__global__ __launch_bounds__(T) void k_shortlist(RangeBatch<ShortlistArgs> b) {
  __shared__ SelShared<T, CAP> sm;
  const int i = range_of(b, blockIdx.x);
  shortlist_body<T, CAP>(b.r[i], blockIdx.x - b.first[i], sm);
}

// Up to 256 queries (one block per CU or fewer) a block takes 1,024 threads, so
// that the headers of the many lists such batches have are read in a few
// rounds; beyond, 256 threads, and 8 queries a CU at once.
hipError_t launch_shortlist_ranges(const ShortlistArgs* a, int n, hipStream_t s) {
  for (int r0 = 0; r0 < n; r0 += kMaxLaunchRanges) {
    RangeBatch<ShortlistArgs> b{};
    uint32_t blocks = 0;
    bool narrow = true;
    b.n = 0;
    for (int r = r0; r < n && b.n < kMaxLaunchRanges; r++) {
      if (a[r].L == 0 || a[r].L > (uint32_t)kMaxShort || a[r].NL > kSelLists)
        return hipErrorInvalidValue;
      narrow &= a[r].L <= 64;
      b.r[b.n] = a[r];
      b.first[b.n] = blocks;
      blocks += a[r].nq;
      b.n++;
    }
    b.first[b.n] = blocks;
    if (blocks == 0) continue;
    if (blocks <= 256)
      hipLaunchKernelGGL((k_shortlist<1024, 4096>), dim3(blocks), dim3(1024), 0, s, b);
    else if (narrow)
      hipLaunchKernelGGL((k_shortlist<256, 2048>), dim3(blocks), dim3(256), 0, s, b);
    else
      hipLaunchKernelGGL((k_shortlist<256, 4096>), dim3(blocks), dim3(256), 0, s, b);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_shortlist(const ShortlistArgs& a, hipStream_t s) {
  return launch_shortlist_ranges(&a, 1, s);
}

// ------------------------------------------------ L-th smallest of n keys
//
// One wavefront per query; the keys (n <= 64 * kKthPerLane) sit in registers
// as order-preserving uint32.  A bisection between their smallest and largest
// counts, with ballots, how many lie at or below the midpoint, and ends as soon
// as L do: the result is the largest of those.  (Some ten steps for 1,024 keys,
// each a chain of 16 compares and bit counts; the 32 steps to a single value
// took 9 to 13 µs a launch, 7 to 12 so.)

constexpr int kKthPerLane = 16;

__global__ __launch_bounds__(256) void k_kth_key(const KthArgs a) {
  const int lane = threadIdx.x & 63;
  const uint32_t q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= a.nq) return;
  uint32_t L = a.rank[0];
  for (int i = 1; i < a.nr; i++) L = q >= a.first[i] ? a.rank[i] : L;
  const uint32_t n = a.n;
  const float* __restrict__ key = a.key + (size_t)q * n;
  uint32_t u[kKthPerLane];
  uint32_t lo = ~0u, hi = 0;
#pragma unroll
  for (int i = 0; i < kKthPerLane; i++) {
    const uint32_t c = i * 64 + lane;
    u[i] = c < n ? rank_bits32(key[c]) : ~0u;
    lo = min(lo, u[i]);
    hi = max(hi, u[i]);
  }
  for (int o = 32; o >= 1; o >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, o));
    hi = max(hi, (uint32_t)__shfl_xor((int)hi, o));
  }
  // the L-th smallest lies in lo .. hi
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    uint32_t cnt = 0;
#pragma unroll
    for (int i = 0; i < kKthPerLane; i++) cnt += __popcll(__ballot(u[i] <= mid));
    if (cnt >= L) hi = mid;
    else lo = mid + 1;
    if (cnt == L) break;
  }
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < kKthPerLane; i++) r = u[i] <= hi ? max(r, u[i]) : r;
  for (int o = 32; o >= 1; o >>= 1) r = max(r, (uint32_t)__shfl_xor((int)r, o));
  if (lane == 0)
    a.thr[q] = (r >= rank_bits32(INFINITY) || n < L)
                   ? INFINITY
                   : __uint_as_float((r >> 31) ? (r & 0x7FFFFFFFu) : ~r);
}

hipError_t launch_kth_key(const KthArgs& a, hipStream_t s) {
  if (a.nq == 0) return hipSuccess;
  if (a.n > 64u * kKthPerLane || a.nr < 1 || a.nr > kKthRanges) return hipErrorInvalidValue;
  for (int i = 0; i < a.nr; i++)
    if (a.rank[i] == 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_kth_key, dim3((a.nq + 3) / 4), dim3(256), 0, s, a);
  return hipGetLastError();
}

// ------------------------------------------------------------- FP64 rerank
//
// The candidates' canonical FP64 rank keys (the sequential fma chains), the k
// best by (key, slot), and the certificate: the k-th key is below the bound
// beta*scale + off (minus the FP64 rounding slack of that expression and, for
// Euclidean, of the keys themselves).  Certified queries get their ids and
// scores written; the others are listed for the next stage.  The first stage
// (shortlists up to 256, k_rerank) takes a block per query, the widening
// retries (1,024 and 4,096, k_rerank1) a wavefront.

// FP64 lower bound on the ordering value of a row whose first-pass key is at
// least `bo` (the rounding slack of the key's conversion included).
__device__ __forceinline__ double lowp_lower(float bo, const QParams& qp, int metric, uint32_t d) {
  if (bo == INFINITY) return INFINITY;
  const double bs = (double)bo * qp.scale;
  double bR = bs + qp.off;
  bR -= 0x1p-40 * (fabs(bs) + fabs(qp.off));
  if (metric == kL2 && bR > 0.0) bR *= 1.0 - (double)(d + 4) * 0x1p-52;
  return bR;
}

// |first-pass estimate - score| / |score| of a result whose first-pass key
// is O (finite), for the error report; 0 where it has no value.
__device__ __forceinline__ double lowp_rel_err(float O, double sc, uint32_t slot,
                                               const QParams& qp, int metric,
                                               const RerankArgs& a) {
  if (!(sc == sc) || sc == 0.0) return 0.0;
  double est;
  if (metric == kL2) {
    // (FP8 keys are the BF16-form key / sq; scale = sq there, 1 for BF16)
    const double xn = a.st.xn[slot];
    const double sp = ((double)O - (double)qp.P * (double)a.w0[slot]) * qp.scale;
    est = sqrt(fmax(qp.nq2 + xn * xn + sp, 0.0));
  } else if (metric == kDot) {
    est = -((double)O - (double)qp.P * (double)a.w0[slot]) * qp.scale;
  } else {
    est = -(double)O / qp.qn;
  }
  return fabs(est - sc) / fabs(sc);
}

// Candidate rows reach the lanes through LDS: per round of 64 candidates
// the wave copies kRC columns of all 64 rows at a time (lane l fetches
// column l%16 of candidates 4u + l/16, u = 0..15: each load instruction
// reads 4 contiguous 128-byte row pieces), then each lane continues its own
// candidate's sequential fma chain over those columns.  The FP64 keys are
// the canonical chains, in index order, as before.
constexpr int kRC = 16;

template <int METRIC>
__device__ __forceinline__ void rerank_body(const RerankArgs& a, uint32_t blk, double* stg,
                                            uint32_t* queue) {
  const int lane = threadIdx.x & 63;
  const uint32_t i = blk * 4 + (threadIdx.x >> 6);
  if (i >= a.nq) return;
  // shortlist row i belongs to query q (its parameters, FP64 row, outputs)
  const uint32_t q = a.qidx ? a.qidx[i] : i;
  const QParams qp = a.qp[q];
  const double* __restrict__ qv = a.Q + (size_t)q * a.ldq;
  const uint32_t ndeg = min(*a.degen_count, (uint32_t)kDegenCap);
  const int kk = (int)a.k;

  auto lower = [&](float bo) __attribute__((always_inline)) -> double {
    return lowp_lower(bo, qp, METRIC, a.d);
  };
  // a flagged query's keys carry no bound: no pruning
  const bool prune = !qp.flags;

  WL<2> L;
  L.init();
  uint64_t tk = ~0ull;
  uint32_t ts = ~0u;
  // the earlier stage's list, and the key below which its shortlists
  // already covered every candidate
  const bool carry = a.carry && a.lk;
  float kprev = -INFINITY;
  if (carry) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
      const int e = p * 64 + lane;
      if (e < kk) {
        L.k[p] = a.lk[(size_t)q * kk + e];
        L.s[p] = a.ls[(size_t)q * kk + e];
      }
    }
    L.at(kk - 1, tk, ts);
    kprev = a.kmax[q];
  }
  float kmax_lane = -INFINITY;
  const uint32_t ncand = a.L + ndeg;

  // Scores up to 64 candidates, lane l's `slot` when `valid`, and enters
  // them into the list.
  auto score = [&](uint32_t slot, bool valid) __attribute__((always_inline)) {
    // rows this lane fetches: candidates 4u + lane/16
    const double* src[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int cand = u * 4 + (lane >> 4);
      const uint32_t sl = __shfl(slot, cand);
      const int ok = __shfl(valid ? 1 : 0, cand);
      src[u] = ok ? a.st.X + (size_t)sl * a.st.ldx : nullptr;
    }
    double acc = 0.0;
    const double* my = stg + lane * (kRC + 1);
    // The next chunk's loads go out once this chunk's values sit in LDS
    // (into the same registers), so they are in flight during its FMAs.
    double vals[16];
    auto fetch = [&](uint32_t c0) __attribute__((always_inline)) {
      const uint32_t e = c0 + (lane & 15);
#pragma unroll
      for (int u = 0; u < 16; u++) vals[u] = (src[u] && e < a.d) ? src[u][e] : 0.0;
    };
    fetch(0);
    for (uint32_t c0 = 0; c0 < a.d; c0 += kRC) {
#pragma unroll
      for (int u = 0; u < 16; u++) stg[(u * 4 + (lane >> 4)) * (kRC + 1) + (lane & 15)] = vals[u];
      __builtin_amdgcn_wave_barrier();
      if (c0 + kRC < a.d) fetch(c0 + kRC);
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t ne = min((uint32_t)kRC, a.d - c0);
#pragma unroll
      for (int t = 0; t < kRC; t++) {
        if ((uint32_t)t < ne) {
          const double x = my[t];
          if (METRIC == kL2) {
            const double tt = x - qv[c0 + t];
            acc = fma(tt, tt, acc);
          } else {
            acc = fma(qv[c0 + t], x, acc);
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    uint64_t K = ~0ull;
    if (valid) {
      double v = acc;
      if (METRIC == kDot) v = -acc;
      else if (METRIC == kCos) v = -(acc / (qp.qn * a.st.xn[slot]));
      K = rank_bits(v);
    }
    uint64_t m = __ballot(valid && lex_lt(K, slot, tk, ts));
    while (m) {
      int src = __ffsll((long long)m) - 1;
      m &= m - 1;
      const uint32_t S = uni32(__shfl(slot, src));
      // a row the carried list already holds (keyed at kprev, or a
      // degenerate row) must not enter twice
      if (carry && __ballot(L.s[0] == S || L.s[1] == S) != 0) continue;
      L.insert(uni64(__shfl(K, src)), S, kk, lane);
      // lanes that no longer beat the (moved) k-th entry drop out
      L.at(kk - 1, tk, ts);
      m &= __ballot(lex_lt(K, slot, tk, ts));
    }
    L.at(kk - 1, tk, ts);
  };

  // Candidates that still need their FP64 row are packed, in order, into
  // this wavefront's queue and scored 64 at a time, so a group fetches 64
  // rows however many of the shortlist's candidates were skipped.
  uint32_t nqd = 0;  // queued (wave-uniform; at most 127)
  uint32_t j0 = 0;
  for (;;) {
    while (nqd < 64 && j0 < ncand) {
      const uint32_t j = j0 + lane;
      uint32_t slot = ~0u;
      if (j < a.L) slot = a.short_slot[(size_t)i * a.L + j];
      else if (j < ncand) slot = a.degen[j - a.L];
      bool valid = slot != ~0u && slot < a.st.nrows &&
                   ((a.st.alive[slot >> 6] >> (slot & 63)) & 1ull);
      const float key = j < a.L ? a.short_key[(size_t)i * a.L + j] : -INFINITY;
      kmax_lane = fmaxf(kmax_lane, key);
      // scored in an earlier stage (its best k are in the carried list)
      if (carry && j < a.L && key < kprev) valid = false;
      // Prune threshold: the list's k-th value once full (+inf: fetch every
      // candidate).  A row whose lower bound exceeds it cannot be in the
      // top k.  (A NaN bound compares false and keeps its row.)
      const double thr = (prune && ts != ~0u) ? rank_value(tk) : INFINITY;
      if (valid && j < a.L && thr < INFINITY && lower(key) > thr) valid = false;
      // a degenerate row that is also shortlisted must not enter twice
      if (valid && j >= a.L) {
        for (uint32_t t = 0; t < a.L; t++)
          if (a.short_slot[(size_t)i * a.L + t] == slot) valid = false;
      }
      const uint64_t vm = __ballot(valid);
      if (valid) queue[nqd + __popcll(vm & ((1ull << lane) - 1ull))] = slot;
      nqd += __popcll(vm);
      j0 += 64;
    }
    __builtin_amdgcn_wave_barrier();
    if (nqd == 0) break;
    const uint32_t n = min(nqd, 64u);
    const uint32_t slot = (uint32_t)lane < n ? queue[lane] : ~0u;
    const uint32_t rest = (uint32_t)lane + 64 < nqd ? queue[lane + 64] : 0u;
    __builtin_amdgcn_wave_barrier();
    if ((uint32_t)lane + 64 < nqd) queue[lane] = rest;
    nqd -= n;
    __builtin_amdgcn_wave_barrier();
    score(slot, (uint32_t)lane < n);
  }

  // certification
  // more degenerate rows than the list holds: nothing can be certified
  bool cert = false;
  const double tau = ts == ~0u ? INFINITY : rank_value(tk);
  if (!qp.flags && *a.degen_count <= (uint32_t)kDegenCap) cert = tau < lower(a.beta[i]);
  if (!cert) {
    if (a.lk) {
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const int e = p * 64 + lane;
        if (e < kk) {
          a.lk[(size_t)q * kk + e] = L.k[p];
          a.ls[(size_t)q * kk + e] = L.s[p];
        }
      }
      for (int off = 32; off >= 1; off >>= 1) kmax_lane = fmaxf(kmax_lane, __shfl_xor(kmax_lane, off));
      if (lane == 0) a.kmax[q] = fmaxf(kmax_lane, kprev);
    }
    if (lane == 0) {
      uint32_t idx = atomicAdd(a.fail_count, 1u);
      a.fail_list[idx] = q;
    }
    return;
  }
  // First-pass keys of this lane's results, for the error report: the
  // shortlist passes through the wavefront's LDS area in chunks of kOC
  // (slot, key) pairs and every lane matches its two result slots there.
  constexpr uint32_t kOC = 1024;  // 8 KB of the 64 * (kRC + 1) doubles
  static_assert(kOC * 8 <= 64 * (kRC + 1) * sizeof(double), "chunk exceeds the stage");
  float O2[2] = {INFINITY, INFINITY};
  {
    uint32_t* oslot = reinterpret_cast<uint32_t*>(stg);
    float* okey = reinterpret_cast<float*>(oslot + kOC);
    for (uint32_t t0 = 0; t0 < a.L; t0 += kOC) {
      const uint32_t nt = min(kOC, a.L - t0);
      for (uint32_t t = lane; t < nt; t += 64) {
        oslot[t] = a.short_slot[(size_t)i * a.L + t0 + t];
        okey[t] = a.short_key[(size_t)i * a.L + t0 + t];
      }
      __builtin_amdgcn_wave_barrier();
      for (uint32_t t = 0; t < nt; t++) {
        const uint32_t sl = oslot[t];
        if (sl == L.s[0]) O2[0] = okey[t];
        if (sl == L.s[1]) O2[1] = okey[t];
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  double err = 0.0;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const int e = p * 64 + lane;
    if (e < kk) {
      uint64_t id = ~0ull;
      double sc = __longlong_as_double(0x7FF8000000000000ll);
      const uint32_t slot = L.s[p];
      if (slot != ~0u) {
        const double v = rank_value(L.k[p]);
        if (v == v) sc = METRIC == kL2 ? sqrt(v) : (v == 0.0 ? 0.0 : -v);
        id = a.st.has_deletes
                 ? (uint64_t)a.st.rank_base[slot >> 6] +
                       (uint64_t)__popcll(a.st.alive[slot >> 6] & ((1ull << (slot & 63)) - 1ull))
                 : slot;
        if (O2[p] != INFINITY) err = fmax(err, lowp_rel_err(O2[p], sc, slot, qp, METRIC, a));
      }
      a.ids[(size_t)q * a.ostride + e] = id;
      a.scores[(size_t)q * a.ostride + e] = sc;
    }
  }
  for (int off = 32; off >= 1; off >>= 1) err = fmax(err, __shfl_xor(err, off));
  if (lane == 0) a.max_rel_err[q] = err;
}

// The widening retries: one wavefront per shortlist row, one metric, held to
// 128 VGPRs for 4 wavefronts per SIMD (the row gather is latency-bound; a few
// spilled dwords cost less than the lost occupancy: measured 12-20 % faster
// than the same code at 3 per SIMD)
template <int METRIC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_rerank1(
    RerankArgs a) {
  __shared__ double stage[4][64 * (kRC + 1)];
  __shared__ uint32_t queue[4][128];
  rerank_body<METRIC>(a, blockIdx.x, stage[threadIdx.x >> 6], queue[threadIdx.x >> 6]);
}

hipError_t launch_rerank_wide(const RerankArgs& a, int metric, hipStream_t s) {
  if (a.nq == 0) return hipSuccess;
  if (!a.carry || !a.lk) return hipErrorInvalidValue;
  const dim3 grid((a.nq + 3) / 4);
  switch (metric) {
    case kL2: hipLaunchKernelGGL(k_rerank1<kL2>, grid, dim3(256), 0, s, a); break;
    case kCos: hipLaunchKernelGGL(k_rerank1<kCos>, grid, dim3(256), 0, s, a); break;
    case kDot: hipLaunchKernelGGL(k_rerank1<kDot>, grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// First-stage rerank (L <= kRrMaxL): one block of 4 wavefronts per query.
// The candidates — shortlist and degenerate rows — are ordered by first-pass
// key; the first `m1` are scored, their k-th FP64 key bounds which of the
// others can still enter the top k (a prefix of the order, since the lower
// bound grows with the key), those are scored too, and every scored row takes
// its place by counting the keys before it.  All the orderings are counts over
// LDS, which costs no more per query at k = 100 than at k = 10, where sorted
// insertions, one at a time through a wavefront, had taken most of the time.
//
// A wavefront scores 16 rows at a time, 64 columns per step: each load
// instruction reads 512 contiguous bytes of one row, and the next step's
// loads are in flight during this step's chains (lane l: row l%16; LDS rows
// are 65 doubles apart, so the 16 chains read distinct banks).  64 columns
// per step rather than 16 because the time of a small batch is the number of
// dependent memory round trips; large ones are bound by the row gather.
// Kernel time against a wavefront per query with sorted insertions: 1 query
// of 128 columns, L = 64 30 → 13.5 µs; 101 queries of 200 columns, k = 100,
// L = 256 208 → 37; 32 queries of 1,536 columns, L = 64 209 → 45; 16,384
// queries of 128 columns, L = 64 299 → 218 (1.07 GB if every row were read);
// 4,096 queries of 768 columns, k = 100, L = 128 541 → 490 (3.2 GB).
constexpr int kRrMaxL = 256;
constexpr int kRrCand = kRrMaxL + kDegenCap;
constexpr int kRrRows = 16, kRrCols = 64;
// Queries from which reading fewer rows beats fewer rounds (16,384 queries,
// L = 64, k = 10: 218 µs in two rounds, 312 in one before the orderings were
// vectorized; 1 query: 13.5 µs in one).
constexpr int kRrBulk = 1024;

struct RrShared {
  double stage[4][kRrRows + 1][kRrCols + 1];  // the last row: the query
  uint64_t k64[kRrCand];
  float okey[kRrCand];
  uint32_t oslot[kRrCand];
  uint32_t count;  // candidates that need a score, or may
  uint64_t tau;    // the k-th FP64 key
  float kmax;
  float errw[4], kmaxw[4];
  int n2;
};
static_assert(sizeof(RrShared) <= 160 * 1024 / 4, "four blocks per CU");

// FP64 rank keys of the ordered candidates c0 .. c0+15 below n (one
// wavefront).
template <bool L2M>
__device__ __forceinline__ void rr_score(const RerankArgs& a, const QParams& qp, int metric,
                                         const double* __restrict__ qv, RrShared& sm, int wave,
                                         int lane, uint32_t c0, uint32_t n) {
  double(*stg)[kRrCols + 1] = sm.stage[wave];
  const double* src[kRrRows];
#pragma unroll
  for (int u = 0; u < kRrRows; u++)
    src[u] = a.st.X + (size_t)uni32(sm.oslot[min(c0 + u, n - 1)]) * a.st.ldx;
  double v[kRrRows], qe = 0.0;
  auto fetch = [&](uint32_t col) __attribute__((always_inline)) {
    const uint32_t e = col + lane;
    const bool in = e < a.d;
    qe = in ? qv[e] : 0.0;
#pragma unroll
    for (int u = 0; u < kRrRows; u++) v[u] = in ? src[u][e] : 0.0;
  };
  double acc = 0.0;
  const double* my = stg[lane & 15];
  const double* qr = stg[kRrRows];
  fetch(0);
  for (uint32_t col = 0; col < a.d; col += kRrCols) {
#pragma unroll
    for (int u = 0; u < kRrRows; u++) stg[u][lane] = v[u];
    stg[kRrRows][lane] = qe;
    __builtin_amdgcn_wave_barrier();
    if (col + kRrCols < a.d) fetch(col + kRrCols);
    __builtin_amdgcn_sched_barrier(0);
    // (columns past d are zero in both operands: they leave the chain as it
    // is, up to the sign of a zero, which ranking and scores fold)
    const uint32_t ne = min((uint32_t)kRrCols, (a.d - col + 7) & ~7u);
    for (uint32_t t0 = 0; t0 < ne; t0 += 8) {
      double x[8], q[8];
#pragma unroll
      for (int t = 0; t < 8; t++) {
        x[t] = my[t0 + t];
        q[t] = qr[t0 + t];
      }
#pragma unroll
      for (int t = 0; t < 8; t++) {
        if (L2M) {
          const double tt = x[t] - q[t];
          acc = fma(tt, tt, acc);
        } else {
          acc = fma(q[t], x[t], acc);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  const uint32_t c = c0 + lane;
  if (lane < kRrRows && c < n) {
    double r = acc;
    if (metric == kDot) r = -acc;
    else if (metric == kCos) r = -(acc / (qp.qn * a.st.xn[sm.oslot[c]]));
    sm.k64[c] = rank_bits(r);
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_rerank(
    RangeBatch<RerankArgs> b) {
  __shared__ RrShared sm;
  // the candidates before they are ordered: in the stage, not yet in use
  // (their keys as order-preserving bits, all ones for the unusable ones)
  uint32_t* ckey = reinterpret_cast<uint32_t*>(&sm.stage[0][0][0]);
  uint32_t* cslot = reinterpret_cast<uint32_t*>(&sm.stage[1][0][0]);
  const int ri = range_of(b, blockIdx.x);
  const RerankArgs& a = b.r[ri];
  const int metric = b.metric[ri];
  const uint32_t q = blockIdx.x - b.first[ri];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const QParams qp = a.qp[q];
  const double* __restrict__ qv = a.Q + (size_t)q * a.ldq;
  const uint32_t ndeg_all = *a.degen_count;
  const uint32_t ndeg = min(ndeg_all, (uint32_t)kDegenCap);
  const uint32_t nc = a.L + ndeg, kk = a.k;
  auto lower = [&](float bo) -> double { return lowp_lower(bo, qp, metric, a.d); };

  // candidates: (slot, key), the unusable ones keyed +inf; degenerate rows
  // first in the order, unless the shortlist holds them too
  float kmax = -INFINITY;
  for (uint32_t j = tid; j < nc; j += 256) {
    uint32_t slot;
    float key = -INFINITY;
    if (j < a.L) {
      slot = a.short_slot[(size_t)q * a.L + j];
      key = a.short_key[(size_t)q * a.L + j];
      kmax = fmaxf(kmax, key);
    } else {
      slot = a.degen[j - a.L];
    }
    const bool ok = slot < a.st.nrows && ((a.st.alive[slot >> 6] >> (slot & 63)) & 1ull);
    cslot[j] = slot;
    ckey[j] = ok ? rank_bits32(key) : ~0u;
  }
  if (tid < 3) ckey[nc + tid] = ~0u;
  if (tid == 0) {
    sm.count = 0;
    sm.tau = ~0ull;
    sm.n2 = 0;
  }
  for (int o = 32; o >= 1; o >>= 1) kmax = fmaxf(kmax, __shfl_xor(kmax, o));
  if (lane == 0) sm.kmaxw[wave] = kmax;
  __syncthreads();
  for (uint32_t j = a.L + tid; j < nc; j += 256) {
    const uint32_t slot = cslot[j];
    bool dup = false;
    for (uint32_t t = 0; t < a.L; t++) dup |= cslot[t] == slot;
    if (dup) ckey[j] = ~0u;
  }
  __syncthreads();
  // order by (key, position), unusable ones out
  for (uint32_t j = tid; j < nc; j += 256) {
    const uint32_t kb = ckey[j];
    if (kb == ~0u) continue;
    uint32_t pos = 0;
    for (uint32_t t = 0; t < nc; t += 4) {
      const uint4 o = *reinterpret_cast<const uint4*>(ckey + t);
      pos += (o.x < kb) | ((o.x == kb) & (t < j));
      pos += (o.y < kb) | ((o.y == kb) & (t + 1 < j));
      pos += (o.z < kb) | ((o.z == kb) & (t + 2 < j));
      pos += (o.w < kb) | ((o.w == kb) & (t + 3 < j));
    }
    sm.oslot[pos] = cslot[j];
    sm.okey[pos] = __uint_as_float((kb >> 31) ? (kb & 0x7FFFFFFFu) : ~kb);
    atomicAdd(&sm.count, 1u);
  }
  __syncthreads();
  const uint32_t n = sm.count;
  // First round.  A large batch is bound by the rows it reads: no more than
  // the k (and the degenerate rows) are read before their k-th key can bound
  // the rest.  A small one is bound by latency: the four wavefronts read 64
  // rows at once.
  uint32_t m1 = (kk + ndeg + kRrRows - 1) & ~(uint32_t)(kRrRows - 1);
  if (a.nq < (uint32_t)kRrBulk) m1 = max(m1, 4u * kRrRows);
  m1 = min(m1, n);
  auto score = [&](uint32_t c0, uint32_t end) {
    for (uint32_t c = c0 + kRrRows * wave; c < end; c += 4 * kRrRows) {
      if (metric == kL2) rr_score<true>(a, qp, metric, qv, sm, wave, lane, c, end);
      else rr_score<false>(a, qp, metric, qv, sm, wave, lane, c, end);
    }
  };
  // entry j's rank among the first m scored rows, by (key, slot)
  auto rank_of = [&](uint32_t j, uint32_t m) {
    const uint64_t K = sm.k64[j];
    const uint32_t S = sm.oslot[j];
    uint32_t r = 0;
    for (uint32_t t = 0; t < m; t++) r += lex_lt(sm.k64[t], sm.oslot[t], K, S);
    return r;
  };
  score(0, m1);
  __syncthreads();
  uint32_t ns = m1;  // rows scored
  if (n > m1) {
    for (uint32_t j = tid; j < m1; j += 256)
      if (rank_of(j, m1) + 1 == kk) sm.tau = sm.k64[j];
    __syncthreads();
    // A row whose lower bound exceeds the k-th value cannot be in the top k
    // (a flagged query's keys carry no bound; a NaN bound keeps its row).
    const double thr = !qp.flags && sm.tau != ~0ull ? rank_value(sm.tau) : INFINITY;
    int mine = 0;
    for (uint32_t j = m1 + tid; j < n; j += 256) mine = !(lower(sm.okey[j]) > thr) ? (int)j + 1 : mine;
    if (mine) atomicMax(&sm.n2, mine);
    __syncthreads();
    ns = max(m1, (uint32_t)sm.n2);
    if (tid == 0) sm.tau = ~0ull;
    score(m1, ns);
    __syncthreads();
  }
  uint32_t rk[2] = {~0u, ~0u};
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const uint32_t j = tid + 256 * p;
    if (j < ns) {
      rk[p] = rank_of(j, ns);
      if (rk[p] + 1 == kk) sm.tau = sm.k64[j];
    }
  }
  __syncthreads();

  // certification (more degenerate rows than the list holds: nothing can be
  // certified)
  const double tau = sm.tau == ~0ull ? INFINITY : rank_value(sm.tau);
  const bool cert =
      !qp.flags && ndeg_all <= (uint32_t)kDegenCap && tau < lower(a.beta[q]);
  if (!cert) {
    if (a.lk) {
#pragma unroll
      for (int p = 0; p < 2; p++)
        if (rk[p] < kk) {
          a.lk[(size_t)q * kk + rk[p]] = sm.k64[tid + 256 * p];
          a.ls[(size_t)q * kk + rk[p]] = sm.oslot[tid + 256 * p];
        }
      for (uint32_t e = ns + tid; e < kk; e += 256) {
        a.lk[(size_t)q * kk + e] = ~0ull;
        a.ls[(size_t)q * kk + e] = ~0u;
      }
    }
    if (tid == 0) {
      if (a.lk)
        a.kmax[q] = fmaxf(fmaxf(sm.kmaxw[0], sm.kmaxw[1]), fmaxf(sm.kmaxw[2], sm.kmaxw[3]));
      a.fail_list[atomicAdd(a.fail_count, 1u)] = q;
      a.max_rel_err[q] = -1.0;
    }
    return;
  }
  double err = 0.0;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    if (rk[p] >= kk) continue;
    const uint32_t j = tid + 256 * p, slot = sm.oslot[j];
    const double v = rank_value(sm.k64[j]);
    double sc = __longlong_as_double(0x7FF8000000000000ll);
    if (v == v) sc = metric == kL2 ? sqrt(v) : (v == 0.0 ? 0.0 : -v);
    const uint64_t id =
        a.st.has_deletes
            ? (uint64_t)a.st.rank_base[slot >> 6] +
                  (uint64_t)__popcll(a.st.alive[slot >> 6] & ((1ull << (slot & 63)) - 1ull))
            : slot;
    const float O = sm.okey[j];
    if (O > -INFINITY && O < INFINITY)
      err = fmax(err, lowp_rel_err(O, sc, slot, qp, metric, a));
    a.ids[(size_t)q * a.ostride + rk[p]] = id;
    a.scores[(size_t)q * a.ostride + rk[p]] = sc;
  }
  for (uint32_t e = ns + tid; e < kk; e += 256) {
    a.ids[(size_t)q * a.ostride + e] = ~0ull;
    a.scores[(size_t)q * a.ostride + e] = __longlong_as_double(0x7FF8000000000000ll);
  }
  for (int off = 32; off >= 1; off >>= 1) err = fmax(err, __shfl_xor(err, off));
  if (lane == 0) sm.stage[wave][0][0] = err;
  __syncthreads();
  if (tid == 0)
    a.max_rel_err[q] = fmax(fmax(sm.stage[0][0][0], sm.stage[1][0][0]),
                            fmax(sm.stage[2][0][0], sm.stage[3][0][0]));
}

hipError_t launch_rerank_ranges(const RerankArgs* a, const int* metric, int n, hipStream_t s) {
  for (int r0 = 0; r0 < n; r0 += kMaxLaunchRanges) {
    RangeBatch<RerankArgs> b{};
    uint32_t blocks = 0;
    b.n = 0;
    for (int r = r0; r < n && b.n < kMaxLaunchRanges; r++) {
      if (metric[r] != kL2 && metric[r] != kCos && metric[r] != kDot) return hipErrorInvalidValue;
      if (a[r].L > (uint32_t)kRrMaxL || a[r].carry || a[r].qidx) return hipErrorInvalidValue;
      b.r[b.n] = a[r];
      b.metric[b.n] = metric[r];
      b.first[b.n] = blocks;
      blocks += a[r].nq;
      b.n++;
    }
    b.first[b.n] = blocks;
    if (blocks == 0) continue;
    hipLaunchKernelGGL(k_rerank, dim3(blocks), dim3(256), 0, s, b);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// ------------------------------------------------------------- fallback plumbing

// Rebuilds a shadow's degenerate-row list from the store: a live slot whose
// penalty is +inf holds a degenerate row (dead slots carry +inf too, and
// are skipped).  Slots deleted or rewritten since their row entered the
// list drop out, so the list holds only rows that are still degenerate.
// `count` must be zero on entry (k_zero_u32); the list's order is
// immaterial (the rerank ranks its rows by key and slot).
__global__ void k_zero_u32(uint32_t* __restrict__ p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

__global__ void k_collect_degen(const float* __restrict__ pen, const uint64_t* __restrict__ alive,
                                uint32_t nslots, uint32_t* __restrict__ count,
                                uint32_t* __restrict__ list) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslots) return;
  if (!((alive[s >> 6] >> (s & 63)) & 1ull) || !(pen[s] == INFINITY)) return;
  const uint32_t idx = atomicAdd(count, 1u);
  if (idx < (uint32_t)kDegenCap) list[idx] = s;
}

hipError_t launch_rebuild_degen(const float* pen, const uint64_t* alive, uint32_t nslots,
                                uint32_t* count, uint32_t* list, hipStream_t s) {
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, count, 1u);
  if (nslots)
    hipLaunchKernelGGL(k_collect_degen, dim3((nslots + 255) / 256), dim3(256), 0, s, pen, alive,
                       nslots, count, list);
  return hipGetLastError();
}

__global__ void k_gather_rows(const double* __restrict__ src, size_t lds,
                              const uint32_t* __restrict__ idx, uint32_t n, uint32_t d,
                              double* __restrict__ dst, size_t ldd) {
  const uint32_t r = blockIdx.x;
  if (r >= n) return;
  const double* s = src + (size_t)idx[r] * lds;
  for (uint32_t c = threadIdx.x; c < d; c += blockDim.x) dst[(size_t)r * ldd + c] = s[c];
}

hipError_t launch_gather_rows(const double* src, size_t lds, const uint32_t* idx, uint32_t n,
                              uint32_t d, double* dst, size_t ldd, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_rows, dim3(n), dim3(64), 0, s, src, lds, idx, n, d, dst, ldd);
  return hipGetLastError();
}

__global__ void k_scatter_results(const uint64_t* __restrict__ ids, const double* __restrict__ sc,
                                  uint32_t k, const uint32_t* __restrict__ idx, uint32_t n,
                                  uint64_t* __restrict__ out_ids, double* __restrict__ out_sc,
                                  uint32_t ostride) {
  const uint32_t r = blockIdx.x;
  if (r >= n) return;
  const size_t o = (size_t)idx[r] * ostride;
  for (uint32_t j = threadIdx.x; j < k; j += blockDim.x) {
    out_ids[o + j] = ids[(size_t)r * k + j];
    out_sc[o + j] = sc[(size_t)r * k + j];
  }
}

hipError_t launch_scatter_results(const uint64_t* ids, const double* sc, uint32_t k,
                                  const uint32_t* idx, uint32_t n, uint64_t* out_ids,
                                  double* out_sc, uint32_t ostride, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_scatter_results, dim3(n), dim3(64), 0, s, ids, sc, k, idx, n, out_ids,
                     out_sc, ostride);
  return hipGetLastError();
}

}  // namespace svdb
