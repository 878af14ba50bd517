// svdb_f64_lists.h — the partial lists of the FP64 scan on the matrix cores
// (internal; host code).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace svdb {

constexpr uint32_t kF64StageRows = 64;  // rows of a row step
constexpr uint32_t kF64MaxCap = 320;    // entries of a list, at most
constexpr uint32_t kF64Queries = 64;    // queries of a block

// Rows of a slice, of P over the store.
inline uint32_t f64_slice_rows(uint32_t nrows, uint32_t P) {
  const uint32_t rows = (uint32_t)(((uint64_t)nrows + P - 1) / P);
  return (rows + kF64StageRows - 1) / kF64StageRows * kF64StageRows;
}

// The sample's share of the rows: one in kF64Share up to 128 columns; wider,
// where an insertion costs less beside the products, as much less (300k × 768,
// 1,024 queries: dot 11.5 ms with 1/16 and a test per query value, 9.95 so; a
// share falling with the square of the width: Euclidean 12.5 → 18.7).
constexpr uint32_t kF64Share = 16;
inline uint32_t f64_share(uint32_t D) { return kF64Share * ((D + 127) / 128); }

// The sample's runs of row steps, 16 minima each, or 0 where there would be less
// than twice k of them: one run per 1,024 rows up to 64, on small stores up to a
// quarter of the rows for enough minima.
constexpr uint32_t kF64MaxRuns = 64;
inline uint32_t f64_sample_runs(uint32_t nrows, int kmax, uint32_t D, size_t most) {
  const uint32_t want = (((uint32_t)kmax + 7) / 8 + 7) / 8 * 8;
  uint32_t S = std::max(nrows / 1024, std::min(want, nrows / 256));
  if (D > 128) S = std::min(S, std::max(want, nrows / f64_share(D) / 64));
  S = (uint32_t)std::min<size_t>({S, kF64MaxRuns, most}) / 8 * 8;
  return 16 * S >= 2 * (uint32_t)kmax ? S : 0;
}

// P lists per query of cap entries each; entries: what they and their counts
// (a count as an entry) take together.
struct F64Lists {
  uint32_t P, cap;
  size_t entries;
};

// Slices for about 512 blocks (two per CU, one round: the fewer and longer a
// query's lists, the sooner their bounds are tight), at least 64 rows each (a
// one-query call over 10,000 rows: 8 slices of 1,250 rows took 193 µs per
// call, 64 slices 88 µs).
//
// A list takes the k that a cut leaves it and twice the rows that the sample's
// bound is expected to bring it, at least 8 + k (a cut takes some 3 µs), or
// its whole slice if that is less or there is no sample.  512 lists of k + 192
// entries a query, whatever would enter them, were 101 MB for 64 queries at k =
// 1 (now 4) and no faster.
//
// Within max_entries, first the lists are shortened to k + 8 entries, then
// there are fewer of them, down to one per 2^27 rows (a queued pair holds the
// row's place in its slice in 28 bits); `entries` says whether that was enough.
inline F64Lists scan_f64_lists(uint32_t nrows, uint32_t nq, int kmax, uint32_t D,
                               size_t max_entries) {
  if (nrows == 0 || nq == 0) return F64Lists{0, 0, 0};
  const uint32_t k = (uint32_t)kmax;
  const uint32_t groups = (nq + kF64Queries - 1) / kF64Queries;
  uint32_t P = (512 + groups - 1) / groups;
  P = std::min<uint32_t>(P, (nrows + kF64StageRows - 1) / kF64StageRows);
  if (P >= 8) P = P / 8 * 8;
  const uint32_t minP = (nrows >> 27) + 1;
  P = std::max(P, minP);
  const bool sample = f64_sample_runs(nrows, kmax, D, kF64MaxRuns) != 0;
  auto lists = [&](uint32_t p, bool tight) {
    const uint32_t rows = f64_slice_rows(nrows, p);
    const uint32_t expected = sample ? f64_share(D) * k / p : rows;
    const uint32_t more = tight ? 8 : std::max(8 + k, 2 * std::min(expected, kF64MaxCap));
    const uint32_t cap = std::min({k + more, kF64MaxCap, rows});
    return F64Lists{p, cap, (size_t)nq * p * (cap + 1)};
  };
  F64Lists l = lists(P, false);
  if (l.entries > max_entries) l = lists(P, true);
  while (l.entries > max_entries && P > minP) {
    P = std::max(minP, P > 8 ? P / 16 * 8 : P / 2);
    l = lists(P, true);
  }
  return l;
}

}  // namespace svdb
