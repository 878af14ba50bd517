// The sizes of the FP64 scan's partial lists (svdb_f64_lists.h) over stores,
// batches, k and limits.
#include <cstdio>

#include "svdb_f64_lists.h"

using namespace svdb;

static int fail(const char* what, uint32_t n, uint32_t nq, int k, uint32_t D, size_t most) {
  printf("%s: %u rows, %u queries, k = %d, %u columns, limit %zu\n", what, n, nq, k, D, most);
  return 1;
}

int main() {
  const uint32_t rows[] = {1, 63, 64, 65, 1000, 2047, 2048, 20000, 50000, 1u << 20, 100000000,
                           (1u << 27) - 1};
  const uint32_t batches[] = {1, 2, 63, 64, 65, 300, 1024, 8192};
  const int ks[] = {1, 2, 3, 10, 64, 65, 100, 127, 128};
  const uint32_t widths[] = {1, 100, 128, 129, 768, 1536, 100000};
  for (uint32_t n : rows)
    for (uint32_t nq : batches)
      for (int k : ks)
        for (uint32_t D : widths) {
          // what a search takes, and the least that it was ever accepted with: 32
          // lists of k entries a query
          const size_t least = (size_t)nq * 32 * k;
          const size_t take[] = {std::max<size_t>((size_t)1 << 25, least), least, least + 100,
                                 4 * least, 0};
          for (size_t most : take) {
            const F64Lists l = scan_f64_lists(n, nq, k, D, most);
            const uint32_t slice = f64_slice_rows(n, l.P ? l.P : 1);
            if (!l.P || l.entries != (size_t)nq * l.P * (l.cap + 1))
              return fail("entries", n, nq, k, D, most);
            if (most && l.entries > most) return fail("past the limit", n, nq, k, D, most);
            if (l.cap > kF64MaxCap || (l.cap <= (uint32_t)k && l.cap < slice))
              return fail("a list that no cut can help", n, nq, k, D, most);
            const uint32_t S = f64_sample_runs(n, k, D, (size_t)l.P * l.cap / 8);
            if (S % 8 || S > kF64MaxRuns || (S && 16 * S < 2 * (uint32_t)k) ||
                (size_t)S * 8 > (size_t)l.P * l.cap || (S && n / S < 64))
              return fail("sample", n, nq, k, D, most);
          }
        }
  // more rows than a slice's place of a pair has bits for
  for (uint32_t n : {1u << 27, 1u << 31, 4294967231u}) {
    const F64Lists l = scan_f64_lists(n, 64, 1, 8, 0);
    if (((uint64_t)f64_slice_rows(n, l.P) - 1) >> 28) return fail("slice", n, 64, 1, 8, 0);
  }
  // (12 bytes an entry) a batch body's lists stay small
  if (scan_f64_lists(50000, 64, 1, 128, 1 << 25).entries * 12 > 5000000)
    return fail("memory", 50000, 64, 1, 128, 1 << 25);
  if (scan_f64_lists(50000, 512, 10, 128, 1 << 25).entries * 12 > 16000000)
    return fail("memory", 50000, 512, 10, 128, 1 << 25);
  puts("ok");
  return 0;
}
