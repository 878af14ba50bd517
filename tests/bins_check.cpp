// The narrowing of svdb_bins.h against a sort: it ends, and at the r-th value, also
// where values reach the type's largest.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "svdb_bins.h"

template <typename U>
static bool check(const std::vector<U>& v, uint32_t r, const char* what) {
  std::vector<U> s(v);
  std::sort(s.begin(), s.end());
  U lo = s.front(), hi = s.back();
  uint32_t rank = r;
  for (int round = 0; lo != hi; round++) {
    const int shift = svdb::bin_shift((U)(hi - lo));
    uint32_t hist[256] = {};
    for (U x : v)
      if (x >= lo && x <= hi) {
        const U b = (U)(x - lo) >> shift;
        if (b > 255) return printf("%s: bin past 255\n", what), false;
        hist[b]++;
      }
    uint32_t bin = 0, cum = 0;
    while (bin < 256 && cum + hist[bin] < rank) cum += hist[bin++];
    if (bin == 256 || round == (int)sizeof(U))
      return printf("%s: rank %u lost in round %d\n", what, r, round), false;
    const U last = svdb::bin_last(lo, hi, bin, shift);
    lo += (U)bin << shift;
    hi = last;
    rank -= cum;
  }
  if (lo != s[r - 1]) return printf("%s: rank %u wrong\n", what, r), false;
  return true;
}

template <typename U>
static bool run(const char* what) {
  std::mt19937_64 g(1);
  const U top = ~(U)0;
  bool ok = true;
  for (int t = 0; t < 400; t++) {
    const int n = 2 + (int)(g() % 300);
    std::vector<U> v(n);
    for (auto& x : v) {
      const U a = (U)g();
      switch (t % 5) {
        case 0: x = a; break;                                       // anywhere
        case 1: x = a % 3 ? top - a % 5000 : a % 5000; break;        // both ends
        case 2: x = top - (a >> (a % (8 * sizeof(U)))); break;       // towards the top
        case 3: x = a % 7; break;                                    // few values
        default: x = (a % 20 ? top - (U)(top >> 9) - a % 4096 : 1 + a % 100);
      }
    }
    for (uint32_t r : {1u, (uint32_t)n / 2 + 1, (uint32_t)n}) ok = ok && check<U>(v, r, what);
  }
  return ok;
}

int main() {
  if (!run<uint32_t>("32 bits") || !run<uint64_t>("64 bits")) return 1;
  puts("ok");
  return 0;
}
