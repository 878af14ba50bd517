// svdb_bins.h — finding the r-th smallest of unsigned values by counts over 256
// bins (internal; device code and host).
//
// Values in [lo, hi] are counted into 256 bins of equal width, and the range
// shrinks to the bin the r-th falls into, until it holds one value.
#pragma once

#include <stdint.h>

namespace svdb {

// The bins are 2^bin_shift wide: the fewest bits that leave 256 of them over
// values hi - lo = w apart.
constexpr int bin_shift(uint32_t w) { return w >> 8 ? 24 - __builtin_clz(w) : 0; }
constexpr int bin_shift(uint64_t w) { return w >> 8 ? 56 - __builtin_clzll(w) : 0; }

// The last value of a bin of [lo, hi], which begins at lo + (bin << shift).  The
// last bin may reach past hi, and past the type's largest value: no sum is taken
// before that is known.
template <typename U>
constexpr U bin_last(U lo, U hi, uint32_t bin, int shift) {
  const U top = ((U)bin << shift) | (((U)1 << shift) - 1);
  return top >= hi - lo ? hi : lo + top;
}

}  // namespace svdb
