// Exact quotients n / d of every n up to 2^31 by a divisor that is fixed for a launch: multiply-high and a shift.
//
// With 2^s < d <= 2^(s+1) and m = ceil(2^(32+s) / d) < 2^32, m * d exceeds 2^(32+s) by e < d <= 2^(s+1), so n * e stays below
// 2^(32+s) for n <= 2^31 and n * m / 2^(32+s) is less than 1 / d above n / d: the same whole number.  Without the shift (m =
// ceil(2^32 / d)) that ends at n * e = 2^32, which dividends just above d reach from d = 65537 on.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define APNN_QUOTIENT_FN __host__ __device__ __forceinline__
#else
#define APNN_QUOTIENT_FN inline
#endif

namespace apnn {

// s (0 for d == 1, whose quotient needs none)
APNN_QUOTIENT_FN int quotient_shift(uint32_t d) { return d >= 2 ? 31 - __builtin_clz(d - 1) : 0; }

// m (0 for d == 1)
inline uint32_t quotient_magic(uint32_t d) {
  return d >= 2 ? (uint32_t)(((1ull << (32 + quotient_shift(d))) + d - 1) / d) : 0u;
}

APNN_QUOTIENT_FN uint32_t quotient(uint32_t n, uint32_t d, uint32_t magic, int shift) {
  return d == 1 ? n : (uint32_t)(((unsigned long long)n * magic) >> 32) >> shift;
}

}  // namespace apnn
