// Quotients n / d of a dividend that passes its divisor by less than 1024 (a tile's pixels over the rows and images of a map),
// by multiply-high.
//
// m = ceil(2^32 / d) exceeds 2^32 / d by e / d, e < d; n * m / 2^32 is the same whole number as n / d while n * e < 2^32, which
// holds for these dividends up to d = 65536 and ends at 65537 (n = 65536).  Beyond, with 2^s < d <= 2^(s+1), m = ceil(2^(32+s) /
// d) < 2^32 exceeds by e < d <= 2^(s+1), so n * e stays below 2^(32+s) for every n up to 2^31: exact with a shift by s.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define APNN_QUOTIENT_FN __host__ __device__ __forceinline__
#else
#define APNN_QUOTIENT_FN inline
#endif

namespace apnn {

constexpr uint32_t kShortDivisor = 65536;

// s (0 for d == 1, whose quotient needs none)
APNN_QUOTIENT_FN int quotient_shift(uint32_t d) { return d >= 2 ? 31 - __builtin_clz(d - 1) : 0; }

// m of the form without (SHORT, d up to kShortDivisor) and with a shift; 0 for d == 1
inline uint32_t quotient_magic(uint32_t d, bool is_short) {
  return d >= 2 ? (uint32_t)(((1ull << (is_short ? 32 : 32 + quotient_shift(d))) + d - 1) / d) : 0u;
}

APNN_QUOTIENT_FN uint32_t multiply_high(uint32_t n, uint32_t m) {
#ifdef __HIP_DEVICE_COMPILE__
  return __umulhi(n, m);
#else
  return (uint32_t)(((unsigned long long)n * m) >> 32);
#endif
}

template <bool SHORT>
APNN_QUOTIENT_FN uint32_t quotient(uint32_t n, uint32_t d, uint32_t magic) {
  if constexpr (SHORT) return d == 1 ? n : multiply_high(n, magic);
  return d == 1 ? n : multiply_high(n, magic) >> quotient_shift(d);
}

}  // namespace apnn
