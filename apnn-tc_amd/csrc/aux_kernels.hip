// Small helper kernels around the hot path.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "dispatch.h"

namespace apnn {

// ---- bit-plane packers ---------------------------------------------------------------------------------
// One kernel for every packer of the library (layout of Bit_compression, APNN-TC-nn/src/kernel.cuh:46-77): a
// source functor turns element (row, channel) into a code, and bits first .. bits-1 of the codes leave as
// planes [bits - first][rows][cpad/32], channel c at bit 31 - c%32.
//
// Bound by memory traffic (4 bytes read per sample against bits / 8 written), so the kernel is built to keep
// loads in flight and stores whole.  Words are numbered across rows (word w = row w / cw, channels 32 * (w %
// cw) ..), a wave owns 2 * UNITS consecutive words, and unit i is one load of words 2i and 2i + 1, one per
// lane half: all UNITS loads are requested before the first code is formed.  Lane l of a half reads channel
// 31 - l, so the compare mask of a bit IS the two packed words; masks are parked in the lane whose index is
// the word (v_writelane), and each plane then leaves in one store of 2 * UNITS consecutive words.
// FLAT: rows without padding (C a multiple of 32): an element's address is its index.  Otherwise a lane
// tracks (row, word of the row) by addition, so rows of any width take the same path and a row of at most 32
// channels costs half a wave, not a whole one.
// Float quantizer, 200704 x 64 samples to two planes (51 MB read, 3.2 MB written): 27.9 us with one 64-sample
// group per wave and an IEEE division per sample, 11.1 us as it is now (54 MB at the
// 5.1 TB/s of a large device copy: 10.6 us).
//
// park_words: old with lanes 2i and 2i + 1 replaced by the two halves of a compare mask.  A vector instruction
// that reads a scalar register written by the vector instruction just before it needs wait states, which the
// compiler does not insert for this opaque assembly: the block waits by itself (s_nop 1).
__device__ __forceinline__ int park_words(int i, unsigned long long mask, int old) {
  asm("s_nop 1\n\t"
      "v_writelane_b32 %0, %1, %3\n\t"
      "v_writelane_b32 %0, %2, %4"
      : "+v"(old)
      : "s"((int)(uint32_t)mask), "s"((int)(uint32_t)(mask >> 32)), "i"(2 * i), "i"(2 * i + 1));
  return old;
}

template <int UNITS, bool FLAT, class Src>
__global__ __launch_bounds__(256) void pack_planes_kernel(Src src, uint32_t *__restrict__ planes, long long words, int C,
                                                          int cw, int first, int bits, long long block0) {
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int ch = 31 - (lane & 31);
  const long long wave = (block0 + blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long w0 = wave * (2 * UNITS);
  if (w0 >= words) return;
  typename Src::Raw raw[UNITS];
  bool ok[UNITS];
  if (FLAT && w0 + 2 * UNITS <= words) {  // whole wave inside: one base address, constant offsets
    const long long e0 = (w0 + half) * 32 + ch;
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      ok[i] = true;
      raw[i] = src.load(e0 + 64 * i);
    }
  } else {
    long long row = (w0 + half) / cw;
    int wi = (int)((w0 + half) - row * cw);
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const int c = wi * 32 + ch;
      ok[i] = w0 + 2 * i + half < words && c < C;
      raw[i] = src.load(ok[i] ? row * C + c : 0ll);
      wi += 2;
      while (wi >= cw) {  // at most twice: cw >= 1
        wi -= cw;
        ++row;
      }
    }
  }
  uint32_t code[UNITS];
#pragma unroll
  for (int i = 0; i < UNITS; ++i) code[i] = ok[i] ? src.code(raw[i]) : 0u;
  const bool store = lane < 2 * UNITS && w0 + lane < words;
  for (int b = first; b < bits; ++b) {
    int park = 0;
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const unsigned long long mask = __ballot((code[i] & (1u << b)) != 0u);
      park = park_words(i, mask, park);
    }
    if (store) planes[(b - first) * words + w0 + lane] = (uint32_t)park;
  }
}

// Codes as they are (Bit_compression).
struct CodeSource {
  typedef uint32_t Raw;
  const uint32_t *values;
  __device__ __forceinline__ Raw load(long long e) const { return values[e]; }
  __device__ __forceinline__ uint32_t code(Raw v) const { return v; }
};

// uint8 samples: the top `bits` bits, a uniform 2^bits-level quantizer of [0, 256).
struct ByteSource {
  typedef uint8_t Raw;
  const uint8_t *values;
  int shift;
  __device__ __forceinline__ Raw load(long long e) const { return values[e]; }
  __device__ __forceinline__ uint32_t code(Raw v) const { return (uint32_t)v >> shift; }
};

// Float samples: one bit, x >= 0 (In128Layer, APNN-TC-nn/src/kernel.cuh:321-340).
struct SignSource {
  typedef float Raw;
  const float *values;
  __device__ __forceinline__ Raw load(long long e) const { return values[e]; }
  __device__ __forceinline__ uint32_t code(Raw v) const { return v >= 0.0f ? 1u : 0u; }
};

// Quantize_val (APNN-TC-nn/src/kernel.cuh:29-44): clip, then rint(((x - min) * levels) / range) in fp32, every
// operation rounded to nearest.  A NaN gives code 0 (it clips to min).
// FAST: the division by the launch-wide range as a multiplication with its correctly rounded reciprocal y and
// one correction, q = t*y, q + (t - q*range)*y with two fused multiply-adds: the correctly rounded quotient
// whenever y is and nothing over- or underflows (P. Markstein, "Computation of elementary functions on the
// IBM RISC System/6000 processor", 1990, theorem on division).  Quotients small enough to underflow round to
// code 0 either way; the host takes this form for ranges between 2^-60 and 2^60 only.  Three operations
// instead of the eleven of an IEEE division.
template <bool FAST>
struct QuantSource {
  typedef float Raw;
  const float *values;
  float min_v, max_v, levels, range, inv_range;
  uint32_t top;
  __device__ __forceinline__ Raw load(long long e) const { return values[e]; }
  __device__ __forceinline__ uint32_t code(Raw x) const {
    x = fminf(fmaxf(x, min_v), max_v);
    const float t = __fmul_rn(__fsub_rn(x, min_v), levels);
    float q;
    if constexpr (FAST) {
      q = __fmul_rn(t, inv_range);
      q = __builtin_fmaf(__builtin_fmaf(-q, range, t), inv_range, q);
    } else {
      q = __fdiv_rn(t, range);
    }
    return min(top, __float2uint_rn(q));
  }
};

template <class Src>
static hipError_t launch_pack_planes(const Src &src, uint32_t *planes, int rows, int C, int cpad, int first, int bits,
                                     hipStream_t s) {
  const int cw = cpad / 32;
  const long long words = (long long)rows * cw;
  const bool flat = C == cpad;
  // 64 words per wave while that still gives every SIMD a wave or two; smaller tensors are cut finer, so that
  // the few waves there are do not walk 32 units one after the other
  auto go = [&](auto units_c, auto flat_c) {
    constexpr int UNITS = decltype(units_c)::value;
    constexpr bool FLAT = decltype(flat_c)::value;
    const long long blocks = (words + 8 * UNITS - 1) / (8 * UNITS);
    // a grid holds fewer than 2^32 threads; tensors of more words go out in parts
    constexpr long long most = (1ll << 24) - 1;
    for (long long b0 = 0; b0 < blocks; b0 += most)
      hipLaunchKernelGGL((pack_planes_kernel<UNITS, FLAT, Src>), dim3((unsigned)(blocks - b0 < most ? blocks - b0 : most)), dim3(256),
                         0, s, src, planes, words, C, cw, first, bits, b0);
  };
  using std::integral_constant;
  if (words >= 64 * 2048) {
    if (flat) go(integral_constant<int, 32>{}, std::true_type{}); else go(integral_constant<int, 32>{}, std::false_type{});
  } else {
    if (flat) go(integral_constant<int, 4>{}, std::true_type{}); else go(integral_constant<int, 4>{}, std::false_type{});
  }
  return hipGetLastError();
}

hipError_t launch_quantize_pack(const float *values, uint32_t *planes, int rows, int C, int cpad, int bits, float min_v,
                                float max_v, hipStream_t s) {
  const float levels = (float)(1 << bits), range = max_v - min_v;
  const uint32_t top = (1u << bits) - 1u;
  if (range >= 0x1p-60f && range <= 0x1p60f && fabsf(min_v) <= 0x1p60f)
    return launch_pack_planes(QuantSource<true>{values, min_v, max_v, levels, range, 1.0f / range, top}, planes, rows, C,
                              cpad, 0, bits, s);
  return launch_pack_planes(QuantSource<false>{values, min_v, max_v, levels, range, 0.0f, top}, planes, rows, C, cpad, 0,
                            bits, s);
}

hipError_t launch_pack_bits(const uint32_t *values, uint32_t *planes, int rows, int C, int cpad, int bits,
                            hipStream_t s) {
  return launch_pack_planes(CodeSource{values}, planes, rows, C, cpad, 0, bits, s);
}

// the top plane only (Bit_compression_fc_hidden)
hipError_t launch_pack_top_plane(const uint32_t *values, uint32_t *plane, int rows, int C, int cpad, int bits,
                                 hipStream_t s) {
  return launch_pack_planes(CodeSource{values}, plane, rows, C, cpad, bits - 1, bits, s);
}

hipError_t launch_quantize_pack_u8(const uint8_t *values, uint32_t *planes, int rows, int C, int cpad, int bits,
                                   hipStream_t s) {
  return launch_pack_planes(ByteSource{values, 8 - bits}, planes, rows, C, cpad, 0, bits, s);
}

hipError_t launch_binarize_pack(const float *values, uint32_t *planes, int rows, int C, int cpad, hipStream_t s) {
  return launch_pack_planes(SignSource{values}, planes, rows, C, cpad, 0, 1, s);
}

// int32 shortcut map -> residual operand of the quantizing epilogue: optional 2x2 max-pool of the source
// map and channel truncation / zero fill (the reference adds the residual to channels below
// residual_channels only and max-pools it when the block halves the map,
// APNN-TC-nn/src/kernel.cuh:779-831).  One thread per four output channels.
__global__ __launch_bounds__(256) void residual_prepare_kernel(const int32_t *__restrict__ in, int32_t *__restrict__ out,
                                                               long long quads, int Ho, int Wo, int in_pitch,
                                                               int channels, int out_channels, int pool) {
  const int q4 = (out_channels + 3) >> 2;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < quads;
       i += (long long)gridDim.x * blockDim.x) {
    const int cq = (int)(i % q4);
    const long long pix = i / q4;
    const int ox = (int)(pix % Wo);
    const long long t = pix / Wo;
    const int oy = (int)(t % Ho);
    const long long b = t / Ho;
    for (int j = 0; j < 4; ++j) {
      const int c = cq * 4 + j;
      if (c >= out_channels) break;
      int v = 0;
      if (c < channels) {
        if (pool) {
          const long long base = ((b * (2 * Ho) + 2 * oy) * (2 * Wo) + 2 * ox) * in_pitch + c;
          const long long down = (long long)(2 * Wo) * in_pitch;
          v = max(max(in[base], in[base + in_pitch]), max(in[base + down], in[base + down + in_pitch]));
        } else {
          v = in[pix * in_pitch + c];
        }
      }
      out[pix * out_channels + c] = v;
    }
  }
}

hipError_t launch_residual_prepare(const int32_t *in, int32_t *out, int B, int Ho, int Wo, int in_pitch, int channels,
                                   int out_channels, int pool, hipStream_t s) {
  const long long quads = (long long)B * Ho * Wo * ((out_channels + 3) / 4);
  long long blocks = (quads + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(residual_prepare_kernel, dim3((unsigned)blocks), dim3(256), 0, s, in, out, quads, Ho, Wo, in_pitch,
                     channels, out_channels, pool);
  return hipGetLastError();
}

}  // namespace apnn
