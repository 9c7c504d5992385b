// Output stage of the FP4 / FP6 matrix-core convolution kernels.
//
// The convolution kernels multiply weights (first operand) by activations (second operand), so a lane of the
// accumulator holds ONE output pixel and its registers hold output channels: register r of a 32x32 block is
// channel 8*(r/4) + 4*g + r%4 of lane half g, pixel = lane % 32.  Everything the output stage does is then
// local to a lane:
//   * a code bit is appended to the lane's packed word by one add-with-carry (w = 2w + compare result), two
//     compares, one select and two of those per 2-bit code; the two lane halves hold alternate nibbles of a
//     word and meet in one half-wave swap that serves two planes at once;
//   * thresholds are read from a table in LDS, four consecutive channels per 16-byte broadcast read, scaled to
//     accumulator units: no multiplication per value.  A channel with the flip flag (codes fall with the value)
//     has the table entries 1 - t in reverse order and its word bits inverted at the end: for integers
//     #{k : -v >= t_k} = nt - #{k : v >= 1 - t_k}, and nt - c inverts all bits of c;
//   * corrections that depend on the pixel (activation sums) are one register per pixel block;
//   * the words of a packed shortcut are the lane's own, read straight into the operand of fold_shortcut_lanes;
//   * the four pixels of a 2x2 pooling window are four neighbouring lanes: the maximum of their codes is taken on
//     the finished bit-planes, two bitwise steps per word pair (codes of three and four bits: on the values, before
//     the search);
//   * int32 results of whole blocks pass 4 KB of LDS per wave, which turns them into rows: a store instruction writes
//     eight rows of 128 bytes.  Stored as a lane holds them, 16 bytes of 64 places, a short reduction with a large
//     result is bound by the partial lines (56x56x64 to 256 channels, 1x1 at batch 64, w1a2: 42.7 us, 35.4 in rows; 3x3
//     on 28x28x512 at batch 64: 69.8 and 62.5).  The shares of the split-K tiles are stored that way.
// With pixels in the registers and channels in the lanes, as these kernels were first built, a compare mask had
// to be reversed and moved to its row by four lane writes per 64 values: 128 vector and about 100 other
// operations per 32x32 block against 88 and 12 LDS reads here.  With the -1 / +1 weights this layout makes free of
// corrections: ResNet18 batch 64 254.0 -> 241.4 us, batch 8 106.0 -> 101.4 us, VGG variant batch 64 563 -> 541 us, w1a3
// 3x3 convolution of 512 channels on 16x16 maps at batch 16 12.8 -> 12.2 us.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "epilogue.h"
#include "kparams.h"

namespace apnn {

// 4-byte-aligned vectors: output and residual rows need not start on 16 bytes
typedef int i4 __attribute__((ext_vector_type(4)));
typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u2u __attribute__((ext_vector_type(2), aligned(4)));

// Threshold table of a work-group's channels, in LDS behind the operand buffers: float or int32 [nt][TB + 4] (a channel's
// thresholds lie in different banks: a search reads them with another index in every lane), then one word per 32 channels with the flip flags (channel c at bit 31 - c%32).  Present for BN codes of up to four
// bits; wider codes search the thresholds in memory.
__host__ __device__ constexpr int conv_table_words(int out_bits, int TB) { return ((1 << out_bits) - 1) * (TB + 4) + TB / 32; }

// words the table takes in a launch (0 where there is none)
__host__ __device__ inline int conv_table_words_of(const KParams &p, int TB) {
  return p.epi == APNN_EPI_BN && p.out_bits <= 4 ? (conv_table_words(p.out_bits, TB) + 3) & ~3 : 0;
}
// Whether codes are found by comparing fp32 values in accumulator units (float table); everything but these and int32
// results takes the general path over int32 values.
__host__ __device__ inline bool conv_float_codes(const KParams &p, int max_bits) {
  return p.epi == APNN_EPI_BN && p.out_bits <= max_bits && p.epi_float != 0 && p.pool != APNN_POOL_AVG2X2 &&
         !(p.pool == APNN_POOL_MAX2X2 && p.out_bits > 2) && p.resid == nullptr && p.save_acc == nullptr &&
         (p.resid_planes == nullptr || p.fold != 0u);
}
inline size_t conv_epilogue_bytes(const KParams &p, int TB) {
  return 4ull * conv_table_words_of(p, TB);
}

// The table is filled by one thread per channel.  load() requests the thresholds (first thing in the kernel, so that
// they arrive under the operands' latency), store() writes them to LDS; a barrier must follow before it is read.
// MAXT: thresholds kept in registers in between, the rest is read by store().
template <int TB, int MAXT, int MAXB>
struct ConvTable {
  int t[MAXT];
  int flip;

  __device__ __forceinline__ static bool present(const KParams &p) { return p.epi == APNN_EPI_BN && p.out_bits <= 4; }

  __device__ __forceinline__ void load(const KParams &p, int b0) {
    if (!present(p) || threadIdx.x >= TB) return;
    const int nt = (1 << p.out_bits) - 1;
    const int gcol = min(b0 + (int)threadIdx.x, p.rowsB - 1);
    const int32_t *src = p.thr + (long long)gcol * nt;
#pragma unroll
    for (int k = 0; k < MAXT; ++k) t[k] = src[min(k, nt - 1)];
    flip = p.flip != nullptr ? p.flip[gcol] : 0;
  }

  // inv: 1 / (value per accumulator unit), a power of two
  __device__ __forceinline__ void store(const KParams &p, int b0, uint32_t *tab, float inv) const {
    static_assert(TB % 64 == 0 || TB == 32, "whole waves, or half a wave");
    const int c = threadIdx.x;
    if (!present(p) || c >= TB) return;
    const int nt = (1 << p.out_bits) - 1;
    const bool as_float = conv_float_codes(p, MAXB), fl = flip != 0;
    auto put = [&](int k, int v) {
      if (as_float) {
        const int lim = 1 << 24;  // no value reaches it
        const int cl = min(max(v, -lim), lim);
        tab[(fl ? nt - 1 - k : k) * (TB + 4) + c] = __float_as_uint((float)(fl ? 1 - cl : cl) * inv);
      } else {
        tab[k * (TB + 4) + c] = (uint32_t)v;
      }
    };
#pragma unroll
    for (int k = 0; k < MAXT; ++k)
      if (k < nt) put(k, t[k]);
    const int32_t *src = p.thr + (long long)min(b0 + c, p.rowsB - 1) * nt;
    for (int k = MAXT; k < nt; ++k) put(k, src[k]);
    const unsigned long long m = __ballot(fl);
    if ((c & 31) == 0) tab[nt * (TB + 4) + (c >> 5)] = __brev((uint32_t)(m >> (c & 32)));
  }
};

// w = 16 w + four code bits, first value on top, for bit 1 and bit 0 of a 2-bit code: bit1 = v >= t1,
// bit0 = v >= (bit1 ? t2 : t0).  One block, because a vector instruction must not read a scalar register within
// two instructions of the vector instruction that wrote it, and the compiler does not see into assembly: each
// mask here is used at least three instructions after its compare.  For the same reason values that come straight from
// matrix instructions have to be settled by the caller (settle_results).
__device__ __forceinline__ void append_codes2(const float (&v)[4], const float (&t0)[4], const float (&t1)[4],
                                              const float (&t2)[4], uint32_t &w1, uint32_t &w0) {
  unsigned long long s0, s1, s2, s3;
  float x0, x1, x2, x3;
  asm("v_cmp_ge_f32_e64 %[s0], %[v0], %[b0]\n\t"
      "v_cmp_ge_f32_e64 %[s1], %[v1], %[b1]\n\t"
      "v_cmp_ge_f32_e64 %[s2], %[v2], %[b2]\n\t"
      "v_cmp_ge_f32_e64 %[s3], %[v3], %[b3]\n\t"
      "v_cndmask_b32_e64 %[x0], %[a0], %[c0], %[s0]\n\t"
      "v_cndmask_b32_e64 %[x1], %[a1], %[c1], %[s1]\n\t"
      "v_cndmask_b32_e64 %[x2], %[a2], %[c2], %[s2]\n\t"
      "v_cndmask_b32_e64 %[x3], %[a3], %[c3], %[s3]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s0]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s1]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s3]\n\t"
      "v_cmp_ge_f32_e64 %[s0], %[v0], %[x0]\n\t"
      "v_cmp_ge_f32_e64 %[s1], %[v1], %[x1]\n\t"
      "v_cmp_ge_f32_e64 %[s2], %[v2], %[x2]\n\t"
      "v_cmp_ge_f32_e64 %[s3], %[v3], %[x3]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s0]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s1]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s2]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s3]"
      : [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2), [s3] "=&s"(s3), [x0] "=&v"(x0), [x1] "=&v"(x1), [x2] "=&v"(x2),
        [x3] "=&v"(x3), [w1] "+v"(w1), [w0] "+v"(w0)
      : [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [a0] "v"(t0[0]), [a1] "v"(t0[1]), [a2] "v"(t0[2]),
        [a3] "v"(t0[3]), [b0] "v"(t1[0]), [b1] "v"(t1[1]), [b2] "v"(t1[2]), [b3] "v"(t1[3]), [c0] "v"(t2[0]),
        [c1] "v"(t2[1]), [c2] "v"(t2[2]), [c3] "v"(t2[3])
      : "vcc");
}

// w = 16 w + four bits from four compare masks, first mask on top (waits for the masks by itself, see above)
__device__ __forceinline__ void append_masks(unsigned long long m0, unsigned long long m1, unsigned long long m2,
                                             unsigned long long m3, uint32_t &w) {
  asm("s_nop 1\n\t"
      "v_addc_co_u32_e64 %[w], vcc, %[w], %[w], %[m0]\n\t"
      "v_addc_co_u32_e64 %[w], vcc, %[w], %[w], %[m1]\n\t"
      "v_addc_co_u32_e64 %[w], vcc, %[w], %[w], %[m2]\n\t"
      "v_addc_co_u32_e64 %[w], vcc, %[w], %[w], %[m3]"
      : [w] "+v"(w)
      : [m0] "s"(m0), [m1] "s"(m1), [m2] "s"(m2), [m3] "s"(m3)
      : "vcc");
}

// the value of lane (this ^ 1) / (this ^ 2) of the same quad
__device__ __forceinline__ uint32_t quad_xor1(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ uint32_t quad_xor2(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true); }

// Maximum of the codes of the four lanes of a quad, bit-sliced (32 codes per word, planes w[NB-1] .. w[0]).
template <int NB>
__device__ __forceinline__ void quad_max(uint32_t (&w)[NB], int nb) {
#pragma unroll
  for (int step = 0; step < 2; ++step) {
    uint32_t ga = ~0u, gb = ~0u;  // own / other code not smaller so far, from the top plane down
#pragma unroll
    for (int b = NB - 1; b >= 0; --b) {
      if (b < nb) {
        const uint32_t a = w[b], o = step == 0 ? quad_xor1(w[b]) : quad_xor2(w[b]);
        w[b] = (a & ga) | (o & gb);
        const uint32_t na = ga & (~gb | a | ~o), no = gb & (~ga | o | ~a);
        ga = na;
        gb = no;
      }
    }
  }
}

// Appends the codes of four channels (one register quad) of NX pixels: v[x][j] against the table's thresholds at
// channel `at`.  fp32 values in accumulator units; bit L of a code compares with the threshold that the bits above
// it select, read and selected as it is needed.
template <int NX, int NB, int TB>
__device__ __forceinline__ void conv_append_quad(const float (&v)[NX][4], const uint32_t *at, uint32_t *(&w)[NX]) {
  struct F4 {
    float v[4];
  };
  auto thr = [&](int k) {
    const float4 t = *reinterpret_cast<const float4 *>(at + k * (TB + 4));
    return F4{{t.x, t.y, t.z, t.w}};
  };
  if constexpr (NB == 2) {
    const F4 t0 = thr(0), t1 = thr(1), t2 = thr(2);
    static_for_e<0, NX>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      append_codes2(v[x], t0.v, t1.v, t2.v, w[x][1], w[x][0]);
    });
  } else {
    __builtin_amdgcn_sched_barrier(0);  // (keeps the threshold reads of later quads from piling up in registers)
    static_for_e<0, NX>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      bool h[NB][4];
      static_for_e<0, NB>([&](auto lc) {
        constexpr int L = NB - 1 - decltype(lc)::value;
        auto pick = [&](auto self, auto bit_c, int base) {
          constexpr int bit = decltype(bit_c)::value;
          if constexpr (bit == L) {
            return thr(base + (1 << L) - 1);
          } else {
            const F4 one = self(self, std::integral_constant<int, bit - 1>{}, base + (1 << bit));
            F4 r = self(self, std::integral_constant<int, bit - 1>{}, base);
#pragma unroll
            for (int j = 0; j < 4; ++j) r.v[j] = h[bit][j] ? one.v[j] : r.v[j];
            return r;
          }
        };
        const F4 t = pick(pick, std::integral_constant<int, NB - 1>{}, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) h[L][j] = v[x][j] >= t.v[j];
        append_masks(__ballot(h[L][0]), __ballot(h[L][1]), __ballot(h[L][2]), __ballot(h[L][3]), w[x][L]);
      });
    });
  }
}

// Words of a packed one- or two-bit shortcut for NX x NY blocks: lane li holds pixel row li's (both halves alike).
template <int NX, int NY>
__device__ __forceinline__ void conv_shortcut_load(const KParams &p, int rbase, int cbase, int li,
                                                   uint32_t (&sc)[NX][NY][2]) {
  const int w32 = p.rowsB >> 5;
  const long long plane = (long long)p.rowsA * w32;
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    const int row = min(rbase + x * 32 + li, p.rowsA - 1);
    const uint32_t *src = p.resid_planes + (long long)row * w32;
#pragma unroll
    for (int y = 0; y < NY; ++y) {
      const int wi = min((cbase >> 5) + y, w32 - 1);  // words past the end belong to outputs that are not stored
      sc[x][y][0] = src[wi];
      sc[x][y][1] = p.resid_bits > 1 ? src[plane + wi] : 0u;
    }
  }
}

// Output stage of one wave for NX pixel blocks of NY channel blocks (NQ = 4: whole blocks of 32 channels) or for a
// share of NQ quads of one channel block (NY = 1, NQ < 4; the split-K tiles).
//   value(x, y, i)   accumulator of channel 8 (i/4) + 4g + i%4 of the share, final except for `vs` (x, y, i: constants)
//   vs               value per accumulator unit (fp32 kernels)
//   rbase            first pixel row;  cbase: first channel of block 0;  q0: first quad of the share
//   MAXB             code widths with a path of their own; wider ones take the general integer path
//   slab             the work-group's operand buffers (1 KB per quad of the share and wave are used, after a barrier)
template <int NX, int NY, int NQ, int TB, int MAXB, class Value>
__device__ __forceinline__ void conv_output(const KParams &p, Value value, float vs, const uint32_t *tab, uint32_t *slab,
                                            int rbase, int cbase, int b0, int q0, int lane) {
  const int li = lane & 31, g = lane >> 5;
  if (p.epi == APNN_EPI_INT32) {
    if constexpr (NQ == 4) {
      __syncthreads();  // every wave is done with the operand buffers
      // 16-byte unit u (channels 4u ..) of row r lies at place u ^ (r % 8): no bank is met twice by eight lanes
      i4 *mine = reinterpret_cast<i4 *>(slab) + (threadIdx.x >> 6) * 256;
      const int r8 = lane >> 3, u = lane & 7;
      static_for_e<0, NX * NY>([&](auto xyc) {
        constexpr int x = decltype(xyc)::value / NY, y = decltype(xyc)::value % NY;
        using X = std::integral_constant<int, x>;
        using Y = std::integral_constant<int, y>;
        static_for_e<0, 4>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          const i4 v = {(int)(value(X{}, Y{}, std::integral_constant<int, 4 * q>{}) * vs),
                        (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 1>{}) * vs),
                        (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 2>{}) * vs),
                        (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 3>{}) * vs)};
          mine[li * 8 + ((2 * q + g) ^ (li & 7))] = v;
        });
        // (LDS operations of one wave complete in order)
        const int col = cbase + y * 32 + 4 * u;
        int *dst = reinterpret_cast<int *>(p.out) + (long long)(rbase + x * 32 + r8) * p.rowsB + col;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const i4 v = mine[(8 * k + r8) * 8 + (u ^ r8)];
          if (rbase + x * 32 + 8 * k + r8 < p.rowsA) {
            if (col + 4 <= p.rowsB) {
              *reinterpret_cast<i4u *>(dst + (long long)(8 * k) * p.rowsB) = v;
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (col + j < p.rowsB) dst[(long long)(8 * k) * p.rowsB + j] = v[j];
            }
          }
        }
      });
      return;
    }
    const bool full = cbase + NY * 32 <= p.rowsB;  // same for the whole wave
    static_for_e<0, NX>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      const int row = rbase + x * 32 + li;
      int *dst = reinterpret_cast<int *>(p.out) + (long long)row * p.rowsB + cbase + 8 * q0 + 4 * g;
      if (row < p.rowsA) {
        static_for_e<0, NY * NQ>([&](auto ic) {
          constexpr int y = decltype(ic)::value / NQ, q = decltype(ic)::value % NQ;
          const i4u v = {(int)(value(xc, std::integral_constant<int, y>{}, std::integral_constant<int, 4 * q>{}) * vs),
                         (int)(value(xc, std::integral_constant<int, y>{}, std::integral_constant<int, 4 * q + 1>{}) * vs),
                         (int)(value(xc, std::integral_constant<int, y>{}, std::integral_constant<int, 4 * q + 2>{}) * vs),
                         (int)(value(xc, std::integral_constant<int, y>{}, std::integral_constant<int, 4 * q + 3>{}) * vs)};
          if (full) {
            *reinterpret_cast<i4u *>(dst + y * 32 + 8 * q) = v;
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (cbase + y * 32 + 8 * (q0 + q) + 4 * g + j < p.rowsB) dst[y * 32 + 8 * q + j] = v[j];
          }
        });
      }
    });
    return;
  }

  const int nb = p.out_bits;
  const int w32 = p.rowsB >> 5;
  const bool pooled = p.pool != APNN_POOL_NONE;
  const int nt = (1 << nb) - 1;
  const bool pending = p.resid_planes != nullptr && p.fold == 0u;  // a packed shortcut the matrix cores did not add

  // planes of pixel block x, NW words from channel block y0 on: pool, combine the lane halves, store
  auto finish = [&](int x, int y0, auto &w, bool flips) {
    constexpr int NW = sizeof(w) / sizeof(w[0]), NB = sizeof(w[0]) / sizeof(uint32_t);
    const int row = rbase + x * 32 + li;
    const int word0 = (cbase >> 5) + y0;
#pragma unroll
    for (int y = 0; y < NW; ++y) {
      if (flips && p.flip != nullptr) {
        // flip flags of the share's channels, this half's nibbles in the layout of w
        const uint32_t f = tab[nt * (TB + 4) + ((cbase - b0) >> 5) + y0 + y] >> (8 * (4 - q0 - NQ));
        const uint32_t fs = (g == 0 ? f >> 4 : f) & (0x0f0f0f0fu >> (8 * (4 - NQ)));
#pragma unroll
        for (int b = 0; b < NB; ++b) w[y][b] ^= fs;
      }
      if (pooled) quad_max<NB>(w[y], nb);
    }
    const bool row_ok = row < p.rowsA && (!pooled || (li & 3) == 0);
    const int orow = pooled ? row >> 2 : row;
#pragma unroll
    for (int b = 0; b < NB; b += 2) {
      if (b < nb) {
        uint32_t word[NW];
#pragma unroll
        for (int y = 0; y < NW; ++y) {
          const uint32_t lo = w[y][b], hi = b + 1 < NB ? w[y][b + 1 < NB ? b + 1 : 0] : 0u;
          // lower lane half: plane b + 1, upper half: plane b
          const auto s = __builtin_amdgcn_permlane32_swap(hi, lo, false, false);
          word[y] = (s[0] << 4) | s[1];
        }
        const int plane = b + 1 - g;
        if (plane < nb && row_ok) {
          uint32_t *dst = reinterpret_cast<uint32_t *>(p.out) + plane * p.out_plane + (long long)orow * w32 + word0;
          if constexpr (NQ == 4) {
            if (NW == 4 && word0 + 4 <= w32) {
              const u4u v = {word[0], word[NW > 1 ? 1 : 0], word[NW > 2 ? 2 : 0], word[NW > 3 ? 3 : 0]};
              *reinterpret_cast<u4u *>(dst) = v;
            } else if (NW == 2 && word0 + 2 <= w32) {
              const u2u v = {word[0], word[NW > 1 ? 1 : 0]};
              *reinterpret_cast<u2u *>(dst) = v;
            } else {
#pragma unroll
              for (int y = 0; y < NW; ++y)
                if (word0 + y < w32) dst[y] = word[y];
            }
          } else if (word0 < w32) {
            // a byte or halfword of the word, channel 0 on top
            if constexpr (NQ == 2) reinterpret_cast<uint16_t *>(dst)[1 - (q0 >> 1)] = (uint16_t)word[0];
            if constexpr (NQ == 1) reinterpret_cast<uint8_t *>(dst)[3 - q0] = (uint8_t)word[0];
          }
        }
      }
    }
  };

  if (conv_float_codes(p, MAXB)) {
    auto run = [&](auto nb_c) {
      constexpr int NB = decltype(nb_c)::value;
      uint32_t w[NX][NY][NB];
      static_for_e<0, NY>([&](auto yc) {
        constexpr int y = decltype(yc)::value;
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
          for (int b = 0; b < NB; ++b) w[x][y][b] = 0;
        static_for_e<0, NQ>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          float v[NX][4];
          uint32_t *wp[NX];
          static_for_e<0, NX>([&](auto xc) {
            constexpr int x = decltype(xc)::value;
            static_for_e<0, 4>([&](auto jc) {
              v[x][decltype(jc)::value] = value(xc, yc, std::integral_constant<int, 4 * q + decltype(jc)::value>{});
            });
            if (q > 0) {
#pragma unroll
              for (int b = 0; b < NB; ++b) w[x][y][b] <<= 4;  // the other lane half's nibble
            }
            wp[x] = w[x][y];
          });
          conv_append_quad<NX, NB, TB>(v, tab + cbase - b0 + y * 32 + 8 * (q0 + q) + 4 * g, wp);
        });
      });
#pragma unroll
      for (int x = 0; x < NX; ++x) finish(x, 0, w[x], true);
    };
    if constexpr (MAXB > 2) {
      if (nb == 4) return run(std::integral_constant<int, 4>{});
      if (nb == 3) return run(std::integral_constant<int, 3>{});
    }
    if (nb == 2) run(std::integral_constant<int, 2>{}); else run(std::integral_constant<int, 1>{});
    return;
  }

  // int32 values: low bits, int32 residual maps, saved sums, average pooling, maxima of three- and four-bit codes,
  // values fp32 could round, wider codes.  A block's values pass through 4 KB of LDS per wave, so that one body
  // (per range of code widths) serves all blocks: unrolled over the registers it would dwarf the kernel around it.  Waves
  // of eight blocks, whose registers are full, take half a block at a time.
  // Pooled thresholds: the four lanes of a window hold the same four pooled values, so each searches one of them and
  // the bits meet in an OR over the quad.
  __syncthreads();  // every wave is done with the operand buffers (split K: with the partial sums)
  int *mine = reinterpret_cast<int *>(slab) + (threadIdx.x >> 6) * (64 * 4 * NQ) + lane * 4;
  const bool bn = p.epi == APNN_EPI_BN;
  auto blocks = [&](auto nb_c) {
    constexpr int NB = decltype(nb_c)::value;
    constexpr int QG = NX * NY >= 8 ? 2 : NQ;  // quads at a time
    // first two planes of the shortcut words, one block ahead
    uint32_t ahead[2] = {0, 0};
    auto request = [&](int blk) {
      const int row = min(rbase + (blk / NY) * 32 + li, p.rowsA - 1), word = min((cbase >> 5) + blk % NY, w32 - 1);
      const uint32_t *src = p.resid_planes + (long long)row * w32 + word;
      ahead[0] = src[0];
      if (p.resid_bits > 1) ahead[1] = src[(long long)p.rowsA * w32];
    };
    if (pending) request(0);
#pragma unroll 1
    for (int blk = 0; blk < NX * NY; ++blk) {
      const int x = blk / NY, y = blk - x * NY;
      const int word = (cbase >> 5) + y;
      const uint32_t first[2] = {ahead[0], ahead[1]};
      if (pending && blk + 1 < NX * NY) request(blk + 1);
      if (word >= w32) continue;  // same for the whole wave
      static_for_e<0, NX * NY>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (blk == k) {
          using X = std::integral_constant<int, k / NY>;
          using Y = std::integral_constant<int, k % NY>;
          static_for_e<0, NQ>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const i4 v = {(int)(value(X{}, Y{}, std::integral_constant<int, 4 * q>{}) * vs),
                          (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 1>{}) * vs),
                          (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 2>{}) * vs),
                          (int)(value(X{}, Y{}, std::integral_constant<int, 4 * q + 3>{}) * vs)};
            *reinterpret_cast<i4 *>(mine + q * 256) = v;  // LDS operations of one wave complete in order
          });
        }
      });
      uint32_t w[1][NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) w[0][b] = 0;
#pragma unroll 1
      for (int qb = 0; qb < NQ; qb += QG) {
        i4 v[QG];
#pragma unroll
        for (int q = 0; q < QG; ++q) v[q] = *reinterpret_cast<const i4 *>(mine + (qb + q) * 256);
        const int row = rbase + x * 32 + li;
        const int gcol = cbase + y * 32 + 8 * (q0 + qb) + 4 * g;  // of quad 0
        const long long o = (long long)row * p.rowsB + gcol;
        if (pending) {
          const uint32_t *src = p.resid_planes + (long long)min(row, p.rowsA - 1) * w32 + word;
          for (int b = 0; b < p.resid_bits; ++b) {
            const uint32_t bits = (b == 0 ? first[0] : b == 1 ? first[1] : src[(long long)b * p.rowsA * w32]) << (8 * (q0 + qb) + 4 * g);
            const int part = (int)((uint32_t)p.resid_scale << b);
#pragma unroll
            for (int q = 0; q < QG; ++q)
#pragma unroll
              for (int j = 0; j < 4; ++j) v[q][j] += ((int)(bits << (8 * q + j)) >> 31) & part;
          }
        }
        if (p.resid != nullptr && row < p.rowsA) {
#pragma unroll
          for (int q = 0; q < QG; ++q) v[q] += *reinterpret_cast<const i4u *>(p.resid + o + 8 * q);
        }
        if (p.save_acc != nullptr && row < p.rowsA) {
#pragma unroll
          for (int q = 0; q < QG; ++q) *reinterpret_cast<i4u *>(p.save_acc + o + 8 * q) = v[q];
        }
        if (p.pool == APNN_POOL_AVG2X2) {
#pragma unroll
          for (int q = 0; q < QG; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              int t = v[q][j];
              t += (int)quad_xor1((uint32_t)t);
              t += (int)quad_xor2((uint32_t)t);
              v[q][j] = t / 4;
            }
        }
        auto append = [&](const int (&code)[QG][4]) {
#pragma unroll
          for (int q = 0; q < QG; ++q)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              w[0][b] <<= 4;  // the other lane half's nibble
#pragma unroll
              for (int j = 0; j < 4; ++j) w[0][b] = __builtin_amdgcn_alignbit(w[0][b], (uint32_t)code[q][j] << (31 - b), 31);
            }
        };
        if (!bn) {
          int code[QG][4];
#pragma unroll
          for (int q = 0; q < QG; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) code[q][j] = v[q][j];
          append(code);
        } else {
          const int c0 = gcol - b0;
          if (p.flip != nullptr) {
            uint32_t flips = 0;  // flag of channel j of quad q at bit 31 - 8q - j
            if constexpr (NB <= 4) {
              flips = tab[nt * (TB + 4) + (c0 >> 5)] << (c0 & 31);
            } else {
#pragma unroll
              for (int q = 0; q < QG; ++q)
#pragma unroll
                for (int j = 0; j < 4; ++j) flips |= (p.flip[gcol + 8 * q + j] ? 0x80000000u : 0u) >> (8 * q + j);
            }
#pragma unroll
            for (int q = 0; q < QG; ++q)
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const int m = (int)(flips << (8 * q + j)) >> 31;
                v[q][j] = (int)(((uint32_t)v[q][j] ^ (uint32_t)m) - (uint32_t)m);
              }
          }
          // codes of N values each, of channels c0 + 8q + at(j)
          auto search = [&](auto &code, const auto &s, int shift) {
            constexpr int N = sizeof(s[0]) / sizeof(int);
            const int *thr = NB <= 4 ? reinterpret_cast<const int *>(tab) + c0 + shift : p.thr + (long long)(gcol + shift) * nt;
            const int pitch = NB <= 4 ? 1 : nt;  // of a channel
#pragma unroll
            for (int q = 0; q < QG; ++q)
#pragma unroll
              for (int j = 0; j < N; ++j) code[q][j] = 0;
            for (int h = (nt + 1) >> 1; h > 0; h >>= 1) {
              int t[QG][N];  // all reads of a level before its first compare
#pragma unroll
              for (int q = 0; q < QG; ++q)
#pragma unroll
                for (int j = 0; j < N; ++j) t[q][j] = thr[(8 * q + j) * pitch + (code[q][j] + h - 1) * (NB <= 4 ? TB + 4 : 1)];
#pragma unroll
              for (int q = 0; q < QG; ++q)
#pragma unroll
                for (int j = 0; j < N; ++j) code[q][j] += s[q][j] >= t[q][j] ? h : 0;
            }
          };
          if (pooled) {
            const int l = li & 3;
            int s[QG][1], code[QG][1];
#pragma unroll
            for (int q = 0; q < QG; ++q) {
              if (p.pool == APNN_POOL_MAX2X2) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  int t = v[q][j];
                  t = max(t, (int)quad_xor1((uint32_t)t));
                  v[q][j] = max(t, (int)quad_xor2((uint32_t)t));
                }
              }
              s[q][0] = l < 2 ? (l == 0 ? v[q][0] : v[q][1]) : (l == 2 ? v[q][2] : v[q][3]);
            }
            search(code, s, l);
#pragma unroll
            for (int q = 0; q < QG; ++q) {
              uint32_t m = 0;  // plane b: nibble b, channel 0 on top
#pragma unroll
              for (int b = 0; b < NB; ++b) m |= (((uint32_t)code[q][0] >> b) & 1u) << (4 * b);
              m <<= 3 - l;
              m |= quad_xor1(m);
              m |= quad_xor2(m);
#pragma unroll
              for (int b = 0; b < NB; ++b) w[0][b] = (w[0][b] << 8) | ((m >> (4 * b)) & 15u);
            }
          } else {
            int s[QG][4], code[QG][4];
#pragma unroll
            for (int q = 0; q < QG; ++q)
#pragma unroll
              for (int j = 0; j < 4; ++j) s[q][j] = v[q][j];
            search(code, s, 0);
            append(code);
          }
        }
      }
      finish(x, y, w, false);
    }
  };
  if (nb <= 2) blocks(std::integral_constant<int, 2>{});
  else if (nb <= 4) blocks(std::integral_constant<int, 4>{});
  else blocks(std::integral_constant<int, 8>{});
}

}  // namespace apnn
