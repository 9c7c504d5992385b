// Large tiles on FP4 / FP6 operands (GEMM entry points 256x128; convolution 128x256 and 128x128): arithmetic and output
// stages of mfma_kernel.h and conv_epilogue.h, another operand supply.
//
// What bounds it.  One 32x32x64 matrix instruction takes 32 clocks of a SIMD; measured with register-only loops, two
// waves per SIMD hide up to six vector operations behind each (33 clocks per instruction), seven cost 36, eight 39,
// and a wave alone pays eight clocks for every vector operation beyond four.  The vector operations per matrix
// instruction are therefore what counts, and everything that is not expansion leaves the loop:
//   - packed words go from global memory to LDS without passing registers (buffer_load ... lds, 16 bytes per lane),
//     one chunk ahead of the products; a row's offset is computed once, the chunk is the scalar offset;
//   - a lane reads four k-steps of a row with one 128-bit LDS read.  K is cut into groups of eight words, the lower
//     lane half takes the first four, the upper the last four, for both operands alike (a permutation of the terms
//     of each dot product);
//   - symmetric one-plane weights are -1 / +1 operands and unsigned ones need no correction, so nothing is counted
//     (wider symmetric weights: activation sums, as in mfma_kernel.h);
//   - the last k-step of a chunk carries the barrier, and expands the first operands of the next chunk.
// w1a2: 6.1 vector operations per matrix instruction in the loop instead of 6.75 plus staging, 212 registers.  8192^3 w1a2
// 226 -> 220 us, 206 to 210 in graph replay (212 with LDS rows permuted for 32 banks).  Of its busy clocks there: matrix pipes 69 %,
// vector pipes 68 %, waves waiting 13 % of their lifetime, 1.89 GHz.  Over 1024 to 16384 bits the time is a line of 22.1 us per
// 1024 bits, 21.6 ns a matrix instruction and SIMD (17.8 in a loop of such instructions with six vector operations and nothing
// else, 13.3 by the clock), and 37 us beside it, in which the 268 MB of results leave.  4096^3 w1a4 58.2 -> 45.2 us (48.0 with FP6
// digits alone), over 8192 bits 81.6 (83 with the other order): 8.4 us per 1024 bits, 33 ns a matrix instruction, vector pipes
// 57 % busy, and 15 us beside it for 67 MB of results.  What holds the loops up beyond the expansion is not known.
// Convolution: a load's lane decodes the tap of its 16 bytes once per chunk; padding pixels are disabled loads, which
// write zeros.  Two tiles of 128x256 per compute unit, three of 128x128.  3x3 convolutions at batch
// 64: 56x56x256 76 -> 66 us, 28x28x512 78 -> 64, 14x14x512 28 -> 23 (bounded by vector work, 9.8 operations per matrix
// instruction with the output stage, and by the last round: 784 tiles of 128x256 on 512 places); the VGG variant at
// batch 64 541 -> 489 us.
//
// LDS rows are KC words (64 or 32 bytes) without padding, as the loads fill them in lane order; the 16-byte units of a
// row are permuted by its index so that any sixteen consecutive rows read from the sixteen groups of four banks (64 banks: a
// 16-byte read takes 2.7 ns of a unit's LDS, 3.7 with eight rows in eight groups).
#pragma once
#include "mfma_kernel.h"

namespace apnn {

typedef int rsrc4 __attribute__((ext_vector_type(4)));

// words per row and chunk: the addresses a load may write (both buffers) stay below 64 KiB
constexpr int async_chunk_words(int PA, int PB, int TA, int TB) {
  return 2 * (PA * TA + PB * TB) * 16 * 4 <= 64 * 1024 ? 16 : 8;
}

template <int PA, int PB, int FA, int FB, int WA, int WB, bool CONV, bool SYM, int OCC>
__global__ __launch_bounds__(256, OCC) void apnn_async_kernel(const KParams pk) {
  KParams p = pk;
  int bid = blockIdx.x;
  if (CONV && pk.pair_tiles > 0 && bid >= pk.pair_tiles) {  // paired launch, see apnn_mfma_kernel
    bid -= pk.pair_tiles;
    p.B = pk.B2;
    p.KW = pk.KW2;
    p.S = pk.S2;
    p.pad = pk.pad2;
    p.magicS = pk.magicS2;
    p.magicS16 = pk.magicS16_2;
    p.planeB = pk.planeB2;
    p.thr = pk.thr2;
    p.flip = pk.flip2;
    p.out = pk.out2;
  }
  static_assert(WA * WB == 4, "four waves tile the output");
  constexpr int DIG = digit_planes(PA, PB);
  constexpr int DA = (PA + DIG - 1) / DIG, DB = (PB + DIG - 1) / DIG;
  constexpr int PW = CONV ? PB : PA;     // planes of the weights, of the activations
  constexpr int PX = CONV ? PA : PB;
  constexpr bool SIGN = SYM && PW == 1;  // -1 / +1 operands: the accumulator is the result
  constexpr bool SUM = SYM && PW > 1;    // activation sums enter the result
  constexpr int FSC = SIGN ? (DIG == 4 ? 8 : 2) : fp_scale(PA, PB);
  if (!SUM) p.sym = 0;
  constexpr int TA = WA * FA * 32, TB = WB * FB * 32;
  constexpr int KC = async_chunk_words(PA, PB, TA, TB);
  constexpr int UPR = KC / 4, RPI = 64 / UPR;  // 16-byte units per row of a chunk, rows per load instruction
  constexpr int NG = KC / 8;                   // groups of four k-steps
  constexpr int RA = TA / RPI, RB = TB / RPI;  // row groups
  static_assert(RA % 4 == 0 && RB % 4 == 0, "row groups go round the four waves");
  constexpr int NA = RA / 4, NB = RB / 4;
  constexpr int BUF = (PA * TA + PB * TB) * KC;  // words
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int wa = wave / WB, wb = wave % WB;

  const int tilesB = (p.rowsB + TB - 1) / TB;
  int trow = bid / tilesB, tcol = bid % tilesB;
  if (p.xcd_rows > 0) {
    const int tilesA = (p.rowsA + TA - 1) / TA;
    const int per_xcd = (tilesA * tilesB) >> 3;
    const int lin = (bid & 7) * per_xcd + (bid >> 3);
    const int per_band = p.xcd_rows * tilesB;
    const int band = lin / per_band, w = lin - band * per_band;
    const int rows_in_band = min(p.xcd_rows, tilesA - band * p.xcd_rows);
    tcol = w / rows_in_band;
    trow = band * p.xcd_rows + (w - tcol * rows_in_band);
  }
  const int a0 = trow * TA, b0 = tcol * TB;

  auto resource = [](const uint32_t *base, long long words) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(base);
    return rsrc4{(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffffu), (int)(uint32_t)(words * 4), 0x00020000};
  };
  rsrc4 rsA[PA], rsB[PB];
#pragma unroll
  for (int pl = 0; pl < PA; ++pl) rsA[pl] = resource(p.A + pl * p.planeA, p.planeA);
#pragma unroll
  for (int pl = 0; pl < PB; ++pl) rsB[pl] = resource(p.B + pl * p.planeB, p.planeB);

  // lane l of a load instruction fills the 16 bytes at 16 * l of a row group: row l / UPR, unit place l % UPR
  const int lrow = lane / UPR;
  const int unit = (lane % UPR) ^ (UPR == 4 ? (lrow >> 2) & 3 : (lrow >> 3) & 1);
  uint32_t voA[NA], voB[NB];  // byte offset of the row's unit (convolution: word offset of the pixel's tap (0, 0), mod 2^32)
  int y0[NA], x0[NA];
#pragma unroll
  for (int n = 0; n < NA; ++n) {
    const int row = a0 + (wave + 4 * n) * RPI + lrow;
    y0[n] = x0[n] = 0;
    if constexpr (CONV) {
      int b = 0;
      pixel_origin(p, row, b, y0[n], x0[n]);
      voA[n] = (((uint32_t)b * (uint32_t)p.Hs + (uint32_t)y0[n]) * (uint32_t)p.Ws + (uint32_t)x0[n]) * (uint32_t)p.C32;
      if (row >= p.rowsA) y0[n] = 1 << 30;  // no tap of it lies in the image
    } else
    voA[n] = row < p.rowsA ? ((uint32_t)row * (uint32_t)p.KW + 4u * unit) * 4u : 0xffffffffu;
  }
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int row = b0 + (wave + 4 * n) * RPI + lrow;
    voB[n] = row < p.rowsB ? ((uint32_t)row * (uint32_t)p.KW + 4u * unit) * 4u : 0xffffffffu;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)smem;
  // (m0 holds the LDS address)
  auto load_lds = [](uint32_t lds, uint32_t voff, rsrc4 rs, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rs), "s"(soff)
                 : "memory", "m0");
  };
  auto fetch = [&](int ch, int buf) {
    const bool ok = ch * KC + 4 * unit < p.KW;
    const uint32_t soff = (uint32_t)(ch * KC * 4);
    const uint32_t base = lds0 + (uint32_t)(buf * BUF * 4);
    uint32_t r = 0, sx = 0, toff = 0;
    if constexpr (CONV) {  // a unit of four words lies within one tap
      const uint32_t kw0 = (uint32_t)(ch * KC + 4 * unit);
      const uint32_t tap = p.c32_shift >= 0 ? kw0 >> p.c32_shift : fast_div(kw0, (uint32_t)p.C32, p.magicC32);
      r = __umul24(tap, p.magicS16) >> 16;
      sx = tap - __umul24(r, (uint32_t)p.S);
      toff = __umul24(__umul24(r, (uint32_t)p.Ws) + sx, (uint32_t)p.C32) + kw0 - __umul24(tap, (uint32_t)p.C32);
    }
#pragma unroll
    for (int n = 0; n < NA; ++n) {
      uint32_t vo;
      if constexpr (CONV) {
        const bool in = ok && (uint32_t)(y0[n] + (int)r) < (uint32_t)p.Hs && (uint32_t)(x0[n] + (int)sx) < (uint32_t)p.Ws;
        vo = in ? (voA[n] + toff) << 2 : 0xffffffffu;
      } else {
        vo = ok ? voA[n] : 0xffffffffu;
      }
#pragma unroll
      for (int pl = 0; pl < PA; ++pl)
        load_lds(base + (uint32_t)((pl * TA + (wave + 4 * n) * RPI) * KC * 4), vo, rsA[pl], CONV ? 0u : soff);
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const uint32_t vo = ok ? voB[n] : 0xffffffffu;
#pragma unroll
      for (int pl = 0; pl < PB; ++pl)
        load_lds(base + (uint32_t)((PA * TA + pl * TB + (wave + 4 * n) * RPI) * KC * 4), vo, rsB[pl], soff);
    }
  };
  // the loads above are invisible to the compiler's wait counts; a disabled one writes zeros
  auto arrive = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  const int nchunks = (p.KW + KC - 1) / KC;
  // convolution: value per accumulator unit, thresholds of the tile's channels behind the operand buffers
  constexpr int log2vs = __builtin_ctz(FSC) + (SUM ? 1 : 0);
  const float inv_vs = 1.0f / (float)(1 << log2vs);
  uint32_t *tab = smem + 2 * BUF;
  constexpr int MAXB = PA >= 3 ? 4 : 2;
  ConvTable<TB, PA >= 3 ? 15 : 3, MAXB> table;
  if constexpr (CONV) table.load(p, b0);
  fetch(0, 0);
  const int rbase = a0 + wa * FA * 32, cbase = b0 + wb * FB * 32;
  constexpr bool LAZY = FA * FB >= 8;
  uint32_t sc[FA][FB][2];
  if constexpr (CONV) {
    if (p.fold != 0u && !LAZY) conv_shortcut_load<FA, FB>(p, rbase, cbase, li, sc);
    table.store(p, b0, tab, inv_vs);
  }

  v16f acc[FA][FB];
#pragma unroll
  for (int x = 0; x < FA; ++x)
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0;
  constexpr int FX = CONV ? FA : FB;
  int psum[FX][PX];  // activation sums (SUM)
#pragma unroll
  for (int y = 0; y < FX; ++y)
#pragma unroll
    for (int pl = 0; pl < PX; ++pl) psum[y][pl] = 0;

  // four k-steps of words of this lane's rows (lower lane half: the first four words of a group, upper: the last four)
  uint4 qA[FA][PA], qB[FB][PB];
  const int rowA = wa * FA * 32 + li, rowB = wb * FB * 32 + li;
  const int swz = UPR == 4 ? (li >> 2) & 3 : (li >> 3) & 1;
  auto read_group = [&](const uint32_t *buf, auto jc) {
    constexpr int j = decltype(jc)::value;
    const int place = ((2 * j + g) ^ swz) * 4;
#pragma unroll
    for (int x = 0; x < FA; ++x)
#pragma unroll
      for (int pl = 0; pl < PA; ++pl)
        qA[x][pl] = *reinterpret_cast<const uint4 *>(buf + (pl * TA + rowA + x * 32) * KC + place);
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int pl = 0; pl < PB; ++pl)
        qB[y][pl] = *reinterpret_cast<const uint4 *>(buf + (PA * TA + pl * TB + rowB + y * 32) * KC + place);
  };
  v8i af[FA][DA], bf[FB][DB];
  auto word = [](const uint4 &q, auto ic) -> uint32_t {
    constexpr int i = decltype(ic)::value;
    return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w;
  };
  auto expand_into = [&](auto ic, v8i (&a)[FA][DA], v8i (&b)[FB][DB]) {
#pragma unroll
    for (int x = 0; x < FA; ++x) {
      uint32_t w[PA];
#pragma unroll
      for (int pl = 0; pl < PA; ++pl) {
        w[pl] = word(qA[x][pl], ic);
        if constexpr (CONV && SUM) psum[x][pl] += __popc(w[pl]);
      }
      if constexpr (!CONV && SIGN) {
        a[x][0] = expand_sign<DIG>(w[0]);
      } else {
        static_for<0, DA>([&](auto dc) { a[x][decltype(dc)::value] = expand_digit<DIG, PA, decltype(dc)::value>(w); });
      }
    }
#pragma unroll
    for (int y = 0; y < FB; ++y) {
      uint32_t w[PB];
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) {
        w[pl] = word(qB[y][pl], ic);
        if constexpr (!CONV && SUM) psum[y][pl] += __popc(w[pl]);
      }
      if constexpr (CONV && SIGN) {
        b[y][0] = expand_sign<DIG>(w[0]);
      } else {
        static_for<0, DB>([&](auto dc) { b[y][decltype(dc)::value] = expand_digit<DIG, PB, decltype(dc)::value>(w); });
      }
    }
  };
  auto mfma_all = [&]() {
#pragma unroll
    for (int x = 0; x < FA; ++x)
#pragma unroll
      for (int y = 0; y < FB; ++y)
        static_for<0, DA>([&](auto dac) {
          static_for<0, DB>([&](auto dbc) {
            constexpr int da = decltype(dac)::value, db = decltype(dbc)::value;
            if constexpr (CONV) {
              acc[x][y] = mfma_digits<DIG, da + db>(bf[y][db], af[x][da], acc[x][y]);
            } else {
              acc[x][y] = mfma_digits<DIG, da + db>(af[x][da], bf[y][db], acc[x][y]);
            }
          });
        });
  };
  constexpr int N_MFMA = FA * FB * DA * DB;
  constexpr int XDIG[5] = {0, 7, 10, 18, 22};
  constexpr int XA = XDIG[DIG] * (PA / DIG) + XDIG[PA % DIG], XB = XDIG[DIG] * (PB / DIG) + XDIG[PB % DIG];
  constexpr int N_VALU = FA * XA + FB * XB + (SUM ? FX * PX : 0);
  constexpr int VALU_PER_MFMA = (N_VALU + N_MFMA - 1) / N_MFMA;
  // matrix products of one k-step and, between them, the expansion of the next
  auto step = [&](auto ic) {
    v8i an[FA][DA], bn[FB][DB];
    mfma_all();
    expand_into(ic, an, bn);
#pragma unroll
    for (int x = 0; x < FA; ++x)
#pragma unroll
      for (int d = 0; d < DA; ++d) af[x][d] = an[x][d];
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int d = 0; d < DB; ++d) bf[y][d] = bn[y][d];
#pragma unroll
    for (int i = 0; i < N_MFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VALU_PER_MFMA, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  arrive();
  if (nchunks > 1) fetch(1, 1);
  read_group(smem, I0{});
  expand_into(I0{}, af, bf);
#pragma unroll 1
  for (int ch = 0; ch < nchunks; ++ch) {
    const uint32_t *cur = smem + (ch & 1) * BUF;
    step(I1{});
    step(I2{});
    step(I3{});
    if constexpr (NG == 2) {
      if (ch * KC + 8 < p.KW) {
        read_group(cur, I1{});
        step(I0{});
        step(I1{});
        step(I2{});
        step(I3{});
      }
    }
    // every wave holds its last words of this chunk in registers, the next chunk has arrived (after the last chunk the
    // words read here are stale: their operands meet no product, their sums are taken back below)
    if (ch + 1 < nchunks) {
      arrive();
      if (ch + 2 < nchunks) fetch(ch + 2, ch & 1);
    }
    read_group(smem + ((ch + 1) & 1) * BUF, I0{});
    step(I0{});
  }
  int ssum[FX];
#pragma unroll
  for (int y = 0; y < FX; ++y) {
    int t = 0;
    if constexpr (SUM) {
#pragma unroll
      for (int pl = 0; pl < PX; ++pl) t += (psum[y][pl] - __popc((CONV ? qA[CONV ? y : 0][CONV ? pl : 0] : qB[CONV ? 0 : y][CONV ? 0 : pl]).x)) << pl;
      t += __shfl_xor(t, 32, 64);
    }
    ssum[y] = t;
  }
  if constexpr (CONV) {
    if (p.fold != 0u) {
      if (LAZY) conv_shortcut_load<FA, FB>(p, rbase, cbase, li, sc);
      fold_shortcut_lanes<FA, FB>(p, acc, sc, lane, log2vs);
    }
    if constexpr (SUM) {
#pragma unroll
      for (int x = 0; x < FA; ++x) {
        const float c = (float)ssum[x] * (-(float)p.wmax * inv_vs);
#pragma unroll
        for (int y = 0; y < FB; ++y)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[x][y][r] += c;
      }
    }
    settle_results(acc);
    conv_output<FA, FB, 4, TB, MAXB>(
        p, [&](auto xc, auto yc, auto ic) { return (float)acc[decltype(xc)::value][decltype(yc)::value][decltype(ic)::value]; },
        (float)(1 << log2vs), tab, smem, rbase, cbase, b0, 0, lane);
  } else {
    EpiOperands<FA, FB> eo;
    epi_prefetch<1, PB >= 3 ? 4 : 2, true>(p, rbase, cbase, lane, eo);
    epi_finish<FSC, 1, false, PB >= 3 ? 4 : 2, true>(p, acc, ssum, smem, wave, lane, a0, b0, wa, wb, eo);
  }
}

template <int PA, int PB, int FA, int FB, int WA, int WB, bool CONV, int OCC>
inline hipError_t launch_async(const KParams &p, hipStream_t stream) {
  constexpr int TA = WA * FA * 32, TB = WB * FB * 32;
  constexpr int KC = async_chunk_words(PA, PB, TA, TB);
  constexpr size_t slab = CONV ? 0 : 4ull * (32 * (FB * 32 + 1) + 32 + FB * 32 + 2 * 32 * FB) * sizeof(int);
  constexpr size_t stage = 2ull * (PA * TA + PB * TB) * KC * sizeof(uint32_t);
  constexpr size_t bytes = stage > slab ? stage : slab;
  static_assert(stage <= 64 * 1024, "LDS addresses of the loads fit 16 bits");
  constexpr size_t most = bytes + (CONV ? (conv_table_words(4, TB) + 4) * 4 : 0);
  static_assert(most <= 160 * 1024, "LDS of a compute unit");
  auto kern = p.sym ? apnn_async_kernel<PA, PB, FA, FB, WA, WB, CONV, true, OCC> : apnn_async_kernel<PA, PB, FA, FB, WA, WB, CONV, false, OCC>;
  if (most > 64 * 1024) {
    static std::atomic<unsigned long long> raised[2];
    const hipError_t e = raise_lds_limit(raised[p.sym != 0], reinterpret_cast<const void *>(kern), most);
    if (e != hipSuccess) return e;
  }
  const long long tilesB = (p.rowsB + TB - 1) / TB, tiles = (long long)((p.rowsA + TA - 1) / TA) * tilesB;
  KParams q = p;
  if (p.pair_tiles != 0) q.pair_tiles = (int)tiles;
  q.xcd_rows = (p.pair_tiles == 0 && tiles % 8 == 0 && tiles >= kXcdOrderMinTiles && tilesB >= 2) ? 8 : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)(q.pair_tiles != 0 ? 2 * tiles : tiles)), dim3(256),
                     bytes + (CONV ? conv_epilogue_bytes(p, TB) : 0), stream, q);
  return hipGetLastError();
}

}  // namespace apnn
