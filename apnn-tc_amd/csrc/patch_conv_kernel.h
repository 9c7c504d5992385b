// Patch-resident convolution on the matrix cores (FP4 operands, see mfma_kernel.h for the encoding).
//
// The implicit-GEMM kernels gather, for every filter tap, the packed activation words of every output pixel of
// their tile and expand them to matrix-core operands in registers -- R*S times per input pixel and once more per
// column tile.  Here the input pixels a tile needs are expanded ONCE into LDS and every tap reads them in place:
//
//   * In the zero-padded frame (stored frame plus `pad` pixels on every side, PHs x PWs per image) the
//     input pixel of output pixel (b, oy, ox) and tap (r, s) has the linear index
//         q = (b*PHs + oy*stride)*PWs + ox*stride  +  r*PWs + s,
//     i.e. a per-pixel base plus a per-tap constant.  A tile of consecutive output pixels therefore
//     needs one contiguous range [q_lo, q_hi] of padded-frame pixels: the patch.
//   * Per chunk of 64 channels the work-group stages the patch (bit-plane words -> FP4 digit
//     operands, 16 bytes per pixel, 32-channel word and digit; padding pixels are zeros) and the
//     filter block of its output channels for all taps (same encoding), then runs
//     taps k-steps of pure LDS reads + MFMA: first operand = filter[tap][channel], second = patch[base(pixel) + tap
//     offset].  The packed words of the next chunk are requested before the k-steps of this one.
//   * One-plane weights are -1 / +1 or 0 / 1 operands (expand_w1) and need no correction.  With two planes, symmetric:
//     per-pixel activation sums are taken once per patch pixel while staging; a pixel's window sum is the sum over taps.
//
// The accumulator holds pixels in the lanes and channels in the registers; the output stage is conv_output.
//
// What bounds it.  With pixels in the registers and channels in the lanes, activation sums for one-plane weights and
// a filter address per word, vector issue did: 62 vector operations per matrix instruction on 56x56x64.  What they became:
// the lane-local output stage, -1 / +1 weights (no sums), filter words at a constant stride from one offset per thread, tap
// loops unrolled for 3x3 (addresses are immediates), operands of a tap read behind the products of the one before.  Then
// residency: the staging of one work-group hides behind the products of others, so registers are cut for four
// work-groups per compute unit (three where a wave has four blocks; what spills is the general output path alone).
// us before -> without and with the cut, w1a2 with threshold codes in graph replay: 56x56x64 to 64 at batch 64 14.6 -> 11.6 ->
// 10.6; 56x56x96 to 256 at batch 64 68.9 -> 53.6 -> 40.0 (256x64 tiles); w1a4 there 169 -> 90.  Left: no pipe is full.  Of the
// busy clocks, matrix / vector / LDS: 56x56x64 16 / 46 / 30 %, 56x56x96 to 256 33 / 51 / 32, 14x14x832 to 512 on 256x64 tiles
// 33 / 19 / 32, waves waiting 35-46 % of their time (profiles/patch_conv_w1a2_counters.md): staging and products of a work-group
// alternate behind two barriers a chunk, and one and a half to four work-groups on a unit cover that in part.  Long reductions
// stay level with async_kernel.h (56x56x256 at batch 64 59 against 61 us).  A 256x128 tile of 4x2 blocks reads less, but two of
// them per unit leave their last round emptier: 62 us there, 68 against 60 on 28x28x512.
// 5x5 filters in a form of their own, all filter words of a chunk in flight at once: 28x28x64 to 192 at batch 64 21.2 us in
// the general form, 16.4 in this one (two work-groups per unit, by the LDS).
#pragma once
#include "mfma_kernel.h"
#include "quotient.h"

namespace apnn {

// What is known of the filter when the kernel is built.  One kernel for all, with the forms on branches, joins the
// accumulators of both tap loops by copies and the loads of both widths by waits (56x56x64 at batch 64 13.6 -> 12.4 us,
// 56x56x256 81 -> 75, on 256x64 tiles before the cut).
//   PF_ANY        any filter, any number of channel words: a loop over the taps
//   PF_3x3_ODD    3x3, an odd number of channel words: 32-bit loads
//   PF_3x3_PAIRS  3x3, an even number of channel words: 64-bit loads
//   PF_5x5_PAIRS  5x5, an even number of channel words
enum PatchForm { PF_ANY = 0, PF_3x3_ODD = 1, PF_3x3_PAIRS = 2, PF_5x5_PAIRS = 3 };
constexpr int patch_form_side(int form) { return form == PF_ANY ? 0 : form == PF_5x5_PAIRS ? 5 : 3; }

// Work-groups per compute unit that the registers are cut for, by the 32x32 blocks of a wave, the form and the activation planes.
// The 5x5 form stages 50 KB of filter: LDS holds two work-groups, and a cut to 128 registers made it reload up to 12 in every
// chunk.  28x28x64 to 192 at batch 8 / 64, us with four work-groups and with two: w1a4 9.9 -> 9.3 / 30.2 -> 28.4, w1a3 8.1 ->
// 7.7 / 24.1 -> 23.0.  2x2 blocks of the 3x3 forms with four planes reloaded 8 to 16: 256x64 tiles on 56x56x96 to 256 at batch
// 64 108 -> 95 with two work-groups instead of three, 14x14x960 to 1024 185 -> 124.  The general form with four planes still
// reloads 8 to 18 a chunk: three work-groups without them are ahead where the filter fills the LDS (16 taps, 27x27x96 to 256 at
// batch 16 18.6 -> 16.8; 25 taps 72.9 -> 67.1) and behind where it does not (2x2 at batch 32 17.9 -> 20.4).
constexpr int patch_occupancy(int blocks, int form, int planes) {
  if (form == PF_5x5_PAIRS || (blocks == 4 && planes == 4 && form != PF_ANY)) return 2;
  return blocks == 4 ? 3 : 4;
}

constexpr int PATCH_NPT = 4;  // patch pixels per thread (patch capacity = 4 * 256 pixels)

// SHORT: maps of at most 65536 rows and columns (quotient.h); others have PF_ANY alone.  With shifts for all 56x56x64 to 64 at
// batch 64 took 10.7 us instead of 10.4, 56x56x96 to 256 w2a2 44.5 instead of 42.6.
template <int PA, int PB, int FA, int FB, int WA, int WB, int FORM, bool SHORT>
__global__ __launch_bounds__(256, patch_occupancy(FA * FB, FORM, PA)) void apnn_patch_conv_kernel(const KParams p) {
  static_assert(WA * WB == 4, "four waves tile the output");
  constexpr int DA = (PA + 1) / 2, DB = (PB + 1) / 2;
  constexpr int NT = 256;
  constexpr int TA = WA * FA * 32, TB = WB * FB * 32;
  static_assert(NT % TB == 0, "a thread stages the filter words of one channel");
  constexpr int MAXB = PA >= 3 ? 4 : 2;
  constexpr bool ONE = PB == 1;  // -1 / +1 or 0 / 1 operands: the accumulator is the result

  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int wa = wave / WB, wb = wave % WB;
  const int tilesB = (p.rowsB + TB - 1) / TB;
  const int a0 = (blockIdx.x / tilesB) * TA;
  const int b0 = (blockIdx.x % tilesB) * TB;
  constexpr int SIDE = patch_form_side(FORM), TAPS = SIDE * SIDE;  // 0: not known
  const int taps = FORM != PF_ANY ? TAPS : p.KW / p.C32;
  const int cap = p.patch_cap;

  uint32_t *patchA = smem;                                 // [DA][2 words][cap][4 dwords]
  uint32_t *filtB = patchA + DA * cap * 8;                 // [DB][2 words][taps][TB][4 dwords]
  int *pixsum = reinterpret_cast<int *>(filtB + DB * taps * TB * 8);  // [cap], two weight planes only
  uint32_t *tab = smem + patch_stage_words(PA, PB, TB, taps, cap);    // thresholds of the tile's channels
  const bool need_sum = !ONE && p.sym != 0;
  const int log2vs = ONE ? 1 : need_sum ? 3 : 2;  // value per accumulator unit
  const float inv_vs = ONE ? 0.5f : need_sum ? 0.125f : 0.25f;

  ConvTable<TB, PA >= 3 ? 15 : 3, MAXB> table;
  table.load(p, b0);

  // ---- tile geometry.  Only the tile's first row is decoded with full divisions (uniform); every
  // other row and patch pixel is a small offset from it, decoded with the quotients of quotient.h ----------------
  const int last_row = min(a0 + TA, p.rowsA) - 1;
  const int R = FORM != PF_ANY ? SIDE : taps / p.S;
  const bool pooled = p.pool_order != 0;
  const int gw = pooled ? p.Wo >> 1 : p.Wo, gh = pooled ? p.Ho >> 1 : p.Ho;  // row grid (windows when pooling)
  const int gst = pooled ? 2 * p.stride : p.stride;                          // its step in the padded frame
  const uint32_t u0 = (uint32_t)(pooled ? a0 >> 2 : a0);
  const uint32_t t0 = u0 / (uint32_t)gw;
  const int gx0 = (int)(u0 - t0 * (uint32_t)gw);
  const int b0i = (int)(t0 / (uint32_t)gh);
  const int gy0 = (int)(t0 - (uint32_t)b0i * (uint32_t)gh);
  // padded-frame base index of tile row k (k >= 0, relative to a0), relative to the frame origin of image b0i
  auto row_base = [&](int k) {
    const int u = pooled ? k >> 2 : k, sub = pooled ? k & 3 : 0;
    int gx = gx0 + u;
    const int cy = (int)quotient<SHORT>((uint32_t)gx, (uint32_t)gw, p.magicGW);
    gx -= cy * gw;
    int gy = gy0 + cy;
    const int cb = (int)quotient<SHORT>((uint32_t)gy, (uint32_t)gh, p.magicGH);
    gy -= cb * gh;
    return (cb * p.PHs + gy * gst + (sub >> 1) * p.stride) * p.PWs + gx * gst + (sub & 1) * p.stride;
  };
  const int q_lo = row_base(0);  // == (gy0*gst)*PWs + gx0*gst
  const int q_hi = row_base(last_row - a0) + (R - 1) * p.PWs + (p.S - 1);
  const int npp = q_hi - q_lo + 1;
  if (npp > cap) {
    // The host sizes the patch for the worst tile, so this is never taken; if it ever were, the tile
    // stays unwritten and the device error word says so instead of the launch looking successful.
    if (tid == 0 && p.err != nullptr) atomicOr(p.err, (int)KERR_PATCH_CAPACITY);
    return;
  }

  // this lane's pixels: LDS word of pixel li of each of its FA blocks
  int prow[FA];
#pragma unroll
  for (int x = 0; x < FA; ++x) prow[x] = row_base(min((wa * FA + x) * 32 + li, last_row - a0)) - q_lo;

  // Global loads go through one buffer descriptor per operand plane (base, size in bytes; the host launches
  // this kernel only for planes below 4 GiB): a load whose offset lies past the descriptor's size returns
  // zeros, so padding pixels, rows past the end and the unused tail of a task batch are the same instruction
  // with the offset 0xffffffff instead of a branch around the load.
  constexpr uint32_t kOff = 0xffffffffu;
  __amdgpu_buffer_rsrc_t rsrcA[PA], rsrcB[PB];
#pragma unroll
  for (int pl = 0; pl < PA; ++pl)
    rsrcA[pl] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p.A + pl * p.planeA), 0,
                                                  (int)(uint32_t)(p.planeA * 4), 0x00020000);
#pragma unroll
  for (int pl = 0; pl < PB; ++pl)
    rsrcB[pl] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p.B + pl * p.planeB), 0,
                                                  (int)(uint32_t)(p.planeB * 4), 0x00020000);
  // word pair at byte offset boff + soff (boff kOff: zeros); without 64-bit loads (odd number of channel words) the
  // second word of the last pair does not exist
  auto load_pair = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t boff, uint32_t soff, auto pair_c, bool second, uint32_t &w0,
                       uint32_t &w1) {
    if constexpr (decltype(pair_c)::value) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)boff, (int)soff, 0);
      w0 = v[0], w1 = v[1];
    } else {
      w0 = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)boff, (int)soff, 0);
      w1 = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(second && boff != kOff ? boff + 4 : kOff), (int)soff, 0);
    }
  };

  // patch pixels this thread stages: byte offset of the pixel (channel word 0) in a plane, or kOff for
  // padding / beyond the range
  uint32_t poff[PATCH_NPT];
  const int pad_v = (p.PHs - p.Hs) >> 1;
  const int yp0 = gy0 * gst, xp0 = gx0 * gst;
#pragma unroll
  for (int j = 0; j < PATCH_NPT; ++j) {
    const int q = tid + j * NT;
    poff[j] = kOff;
    if (j * NT < npp && q < npp) {
      int xp = xp0 + q;
      const int cy = (int)quotient<SHORT>((uint32_t)xp, (uint32_t)p.PWs, p.magicPW);
      xp -= cy * p.PWs;
      int yp = yp0 + cy;
      const int ci = (int)quotient<SHORT>((uint32_t)yp, (uint32_t)p.PHs, p.magicPH);
      yp -= ci * p.PHs;
      const int img = b0i + ci;
      const int iy = yp - pad_v, ix = xp - pad_v;
      if (img < p.batch && iy >= 0 && iy < p.Hs && ix >= 0 && ix < p.Ws)
        poff[j] = ((((uint32_t)img * (uint32_t)p.Hs + (uint32_t)iy) * (uint32_t)p.Ws + (uint32_t)ix) * (uint32_t)p.C32) << 2;
    }
  }
  // filter words this thread stages: one channel, taps tap0, tap0 + TSTEP, ...; FT of them held in registers
  constexpr int TSTEP = NT / TB, FT = FORM == PF_5x5_PAIRS ? (TAPS + TSTEP - 1) / TSTEP : TSTEP >= 4 ? 3 : 5;
  const int fcol = tid % TB, tap0 = tid / TB;
  const uint32_t foff = b0 + fcol < p.rowsB
                            ? ((uint32_t)(b0 + fcol) * (uint32_t)taps + (uint32_t)tap0) * (uint32_t)p.C32 << 2
                            : kOff;

  const bool pair_ok = FORM == PF_3x3_PAIRS || FORM == PF_5x5_PAIRS || (FORM == PF_ANY && (p.C32 & 1) == 0);  // 64-bit loads of a channel-word pair
  const int nchunks = (p.C32 + 1) >> 1;
  uint32_t pw0[PATCH_NPT][PA], pw1[PATCH_NPT][PA], fw0[FT][PB], fw1[FT][PB];
  auto filter_load_w = [&](int cw, int first, auto pair_c) {
#pragma unroll
    for (int j = 0; j < FT; ++j) {
      const uint32_t boff = tap0 + first + j * TSTEP < taps ? foff : kOff;
      const uint32_t soff = (uint32_t)((first + j * TSTEP) * p.C32 + cw) << 2;
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) load_pair(rsrcB[pl], boff, soff, pair_c, cw + 1 < p.C32, fw0[j][pl], fw1[j][pl]);
    }
  };
  // packed words of a chunk: patch pixels and the first batch of filter words (one branch on the load width around
  // all of them)
  auto request_w = [&](int cw, auto pair_c) {
#pragma unroll
    for (int j = 0; j < PATCH_NPT; ++j) {
      if (j * NT < npp) {
#pragma unroll
        for (int pl = 0; pl < PA; ++pl)
          load_pair(rsrcA[pl], poff[j], (uint32_t)cw << 2, pair_c, cw + 1 < p.C32, pw0[j][pl], pw1[j][pl]);
      }
    }
    filter_load_w(cw, 0, pair_c);
  };
  auto request = [&](int cw) {
    if (pair_ok) request_w(cw, std::true_type{}); else request_w(cw, std::false_type{});
  };
  // Operands of a pixel's (channel's) two words; the words lie in blocks of their own, so that consecutive lanes read and
  // write consecutive 16-byte units (level with the words side by side: reads 32 bytes apart meet no bank twice either).
  auto put = [](uint32_t *at, int block, const v8i &e0, const v8i &e1) {
    *reinterpret_cast<uint4 *>(at) = make_uint4((uint32_t)e0[0], (uint32_t)e0[1], (uint32_t)e0[2], (uint32_t)e0[3]);
    *reinterpret_cast<uint4 *>(at + block) = make_uint4((uint32_t)e1[0], (uint32_t)e1[1], (uint32_t)e1[2], (uint32_t)e1[3]);
  };
  auto filter_store = [&](int first) {
#pragma unroll
    for (int j = 0; j < FT; ++j) {
      const int tap = tap0 + first + j * TSTEP;
      if (tap < taps) {
        if constexpr (ONE) {
          put(filtB + (tap * TB + fcol) * 4, taps * TB * 4, expand_w1<2>(fw0[j][0], p.sym != 0), expand_w1<2>(fw1[j][0], p.sym != 0));
        } else {
          static_for<0, DB>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            put(filtB + ((2 * d * taps + tap) * TB + fcol) * 4, taps * TB * 4, expand_fp4<PB, d>(fw0[j]), expand_fp4<PB, d>(fw1[j]));
          });
        }
      }
    }
  };

  request(0);
  const int rbase = a0 + wa * FA * 32, cbase = b0 + wb * FB * 32;
  table.store(p, b0, tab, inv_vs);

  v16f acc[FA][FB];
#pragma unroll
  for (int x = 0; x < FA; ++x)
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0;
  int ssum[FA];
#pragma unroll
  for (int x = 0; x < FA; ++x) ssum[x] = 0;

  // operands of one tap: patch at pa (and sums at ps), filter block at fb
  auto tap_read = [&](const uint32_t *pa, const uint32_t *fb, const int *ps, int dstride, v8i (&af)[FA][DA],
                      v8i (&bf)[FB][DB]) {
#pragma unroll
    for (int x = 0; x < FA; ++x) {
      if constexpr (!ONE) ssum[x] += ps[prow[x]];
#pragma unroll
      for (int d = 0; d < DA; ++d) {
        const uint4 v = *reinterpret_cast<const uint4 *>(pa + (2 * d * cap + prow[x]) * 4);
        af[x][d] = v8i{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const uint4 v = *reinterpret_cast<const uint4 *>(fb + d * dstride + y * 32 * 4);
        bf[y][d] = v8i{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      }
  };
  auto tap_products = [&](const v8i (&af)[FA][DA], const v8i (&bf)[FB][DB]) {
#pragma unroll
    for (int x = 0; x < FA; ++x)
#pragma unroll
      for (int y = 0; y < FB; ++y)
        static_for<0, DA>([&](auto dac) {
          static_for<0, DB>([&](auto dbc) {
            constexpr int da = decltype(dac)::value, db = decltype(dbc)::value;
            acc[x][y] = mfma_digits<2, da + db>(bf[y][db], af[x][da], acc[x][y]);
          });
        });
  };

  for (int cc = 0; cc < nchunks; ++cc) {
    const int cw = cc * 2;
    if (cc > 0) __syncthreads();  // every wave has finished reading the previous chunk
#pragma unroll
    for (int j = 0; j < PATCH_NPT; ++j) {
      const int q = tid + j * NT;
      if (j * NT < npp && q < npp) {
        if constexpr (!ONE) {
          int ps = 0;
#pragma unroll
          for (int pl = 0; pl < PA; ++pl) ps += (__popc(pw0[j][pl]) + __popc(pw1[j][pl])) << pl;
          pixsum[q] = ps;
        }
        static_for<0, DA>([&](auto dc) {
          constexpr int d = decltype(dc)::value;
          put(patchA + (2 * d * cap + q) * 4, cap * 4, expand_fp4<PA, d>(pw0[j]), expand_fp4<PA, d>(pw1[j]));
        });
      }
    }
    filter_store(0);
    for (int first = FT * TSTEP; first < taps; first += FT * TSTEP) {
      if (pair_ok) filter_load_w(cw, first, std::true_type{}); else filter_load_w(cw, first, std::false_type{});
      filter_store(first);
    }
    __syncthreads();
    if (cc + 1 < nchunks) request(cw + 2);

    const uint32_t *pa = patchA + g * cap * 4;
    const uint32_t *fb = filtB + (g * taps * TB + wb * FB * 32 + li) * 4;
    if constexpr (FORM != PF_ANY) {
      // a tap's operands are read while the one before is multiplied; the scheduler does not see past a tap, or it
      // would hoist the reads of all of them and spill
      v8i af[2][FA][DA], bf[2][FB][DB];
      int pitch = p.PWs;
      asm("" : "+s"(pitch));  // keeps the addresses of the taps from being held in registers over all chunks
      auto read = [&](auto tc) {
        constexpr int tap = decltype(tc)::value;
        const int toff = tap / SIDE * pitch + tap % SIDE;
        tap_read(pa + toff * 4, fb + tap * TB * 4, pixsum + toff, TAPS * TB * 8, af[tap & 1], bf[tap & 1]);
      };
      read(std::integral_constant<int, 0>{});
      static_for<0, TAPS>([&](auto tc) {
        constexpr int tap = decltype(tc)::value;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (tap + 1 < TAPS) read(std::integral_constant<int, tap + 1>{});
        tap_products(af[tap & 1], bf[tap & 1]);
      });
      __builtin_amdgcn_sched_barrier(0);
    } else {
      int toff = 0, sx = 0;
#pragma unroll 1
      for (int tap = 0; tap < taps; ++tap) {
        v8i af[FA][DA], bf[FB][DB];
        tap_read(pa + toff * 4, fb + tap * TB * 4, pixsum + toff, taps * TB * 8, af, bf);
        tap_products(af, bf);
        ++toff;
        if (++sx == p.S) {
          sx = 0;
          toff += p.PWs - p.S;
        }
      }
    }
  }

  if (p.fold != 0u) {
    uint32_t sc[FA][FB][2];
    conv_shortcut_load<FA, FB>(p, rbase, cbase, li, sc);
    fold_shortcut_lanes<FA, FB>(p, acc, sc, lane, log2vs);
  }
  if (need_sum) {
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
}

enum PatchTile { PT_128x128 = 0, PT_256x64 = 1, PT_64x128 = 2, PT_128x64 = 3, PT_64x64 = 4, PT_COUNT = 5 };
static_assert(PT_COUNT == kPatchTileCount, "tile tables of dispatch.h");

template <int PA, int PB, int FA, int FB, int WA, int WB, int FORM, bool SHORT = true>
inline hipError_t launch_patch_form(const KParams &p, hipStream_t stream) {
  constexpr int TA = WA * FA * 32, TB = WB * FB * 32;
  const size_t smem_bytes = patch_stage_words(PA, PB, TB, p.KW / p.C32, p.patch_cap) * 4 + conv_epilogue_bytes(p, TB);
  if (smem_bytes > 160 * 1024 || p.patch_cap > PATCH_NPT * 256) return hipErrorNotSupported;
  auto kern = apnn_patch_conv_kernel<PA, PB, FA, FB, WA, WB, FORM, SHORT>;
  if (smem_bytes > 64 * 1024) {
    static std::atomic<unsigned long long> raised;
    const hipError_t e = raise_lds_limit(raised, reinterpret_cast<const void *>(kern), 160 * 1024);
    if (e != hipSuccess) return e;
  }
  const long long tiles = (long long)((p.rowsA + TA - 1) / TA) * ((p.rowsB + TB - 1) / TB);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(256), smem_bytes, stream, p);
  return hipGetLastError();
}

// ODD, BIG: whether the forms for odd channel words and for 5x5 filters are built
template <int PA, int PB, int FA, int FB, int WA, int WB, bool ODD = false, bool BIG = false>
inline hipError_t launch_patch(const KParams &p, hipStream_t stream) {
  if (p.KW == 9 * p.C32 && p.S == 3) {
    if ((p.C32 & 1) == 0) return launch_patch_form<PA, PB, FA, FB, WA, WB, PF_3x3_PAIRS>(p, stream);
    if constexpr (ODD) return launch_patch_form<PA, PB, FA, FB, WA, WB, PF_3x3_ODD>(p, stream);
  }
  if constexpr (BIG) {
    if (p.KW == 25 * p.C32 && p.S == 5 && (p.C32 & 1) == 0) return launch_patch_form<PA, PB, FA, FB, WA, WB, PF_5x5_PAIRS>(p, stream);
  }
  return launch_patch_form<PA, PB, FA, FB, WA, WB, PF_ANY>(p, stream);
}

// Maps beyond the short quotients
template <int PA, int PB>
inline hipError_t launch_patch_long(int tile, const KParams &p, hipStream_t stream) {
  switch (tile) {
    case PT_128x128: return launch_patch_form<PA, PB, 2, 2, 2, 2, PF_ANY, false>(p, stream);
    case PT_256x64: return launch_patch_form<PA, PB, 2, 2, 4, 1, PF_ANY, false>(p, stream);
    case PT_64x128: return launch_patch_form<PA, PB, 1, 2, 2, 2, PF_ANY, false>(p, stream);
    case PT_128x64: return launch_patch_form<PA, PB, 1, 2, 4, 1, PF_ANY, false>(p, stream);
    case PT_64x64: return launch_patch_form<PA, PB, 1, 1, 2, 2, PF_ANY, false>(p, stream);
    default: return hipErrorNotSupported;
  }
}

template <int PA, int PB>
inline hipError_t launch_patch_tile(int tile, const KParams &p, hipStream_t stream) {
  if (p.geo_fast) {
    switch (tile) {
      case PT_128x128: return launch_patch<PA, PB, 2, 2, 2, 2>(p, stream);
      case PT_256x64: return launch_patch<PA, PB, 2, 2, 4, 1, true>(p, stream);
      case PT_64x128: return launch_patch<PA, PB, 1, 2, 2, 2>(p, stream);
      case PT_128x64: return launch_patch<PA, PB, 1, 2, 4, 1, true, true>(p, stream);
      case PT_64x64: return launch_patch<PA, PB, 1, 1, 2, 2>(p, stream);
      default: return hipErrorNotSupported;
    }
  }
  return launch_patch_long<PA, PB>(tile, p, stream);
}

}  // namespace apnn
