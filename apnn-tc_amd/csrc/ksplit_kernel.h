// GEMM entry points on FP4 / FP6 operands where the tiles of mfma_kernel.h are few: eight waves share one tile's K.
//
// What bounds such products.  With one work-group of four waves per compute unit a SIMD holds a single wave, which issues
// a vector operation only every eight clocks (two waves together: every four), and the expansion of the bit-planes is most
// of what a wave does: 22 operations per 32x32 operand block and k-step for four planes, 33 clocks for the product.  So
//   - eight waves work on a tile, WA of them along the weight rows, KS shares of K each: two waves per SIMD at one
//     work-group per unit, whatever the tile;
//   - a wave's tile is as large as its registers allow (FA x FB blocks), because expansion work goes with its circumference;
//   - a chunk is 32 words of every row, one cache line: eight lanes load a row's 128 bytes.  (Loaded row by row straight into
//     registers, 32 bytes of a line at a time, the lines' way through L1 took three times as long as the expansion.)  The
//     16-byte units of a row are permuted by its index in LDS, so that sixteen rows are read without one of the 64 banks met
//     twice (by half the index; the whole index, which repeats after eight rows, was 2 to 3 % slower);
//   - the eight units of a row go to the KS waves: two to each of four, whose lane halves take one each (four k-steps a
//     chunk), or one to each of eight, whose lane halves take half of it (two k-steps).  Both operands alike: a permutation
//     of the terms of each dot product.  A last chunk of up to half its words is spread over the waves word by word instead
//     (1152 bits, us: 2048x2048 w1a8 20.2 -> 17.9, 1000x2016 w2a2 8.05 -> 7.70, w4a4 11.5 -> 10.6; beyond half the reads word by word cost 1 to 2 %).
// The partial tiles meet in LDS in the accumulator's register layout, RB blocks of every wave at a time; wave k of a row
// group sums block k over the KS shares and finishes it like a wave of the other kernels (epi_finish).
//
// us in graph replay, the tiles these products took before first: w4a4 4096x333x4096 (64x64 tiles, 384 on 256 units) 25.5 ->
// 13.6, over 8192 bits 43.9 -> 20.4; w2a2 1000x2016x2048 packed (128x64) 11.1 -> 8.3, over 8192 bits 27.5 -> 15.6; w1a4 and
// w1a8 there 12.1 -> 8.3 and 18.6 -> 11.3.  Left (profiles/ksplit_wide_patch_counters.md): a chunk of 1024 bits takes 1.1
// us (w2a2, the slope over 3072 to 8192 bits; w4a4 on 64x96 tiles 1.7), vector pipes a third and matrix pipes a tenth of the
// launch busy, waves waiting half of their time; 5 to 7 us lie beside the loop, launch included, not taken apart further.  Words
// of the next chunk held in a second register set gained 2 % and spilled with four activation planes: taken out.
#pragma once
#include "mfma_kernel.h"

namespace apnn {

// blocks of a wave that meet in LDS at a time: 4 KB each, at most 128 KB of all eight waves
constexpr int ksplit_round_blocks(int blocks) { return blocks <= 4 ? blocks : (blocks + 1) / 2; }
constexpr size_t ksplit_part_words(int FA, int FB, int WA, int KS) {
  return (size_t)WA * KS * ((size_t)ksplit_round_blocks(FA * FB) * 1024 + FB * 32);
}
// rows of all planes that a chunk stages; LDS buffers of a chunk: two where they fit
constexpr int ksplit_rows(int PA, int PB, int FA, int FB, int WA) { return PA * WA * FA * 32 + PB * FB * 32; }
constexpr int ksplit_buffers(int rows) { return 2 * rows * 128 <= 160 * 1024 ? 2 : 1; }

// k-steps of a wave in a full chunk, words of a row in its lane half
constexpr int ksplit_steps(int KS) { return KS == 8 ? 2 : 4; }
// whether the last chunk holds at most half its words
constexpr bool ksplit_tail(int KW, int KS) { return (KW & 31) > 0 && (KW & 31) <= KS * ksplit_steps(KS); }

// TAIL: ksplit_tail; a kernel of its own, as its code behind the loop took products of whole chunks 0.07 us on their way to the
// output stage (0.14 in front of it)
template <int PA, int PB, int FA, int FB, int WA, int KS, bool SYM, bool TAIL>
__global__ __launch_bounds__(64 * WA * KS, 1) void apnn_ksplit_kernel(const KParams pk) {
  KParams p = pk;
  static_assert(WA * KS == 8, "eight waves");
  constexpr int DIG = digit_planes(PA, PB);
  constexpr int DA = (PA + DIG - 1) / DIG, DB = (PB + DIG - 1) / DIG;
  constexpr bool SIGN = SYM && PA == 1;  // -1 / +1 operands: the accumulator is the result
  constexpr bool SUM = SYM && PA > 1;    // activation sums enter the result
  constexpr int FSC = SIGN ? (DIG == 4 ? 8 : 2) : fp_scale(PA, PB);
  if (!SUM) p.sym = 0;
  constexpr int TA = WA * FA * 32, TB = FB * 32, NBLK = FA * FB;
  constexpr int RB = ksplit_round_blocks(NBLK);
  static_assert(NBLK <= KS * ((NBLK + RB - 1) / RB) && NBLK <= KS, "a wave finishes one block");
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int wa = wave / KS, ks = wave % KS;

  const int tilesB = (p.rowsB + TB - 1) / TB;
  const int bid = blockIdx.x;
  int trow = bid / tilesB, tcol = bid % tilesB;
  if (p.xcd_rows > 0) {  // see apnn_mfma_kernel
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

  // staging: thread t of a batch of 64 rows loads unit t % 8 of row t / 8 (eight rows of one plane per wave)
  constexpr int ROWS = ksplit_rows(PA, PB, FA, FB, WA), NI = ROWS / 64, NBUF = ksplit_buffers(ROWS);
  static_assert(ROWS % 64 == 0, "whole batches of rows");
  const int su = lane & 7, sr = lane >> 3;
  uint32_t voff[NI];
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int rp = wave * 8 + it * 64;
    const bool isA = rp < PA * TA;
    const int row = (isA ? a0 + rp % TA : b0 + (rp - PA * TA) % TB) + sr;
    voff[it] = row < (isA ? p.rowsA : p.rowsB) ? ((uint32_t)row * (uint32_t)p.KW + 4u * su) * 4u : 0xffffffffu;
  }
  uint4 st[NI];
  auto fetch = [&](int ch) {
    const bool ok = ch * 32 + 4 * su < p.KW;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int rp = wave * 8 + it * 64;
      const bool isA = rp < PA * TA;
      const uint32_t *base = isA ? p.A + (rp / TA) * p.planeA : p.B + ((rp - PA * TA) / TB) * p.planeB;
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(base), 0,
                                                          (int)(uint32_t)((isA ? p.planeA : p.planeB) * 4), 0x00020000);
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(ok ? voff[it] : 0xffffffffu), ch * 128, 0);
      st[it] = make_uint4(v[0], v[1], v[2], v[3]);
    }
  };
  // Units are permuted by the row; for eight waves, which read half units, the halves are too (by the whole index: by half of
  // it 4096x333 over 4096 and 8192 bits took 2 to 3 % longer).
  const int wrow = wave * 8 + sr;
  const uint32_t swr = (uint32_t)(wrow * 32 + (KS == 8 ? (2 * su ^ (wrow & 15)) * 2 : (su ^ ((wrow >> 1) & 7)) * 4));
  auto stage = [&](uint32_t *buf) {
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      if constexpr (KS == 8) {
        *reinterpret_cast<uint2 *>(buf + swr + it * 64 * 32) = make_uint2(st[it].x, st[it].y);
        *reinterpret_cast<uint2 *>(buf + (swr ^ 2u) + it * 64 * 32) = make_uint2(st[it].z, st[it].w);
      } else {
        *reinterpret_cast<uint4 *>(buf + swr + it * 64 * 32) = st[it];
      }
    }
  };
  constexpr int NW = ksplit_steps(KS);
  const int nchunks = (p.KW + 31) >> 5, nfull = TAIL ? nchunks - 1 : nchunks;
  fetch(0);

  v16f acc[FA][FB];
#pragma unroll
  for (int x = 0; x < FA; ++x)
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0;
  int psum[FB][PB];
#pragma unroll
  for (int y = 0; y < FB; ++y)
#pragma unroll
    for (int pl = 0; pl < PB; ++pl) psum[y][pl] = 0;

  // this wave's words of a chunk
  uint32_t qA[FA][PA][NW], qB[FB][PB][NW];
  const int place = KS == 8 ? ((2 * ks + g) ^ (li & 15)) * 2 : ((2 * ks + g) ^ ((li >> 1) & 7)) * 4;
  auto read = [&](const uint32_t *buf) {
    auto get = [&](int row, uint32_t (&q)[NW]) {
      const uint32_t *at = buf + (row + li) * 32 + place;
      if constexpr (NW == 4) {
        const uint4 v = *reinterpret_cast<const uint4 *>(at);
        q[0] = v.x, q[1] = v.y, q[2] = v.z, q[3] = v.w;
      } else {
        const uint2 v = *reinterpret_cast<const uint2 *>(at);
        q[0] = v.x, q[1] = v.y;
      }
    };
#pragma unroll
    for (int x = 0; x < FA; ++x)
#pragma unroll
      for (int pl = 0; pl < PA; ++pl) get(pl * TA + (wa * FA + x) * 32, qA[x][pl]);
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) get(PA * TA + pl * TB + y * 32, qB[y][pl]);
  };
  v8i af[FA][DA], bf[FB][DB];
  auto expand = [&](auto ic, v8i (&a)[FA][DA], v8i (&b)[FB][DB]) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int x = 0; x < FA; ++x) {
      uint32_t w[PA];
#pragma unroll
      for (int pl = 0; pl < PA; ++pl) w[pl] = qA[x][pl][i];
      if constexpr (SIGN) {
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
        w[pl] = qB[y][pl][i];
        if constexpr (SUM) psum[y][pl] += __popc(w[pl]);
      }
      static_for<0, DB>([&](auto dc) { b[y][decltype(dc)::value] = expand_digit<DIG, PB, decltype(dc)::value>(w); });
    }
  };
  auto mfma_all = [&]() {
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int x = 0; x < FA; ++x)
        static_for<0, DA>([&](auto dac) {
          static_for<0, DB>([&](auto dbc) {
            constexpr int da = decltype(dac)::value, db = decltype(dbc)::value;
            acc[x][y] = mfma_digits<DIG, da + db>(af[x][da], bf[y][db], acc[x][y]);
          });
        });
  };
  constexpr int N_MFMA = FA * FB * DA * DB;
  constexpr int XDIG[5] = {0, 7, 10, 18, 22};
  constexpr int XA = XDIG[DIG] * (PA / DIG) + XDIG[PA % DIG], XB = XDIG[DIG] * (PB / DIG) + XDIG[PB % DIG];
  constexpr int N_VALU = FA * XA + FB * XB + (SUM ? FB * PB : 0);
  constexpr int VALU_PER_MFMA = (N_VALU + N_MFMA - 1) / N_MFMA;
  // words, staged words and the operands of two k-steps beside the accumulators (w2a8, 264, spills)
  static_assert(NBLK * 16 + NW * (FA * PA + FB * PB) + 4 * NI + 2 * (FA * DA + FB * DB) * (DIG == 4 ? 6 : 4) <= 256, "registers");
  // Matrix products of one k-step and, between them, the expansion of the next.  Two waves that expand and multiply in
  // turns get in each other's way: while one waits for the matrix pipe the other issues a vector operation every eight
  // clocks only (1000x2016x2048 w2a2 packed 8.8 -> 8.5 us, w1a8 11.9 -> 11.3, w4a4 4096x333x4096 14.1 -> 13.6).
  auto step = [&](auto ic) {
    v8i an[FA][DA], bn[FB][DB];
    mfma_all();
    expand(ic, an, bn);
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
  auto buffer = [&](int ch) { return smem + (NBUF == 2 ? (ch & 1) * ROWS * 32 : 0); };
  stage(buffer(0));
  if (nchunks > 1) fetch(1);
  __syncthreads();
#pragma unroll 1
  for (int ch = 0; ch < nfull; ++ch) {
    read(buffer(ch));
    if constexpr (NBUF == 1) __syncthreads();  // every wave holds its words
    if (ch + 1 < nchunks) {
      stage(buffer(ch + 1));
      if (ch + 2 < nchunks) fetch(ch + 2);
    }
    expand(std::integral_constant<int, 0>{}, af, bf);
    static_for<1, NW>([&](auto ic) { step(ic); });
    mfma_all();
    __syncthreads();
  }
  if constexpr (TAIL) {  // the words evenly: a k-step of all waves takes 2 KS of a row's
    const uint32_t *buf = buffer(nfull);
    const int n = ((p.KW & 31) + 2 * KS - 1) / (2 * KS);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      const int w = (2 * ks + g) * n + i;
      const uint32_t *at = buf + li * 32 + (KS == 8 ? ((w >> 1) ^ (li & 15)) * 2 + (w & 1) : ((w >> 2) ^ ((li >> 1) & 7)) * 4 + (w & 3));
#pragma unroll
      for (int x = 0; x < FA; ++x)
#pragma unroll
        for (int pl = 0; pl < PA; ++pl) qA[x][pl][0] = at[(pl * TA + (wa * FA + x) * 32) * 32];
#pragma unroll
      for (int y = 0; y < FB; ++y)
#pragma unroll
        for (int pl = 0; pl < PB; ++pl) qB[y][pl][0] = at[(PA * TA + pl * TB + y * 32) * 32];
      expand(std::integral_constant<int, 0>{}, af, bf);
      mfma_all();
    }
    __syncthreads();
  }

  int *sums = reinterpret_cast<int *>(smem) + WA * KS * RB * 1024;  // [8 waves][FB][32]
  if constexpr (SUM) {
#pragma unroll
    for (int y = 0; y < FB; ++y) {
      int t = 0;
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) t += psum[y][pl] << pl;
      t += __shfl_xor(t, 32, 64);
      if (g == 0) sums[(wave * FB + y) * 32 + li] = t;
    }
  }
  v16f own[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) own[0][0][r] = 0;
  float4 *part = reinterpret_cast<float4 *>(smem);  // [8 waves][RB][4 quads][64 lanes]
  constexpr int ROUNDS = (NBLK + RB - 1) / RB;
  static_for<0, ROUNDS>([&](auto rc) {
    constexpr int round = decltype(rc)::value;
    if (round > 0) __syncthreads();  // the sums of the round before have been read
    static_for<0, RB>([&](auto bc) {
      constexpr int b = decltype(bc)::value, blk = round * RB + b;
      if constexpr (blk < NBLK) {
        if (ks == blk) {  // its own block stays in registers
          own[0][0] = acc[blk / FB][blk % FB];
          return;
        }
        static_for<0, 4>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          const v16f &v = acc[blk / FB][blk % FB];
          part[((wave * RB + b) * 4 + q) * 64 + lane] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        });
      }
    });
    __syncthreads();
    if (ks / RB == round && ks < NBLK) {
#pragma unroll
      for (int i = 1; i < KS; ++i) {
        const int w = (ks + i) % KS;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 v = part[(((wa * KS + w) * RB + ks % RB) * 4 + q) * 64 + lane];
          own[0][0][4 * q] += v.x;
          own[0][0][4 * q + 1] += v.y;
          own[0][0][4 * q + 2] += v.z;
          own[0][0][4 * q + 3] += v.w;
        }
      }
    }
  });
  if (ks >= NBLK) {
    __syncthreads();  // the barrier of epi_finish
    return;
  }
  int own_sum[1] = {0};
  if constexpr (SUM) {
#pragma unroll
    for (int w = 0; w < KS; ++w) own_sum[0] += sums[((wa * KS + w) * FB + ks % FB) * 32 + li];
  }
  EpiOperands<1, 1> eo;
  const int rbase = a0 + (wa * FA + ks / FB) * 32, cbase = b0 + (ks % FB) * 32;
  epi_prefetch<1, PB >= 3 ? 4 : 2, true>(p, rbase, cbase, lane, eo);
  epi_finish<FSC, 1, false, PB >= 3 ? 4 : 2, true>(p, own, own_sum, smem, wave, lane, rbase, cbase, 0, 0, eo);
}

template <int PA, int PB, int FA, int FB, int WA, int KS>
inline hipError_t launch_ksplit(const KParams &p, hipStream_t stream) {
  constexpr int TA = WA * FA * 32, TB = FB * 32;
  constexpr size_t slab = 8ull * (32 * 33 + 32 + 32 + 64) * sizeof(int);  // epi_finish, one block per wave
  constexpr size_t part = ksplit_part_words(FA, FB, WA, KS) * sizeof(uint32_t);
  constexpr int rows = ksplit_rows(PA, PB, FA, FB, WA);
  constexpr size_t chunk = (size_t)ksplit_buffers(rows) * rows * 128;
  constexpr size_t need = part > chunk ? part : chunk, bytes = need > slab ? need : slab;
  static_assert(bytes <= 160 * 1024, "LDS of a compute unit");
  const bool tail = ksplit_tail(p.KW, KS);
  auto kern = p.sym ? (!tail ? apnn_ksplit_kernel<PA, PB, FA, FB, WA, KS, true, false> : apnn_ksplit_kernel<PA, PB, FA, FB, WA, KS, true, true>)
                    : (!tail ? apnn_ksplit_kernel<PA, PB, FA, FB, WA, KS, false, false> : apnn_ksplit_kernel<PA, PB, FA, FB, WA, KS, false, true>);
  static std::atomic<unsigned long long> raised[4];
  const hipError_t e = raise_lds_limit(raised[2 * (p.sym != 0) + tail], reinterpret_cast<const void *>(kern), bytes);
  if (e != hipSuccess) return e;
  const long long tilesB = (p.rowsB + TB - 1) / TB, tiles = (long long)((p.rowsA + TA - 1) / TA) * tilesB;
  KParams q = p;
  q.xcd_rows = (tiles % 8 == 0 && tiles >= kXcdOrderMinTiles && tilesB >= 2) ? 8 : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(512), bytes, stream, q);
  return hipGetLastError();
}

}  // namespace apnn
