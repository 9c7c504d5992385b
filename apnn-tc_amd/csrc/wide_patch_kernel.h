// Patch-resident convolution with packed weights: large tiles over many channels (FP4 / FP6 operands, see mfma_kernel.h).
//
// The implicit-GEMM kernels of async_kernel.h expand an activation word once for every filter tap and for every wave that
// needs it: 6 vector operations per matrix instruction (w1a2), 9.8 with four activation planes, which is what bounds them.
// Here, as in patch_conv_kernel.h, the input pixels of a tile are expanded ONCE per pass over 256 channels and every tap
// reads ready operands from LDS; weights, whose expansion is cheap and shared by all pixels of a wave, stay packed: they go
// straight to LDS (as in async_kernel.h) and are expanded in registers.  In the loop that leaves the weights' expansion, 3.5
// vector operations per matrix instruction, and two 16-byte reads of activations per k-step and wave.
//
//   - a pass is eight channel words of all taps, a group one tap of it: four k-steps, the lower lane half on the first four
//     words, the upper on the last four.  Groups follow each other pass by pass, tap by tap; a group's weights come one group
//     ahead (two groups a chunk were no faster, and 8 KB more: 56x56x256 w1a2 67 instead of 60 us);
//   - the patch is the contiguous range of padded-frame pixels of a tile of consecutive output pixels (patch_conv_kernel.h), in a
//     frame whose rows and images share the padding between them, stored [word][pixel]: consecutive lanes read consecutive 16-byte units;
//   - three work-groups per compute unit (two with FP6 digits): one stages its patch while the others multiply.
//
// 128x128 tiles only: of 128x256 tiles one or two fit a compute unit (the patch is the same, the weights twice as long), and
// they were 4 to 20 % slower everywhere but near 784 tiles.  Graph replay at batch 64, implicit GEMM first: 14x14x512 to 512
// w1a2 20.5 -> 18.9 us, w1a3 27.7 -> 23.3, w1a4 34.5 -> 26.8, w2a2 23.4 -> 21.7; 28x28x512 to 512 w1a2 57.3 -> 54.2, w1a3
// 78.7 -> 72.4, w1a4 94.3 -> 84.5, w2a2 73.8 -> 62.4.  Of the busy clocks of 28x28x512 w1a2: matrix pipes 51 %, vector pipes
// 61 %, LDS 44 %, of which 45 % bank conflicts whose source is not known (profiles/ksplit_wide_patch_counters.md).
#pragma once
#include "async_kernel.h"
#include "quotient.h"
#include "wide_patch.h"

namespace apnn {

constexpr int WIDE_NPT = kWidePatchPixels * 2 / 256;  // half pixels (four words) a thread stages

// SHORT: maps of at most 65536 rows and columns (quotient.h; with shifts 13.2 -> 13.4 us at one tile per unit)
template <int PA, int PB, bool SYM, bool SHORT>
__global__ __launch_bounds__(256, wide_patch_units(PA)) void apnn_wide_patch_kernel(const KParams pk) {
  KParams p = pk;
  constexpr int FA = 2, FB = 2, WA = 2, WB = 2;  // four waves of two by two 32x32 accumulators
  constexpr int DIG = digit_planes(PA, PB);
  constexpr int DB = (PB + DIG - 1) / DIG;
  static_assert(PA <= DIG, "one digit of activations");
  constexpr bool SIGN = SYM && PB == 1;  // -1 / +1 operands: the accumulator is the result
  constexpr bool SUM = SYM && PB > 1;    // activation sums enter the result
  constexpr int FSC = SIGN ? (DIG == 4 ? 8 : 2) : fp_scale(PA, PB);
  if (!SUM) p.sym = 0;
  constexpr int TA = WA * FA * 32, TB = WB * FB * 32;
  constexpr int KC = 8, UPR = KC / 4, RPI = 64 / UPR, NB = TB / RPI / 4;
  static_assert(TB % (RPI * 4) == 0, "row groups go round the four waves");
  constexpr int BUF = PB * TB * KC;  // words
  constexpr int MAXB = PA >= 3 ? 4 : 2;

  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  const int cap = p.patch_cap;
  uint32_t *patch = smem + 2 * BUF;                   // [8 words][cap][4 dwords]
  uint32_t *patch2 = patch + 32 * cap;                // FP6: [8 words][cap][2 dwords]
  int *pixsum = reinterpret_cast<int *>(patch2 + (DIG == 4 ? 16 * cap : 0));  // [2 halves][cap], two weight planes
  uint32_t *tab = smem + wide_stage_words(PA, PB, TB, cap);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int wa = wave / WB, wb = wave % WB;
  const int tilesB = (p.rowsB + TB - 1) / TB;
  int trow = blockIdx.x / tilesB, tcol = blockIdx.x % tilesB;
  if (p.xcd_rows > 0) {  // see apnn_mfma_kernel
    const int tilesA = (p.rowsA + TA - 1) / TA;
    const int per_xcd = (tilesA * tilesB) >> 3;
    const int lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const int per_band = p.xcd_rows * tilesB;
    const int band = lin / per_band, w = lin - band * per_band;
    const int rows_in_band = min(p.xcd_rows, tilesA - band * p.xcd_rows);
    tcol = w / rows_in_band;
    trow = band * p.xcd_rows + (w - tcol * rows_in_band);
  }
  const int a0 = trow * TA, b0 = tcol * TB;

  constexpr int log2vs = __builtin_ctz(FSC) + (SUM ? 1 : 0);
  const float inv_vs = 1.0f / (float)(1 << log2vs);
  ConvTable<TB, PA >= 3 ? 15 : 3, MAXB> table;
  table.load(p, b0);

  // ---- tile geometry (see patch_conv_kernel.h) ----------------------------------------------------------------------
  const int taps = p.KW / p.C32, R = taps / p.S, passes = p.C32 >> 3;
  const int last_row = min(a0 + TA, p.rowsA) - 1;
  const bool pooled = p.pool_order != 0;
  const int gw = pooled ? p.Wo >> 1 : p.Wo, gh = pooled ? p.Ho >> 1 : p.Ho;
  const int gst = pooled ? 2 * p.stride : p.stride;
  const uint32_t u0 = (uint32_t)(pooled ? a0 >> 2 : a0);
  const uint32_t t0 = u0 / (uint32_t)gw;
  const int gx0 = (int)(u0 - t0 * (uint32_t)gw);
  const int b0i = (int)(t0 / (uint32_t)gh);
  const int gy0 = (int)(t0 - (uint32_t)b0i * (uint32_t)gh);
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
  const int q_lo = row_base(0);
  const int npp = row_base(last_row - a0) + (R - 1) * p.PWs + (p.S - 1) - q_lo + 1;
  if (npp > cap) {  // never, see patch_conv_kernel.h
    if (tid == 0 && p.err != nullptr) atomicOr(p.err, (int)KERR_PATCH_CAPACITY);
    return;
  }
  int prow[FA];  // this lane's pixels in the patch
#pragma unroll
  for (int x = 0; x < FA; ++x) prow[x] = row_base(min((wa * FA + x) * 32 + li, last_row - a0)) - q_lo;

  // ---- patch: half pixels tid, tid + 256, ... (pixel h / 2, words 4 (h % 2) ..) --------------------------------------
  __amdgpu_buffer_rsrc_t rsrcA[PA];
#pragma unroll
  for (int pl = 0; pl < PA; ++pl)
    rsrcA[pl] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p.A + pl * p.planeA), 0,
                                                  (int)(uint32_t)(p.planeA * 4), 0x00020000);
  uint32_t poff[WIDE_NPT];
  const int pad_v = p.PHs - p.Hs;  // (the frame ends with its last stored row and pixel, see wide_patch_frame)
  const int yp0 = gy0 * gst, xp0 = gx0 * gst;
#pragma unroll
  for (int j = 0; j < WIDE_NPT; ++j) {
    const int q = (tid + j * 256) >> 1;
    poff[j] = 0xffffffffu;
    if (q < npp) {
      int xp = xp0 + q;
      const int cy = (int)quotient<SHORT>((uint32_t)xp, (uint32_t)p.PWs, p.magicPW);
      xp -= cy * p.PWs;
      int yp = yp0 + cy;
      const int ci = (int)quotient<SHORT>((uint32_t)yp, (uint32_t)p.PHs, p.magicPH);
      yp -= ci * p.PHs;
      const int img = b0i + ci;
      const int iy = yp - pad_v, ix = xp - pad_v;
      if (img < p.batch && iy >= 0 && iy < p.Hs && ix >= 0 && ix < p.Ws)
        poff[j] = ((((uint32_t)img * (uint32_t)p.Hs + (uint32_t)iy) * (uint32_t)p.Ws + (uint32_t)ix) * (uint32_t)p.C32 + 4u * (tid & 1)) << 2;
    }
  }
  uint4 pw[WIDE_NPT][PA];
  auto request = [&](int pass) {
#pragma unroll
    for (int j = 0; j < WIDE_NPT; ++j)
      if (j * 128 < npp) {
#pragma unroll
        for (int pl = 0; pl < PA; ++pl) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrcA[pl], (int)poff[j], pass * 32, 0);
          pw[j][pl] = make_uint4(v[0], v[1], v[2], v[3]);
        }
      }
  };
  auto word = [](const uint4 &q, auto ic) -> uint32_t {
    constexpr int i = decltype(ic)::value;
    return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w;
  };
  auto publish = [&]() {
#pragma unroll
    for (int j = 0; j < WIDE_NPT; ++j) {
      const int q = (tid + j * 256) >> 1, h = tid & 1;
      if (j * 128 < npp && q < npp) {
        int sum = 0;
        static_for<0, 4>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          uint32_t w[PA];
#pragma unroll
          for (int pl = 0; pl < PA; ++pl) {
            w[pl] = word(pw[j][pl], ic);
            if constexpr (SUM) sum += __popc(w[pl]) << pl;
          }
          const v8i e = expand_digit<DIG, PA, 0>(w);
          const int at = (4 * h + i) * cap + q;
          *reinterpret_cast<uint4 *>(patch + at * 4) = make_uint4((uint32_t)e[0], (uint32_t)e[1], (uint32_t)e[2], (uint32_t)e[3]);
          if constexpr (DIG == 4) *reinterpret_cast<uint2 *>(patch2 + at * 2) = make_uint2((uint32_t)e[4], (uint32_t)e[5]);
        });
        if constexpr (SUM) pixsum[h * cap + q] = sum;
      }
    }
  };

  // ---- weights: a group's straight to LDS, as in async_kernel.h ---------------------------------------------
  rsrc4 rsB[PB];
#pragma unroll
  for (int pl = 0; pl < PB; ++pl) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(p.B + pl * p.planeB);
    rsB[pl] = rsrc4{(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffffu), (int)(uint32_t)(p.planeB * 4), 0x00020000};
  }
  const int lrow = lane / UPR;
  const int unit = (lane % UPR) ^ ((lrow >> 3) & 1);
  uint32_t voB[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int row = b0 + (wave + 4 * n) * RPI + lrow;
    voB[n] = row < p.rowsB ? ((uint32_t)row * (uint32_t)p.KW + 4u * unit) * 4u : 0xffffffffu;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)smem;
  const int groups = taps * passes;
  int fpass = 0, ftap = 0;  // pass and tap of the next group to fetch
  auto fetch = [&](int buf) {
    const uint32_t k = (uint32_t)(ftap * p.C32 + 8 * fpass) * 4u;
    if (++ftap == taps) {
      ftap = 0;
      ++fpass;
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const uint32_t vo = voB[n] == 0xffffffffu ? 0xffffffffu : voB[n] + k;
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) {
        const uint32_t lds = lds0 + (uint32_t)((buf * BUF + (pl * TB + (wave + 4 * n) * RPI) * KC) * 4);
        // (m0 holds the LDS address)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     :
                     : "s"(lds), "v"(vo), "s"(rsB[pl])
                     : "memory", "m0");
      }
    }
  };
  auto arrive = [&]() {  // the loads above are invisible to the compiler's wait counts
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  request(0);
  fetch(0);
  const int rbase = a0 + wa * FA * 32, cbase = b0 + wb * FB * 32;
  uint32_t sc[FA][FB][2];
  if (p.fold != 0u) conv_shortcut_load<FA, FB>(p, rbase, cbase, li, sc);
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

  // Weights of a group (this lane's four words of every row), in two halves: see async_kernel.h
  uint2 qB[2][FB][PB];
  const int rowB = wb * FB * 32 + li;
  const int swz = (li >> 3) & 1;
  auto read_half = [&](const uint32_t *buf, auto hc) {
    constexpr int h = decltype(hc)::value;
    const int place = (g ^ swz) * 4 + 2 * h;
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) qB[h][y][pl] = *reinterpret_cast<const uint2 *>(buf + (pl * TB + rowB + y * 32) * KC + place);
  };
  v8i af[FA], bf[FB][DB];
  auto read_x = [&](auto ic, int toff, v8i (&a)[FA]) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int x = 0; x < FA; ++x) {
      const int at = (4 * g + i) * cap + prow[x] + toff;
      const uint4 v = *reinterpret_cast<const uint4 *>(patch + at * 4);
      a[x] = v8i{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      if constexpr (DIG == 4) {
        const uint2 u = *reinterpret_cast<const uint2 *>(patch2 + at * 2);
        a[x][4] = (int)u.x;
        a[x][5] = (int)u.y;
      }
    }
  };
  auto expand_w = [&](auto ic, v8i (&b)[FB][DB]) {
    constexpr int i = decltype(ic)::value, h = i / 2;
#pragma unroll
    for (int y = 0; y < FB; ++y) {
      uint32_t w[PB];
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) w[pl] = i % 2 == 0 ? qB[h][y][pl].x : qB[h][y][pl].y;
      if constexpr (SIGN) {
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
        static_for<0, DB>([&](auto dbc) {
          constexpr int db = decltype(dbc)::value;
          acc[x][y] = mfma_digits<DIG, db>(bf[y][db], af[x], acc[x][y]);
        });
  };
  constexpr int N_MFMA = FA * FB * DB;
  constexpr int XDIG[5] = {0, 7, 10, 18, 22};
  constexpr int N_VALU = FB * (XDIG[DIG] * (PB / DIG) + XDIG[PB % DIG]);
  constexpr int VALU_PER_MFMA = (N_VALU + N_MFMA - 1) / N_MFMA;
  // matrix products of one k-step and, between them, the operands of the next
  auto step = [&](auto ic, int toff) {
    v8i an[FA], bn[FB][DB];
    read_x(ic, toff, an);
    __builtin_amdgcn_sched_barrier(0);  // the reads go ahead of the products they travel behind
    mfma_all();
    expand_w(ic, bn);
#pragma unroll
    for (int x = 0; x < FA; ++x) af[x] = an[x];
#pragma unroll
    for (int y = 0; y < FB; ++y)
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        bf[y][d] = bn[y][d];
        // (made here, behind the products: not where a branch further on first needs them)
        static_for<0, DIG == 4 ? 6 : 4>([&](auto ec) {
          int e = bf[y][d][decltype(ec)::value];
          asm volatile("" : "+v"(e));
          bf[y][d][decltype(ec)::value] = e;
        });
      }
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

  publish();
  arrive();
  if (groups > 1) fetch(1);
  int group = 0;
  read_half(smem, I0{});
  read_half(smem, I1{});
#pragma unroll 1
  for (int pass = 0; pass < passes; ++pass) {
    if (pass > 0) {
      request(pass);
      __syncthreads();  // every wave has read the last pass
      publish();
      __syncthreads();
    }
    int toff = 0, sx = 0;
    read_x(I0{}, 0, af);
    expand_w(I0{}, bf);
#pragma unroll 1
    for (int tap = 0; tap < taps; ++tap) {
      if constexpr (SUM) {
#pragma unroll
        for (int x = 0; x < FA; ++x) ssum[x] += pixsum[g * cap + prow[x] + toff];
      }
      step(I1{}, toff);
      // every wave holds the group's words when it has begun (after the last group of all the words read here are stale and
      // meet no product)
      if (group + 1 < groups) {
        arrive();
        if (group + 2 < groups) fetch(group & 1);
      }
      ++group;
      read_half(smem + (group & 1) * BUF, I0{});
      step(I2{}, toff);
      step(I3{}, toff);
      read_half(smem + (group & 1) * BUF, I1{});
      ++toff;
      if (++sx == p.S) {
        sx = 0;
        toff += p.PWs - p.S;
      }
      // (after the last tap of a pass the operands made here are of no use: the next pass reads its own)
      step(I0{}, tap + 1 < taps ? toff : 0);
    }
  }

  if (p.fold != 0u) fold_shortcut_lanes<FA, FB>(p, acc, sc, lane, log2vs);
  if constexpr (SUM) {
#pragma unroll
    for (int x = 0; x < FA; ++x) {
      const float c = (float)(ssum[x] + __shfl_xor(ssum[x], 32, 64)) * (-(float)p.wmax * inv_vs);
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

template <int PA, int PB>
inline hipError_t launch_wide_patch(const KParams &p, hipStream_t stream) {
  constexpr int TA = kMfmaTileA[MT_128x128_P], TB = kMfmaTileB[MT_128x128_P];
  if (p.patch_cap > kWidePatchPixels || (p.C32 & 7) != 0) return hipErrorNotSupported;
  static_assert(2 * PB * TB * 8 * 4 <= 64 * 1024, "LDS addresses of the loads fit 16 bits");
  const size_t bytes = wide_stage_words(PA, PB, TB, p.patch_cap) * 4 + conv_epilogue_bytes(p, TB);
  if (bytes > 160 * 1024) return hipErrorNotSupported;
  auto kern = p.sym ? (p.geo_fast ? apnn_wide_patch_kernel<PA, PB, true, true> : apnn_wide_patch_kernel<PA, PB, true, false>)
                    : (p.geo_fast ? apnn_wide_patch_kernel<PA, PB, false, true> : apnn_wide_patch_kernel<PA, PB, false, false>);
  if (bytes > 64 * 1024) {
    static std::atomic<unsigned long long> raised[4];
    const hipError_t e = raise_lds_limit(raised[2 * (p.sym != 0) + (p.geo_fast != 0)], reinterpret_cast<const void *>(kern), 160 * 1024);
    if (e != hipSuccess) return e;
  }
  const long long tilesB = (p.rowsB + TB - 1) / TB, tiles = (long long)((p.rowsA + TA - 1) / TA) * tilesB;
  KParams q = p;
  q.xcd_rows = (tiles % 8 == 0 && tiles >= kXcdOrderMinTiles && tilesB >= 2) ? 8 : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(256), bytes, stream, q);
  return hipGetLastError();
}

}  // namespace apnn
