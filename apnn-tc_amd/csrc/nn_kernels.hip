// Kernels on either side of the low-bit path of a network: the int8 first convolution with its
// threshold quantizer, max-pool + bit-plane packing of the resulting codes, global average pooling
// of packed codes, code unpacking and the int8 classifier.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "../../include/apnn_tc.h"
#include "dispatch.h"

namespace apnn {

// ---- int8 first convolution + per-channel thresholds -> codes ------------------------------------
// X: [B][H][W][C] int8 (or uint8 minus zero_point when zero_point != 0), Wt: [COUT][R][S][C] int8
// (C tiny: 3), thr: [COUT][2^bits-1] int32.
// One work-group computes a strip of 64 output pixels x COUT_T=64 channels; the filter block is
// staged in LDS once, each thread owns one pixel and 16 channels.
template <int COUT_T>
__global__ __launch_bounds__(256) void conv_i8_bn_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                         const int32_t *__restrict__ thr,
                                                         uint8_t *__restrict__ codes, int32_t *__restrict__ acc_out,
                                                         int B, int H, int W, int C, int COUT, int R, int S,
                                                         int stride, int pad, int Ho, int Wo, int bits, int zero_point) {
  extern __shared__ int8_t wlds[];  // [COUT_T][R*S*C]
  const int K = R * S * C;
  const int co0 = blockIdx.y * COUT_T;
  for (int i = threadIdx.x; i < COUT_T * K; i += 256) {
    const int co = co0 + i / K;
    wlds[i] = co < COUT ? Wt[(long long)co * K + (i % K)] : (int8_t)0;
  }
  __syncthreads();
  const int pl = threadIdx.x & 63;          // pixel within the strip
  const int cg = threadIdx.x >> 6;          // channel group: 16 channels
  const long long pix = (long long)blockIdx.x * 64 + pl;
  const long long npix = (long long)B * Ho * Wo;
  if (pix >= npix) return;
  const int ox = (int)(pix % Wo);
  const int oy = (int)((pix / Wo) % Ho);
  const int b = (int)(pix / ((long long)Wo * Ho));
  int acc[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = 0;
  for (int r = 0; r < R; ++r) {
    const int iy = oy * stride + r - pad;
    if (iy < 0 || iy >= H) continue;
    for (int s = 0; s < S; ++s) {
      const int ix = ox * stride + s - pad;
      if (ix < 0 || ix >= W) continue;
      const int8_t *xp = X + (((long long)b * H + iy) * W + ix) * C;
      const int8_t *wp = wlds + (cg * 16) * K + (r * S + s) * C;
      for (int c = 0; c < C; ++c) {
        const int xv = zero_point ? (int)(uint8_t)xp[c] - zero_point : (int)xp[c];
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] += xv * (int)wp[j * K + c];
      }
    }
  }
  const int nt = (1 << bits) - 1;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int co = co0 + cg * 16 + j;
    if (co >= COUT) break;
    if (acc_out != nullptr) acc_out[pix * COUT + co] = acc[j];
    if (codes != nullptr) {
      int code = 0;
      for (int k = 0; k < nt; ++k) code += acc[j] >= thr[co * nt + k] ? 1 : 0;
      codes[pix * COUT + co] = (uint8_t)code;
    }
  }
}

// ---- int8 first convolution on the matrix cores ------------------------------------------------------
// Implicit GEMM: rows = 32 consecutive output pixels of one output row (one wave), columns = 64 output
// channels (two 32x32 blocks), K = R*S*C rounded up to k-steps of 32 with v_mfma_i32_32x32x32_i8.
// The filter block [64][T*32] (zero padded) and, per wave, the input patch that the 32 pixels touch
// (R rows x ((31*stride + S) * C) bytes, already minus the zero point, zero outside the image) sit in
// LDS; a small table maps k -> (patch row offset) so that any R, S, C works.
typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef int v16i_t __attribute__((ext_vector_type(16)));

__global__ __launch_bounds__(256) void conv_i8_mfma_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                           const int32_t *__restrict__ thr,
                                                           uint8_t *__restrict__ codes, int32_t *__restrict__ acc_out,
                                                           int B, int H, int W, int C, int COUT, int R, int S,
                                                           int stride, int pad, int Ho, int Wo, int bits,
                                                           int zero_point, int T, int rowlen, int patch_bytes) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int K = R * S * C, KP = T * 32;
  int8_t *wl = reinterpret_cast<int8_t *>(lds);                          // [64][KP]
  uint16_t *tab = reinterpret_cast<uint16_t *>(lds + 64 * KP);           // [KP]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, g = lane >> 5;
  int8_t *patch = reinterpret_cast<int8_t *>(lds + 64 * KP + 2 * KP) + wave * patch_bytes;
  const int co0 = blockIdx.y * 64;

  for (int i = tid; i < 64 * KP; i += 256) {
    const int co = co0 + i / KP, k = i % KP;
    wl[i] = (co < COUT && k < K) ? Wt[(long long)co * K + k] : (int8_t)0;
  }
  for (int k = tid; k < KP; k += 256) tab[k] = k < K ? (uint16_t)((k / (S * C)) * rowlen + (k % (S * C))) : (uint16_t)0xFFFF;

  const int gpr = (Wo + 31) / 32;
  const long long group = (long long)blockIdx.x * 4 + wave;
  const bool active = group < (long long)B * Ho * gpr;
  const int gx = (int)(group % gpr);
  const int oy = (int)((group / gpr) % Ho);
  const int b = (int)(group / ((long long)gpr * Ho));
  const int ox0 = gx * 32;
  if (active) {
    for (int idx = lane; idx < R * rowlen; idx += 64) {
      const int r = idx / rowlen, j = idx % rowlen;
      const int iy = oy * stride + r - pad;
      const int ix = ox0 * stride - pad + j / C;
      int v = 0;
      if (iy >= 0 && iy < H && ix >= 0 && ix < W) {
        const int8_t raw = X[(((long long)b * H + iy) * W + ix) * C + (j % C)];
        v = zero_point ? (int)(uint8_t)raw - zero_point : (int)raw;
      }
      patch[idx] = (int8_t)v;
    }
  }
  __syncthreads();
  if (!active) return;

  v16i_t acc[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nb][r] = 0;
  const int pix_off = li * stride * C;  // this lane's pixel inside the patch row
  for (int t = 0; t < T; ++t) {
    const int kb = t * 32 + g * 16;
    uint32_t a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0;
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const uint32_t off = tab[kb + q * 4 + bb];
        const uint32_t byte = off == 0xFFFFu ? 0u : (uint32_t)(uint8_t)patch[off + pix_off];
        word |= byte << (8 * bb);
      }
      a[q] = word;
    }
    const v4i_t af = {(int)a[0], (int)a[1], (int)a[2], (int)a[3]};
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const v4i_t bf = *reinterpret_cast<const v4i_t *>(wl + (nb * 32 + li) * KP + kb);
      acc[nb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, acc[nb], 0, 0, 0);
    }
  }
  const int nt = (1 << bits) - 1;
  const long long row0 = ((long long)b * Ho + oy) * Wo;
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int co = co0 + nb * 32 + li;
    if (co >= COUT) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int ox = ox0 + 8 * (r >> 2) + 4 * g + (r & 3);
      if (ox >= Wo) continue;
      const long long o = (row0 + ox) * COUT + co;
      const int v = acc[nb][r];
      if (acc_out != nullptr) acc_out[o] = v;
      if (codes != nullptr) {
        int code = 0;
        for (int k = 0; k < nt; ++k) code += v >= thr[co * nt + k] ? 1 : 0;
        codes[o] = (uint8_t)code;
      }
    }
  }
}

// ---- int8 first convolution for C <= 4 (images), dword-per-pixel patch ------------------------------
// Same implicit GEMM as above, but the LDS patch stores every input pixel as one dword
// (c0, c1, c2, c3-or-zero), and K is laid out per filter row as S pixels x 4 bytes rounded up to whole
// k-steps of 32.  A lane's 16 operand bytes of a k-step are then four consecutive, 4-byte aligned
// dwords of the patch -- four LDS dword reads instead of thirty-two byte reads through a k table.  The
// padding bytes of K carry zero weights, so whatever the patch holds there does not matter.
// Output: uint8 codes, int32 sums and / or MSB-first bit-planes [bits][B*Ho*Wo][COUT/32].
__global__ __launch_bounds__(256) void conv_i8_c4_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                         const int32_t *__restrict__ thr,
                                                         uint8_t *__restrict__ codes, int32_t *__restrict__ acc_out,
                                                         uint32_t *__restrict__ planes, int B, int H, int W, int C,
                                                         int COUT, int R, int S, int stride, int pad, int Ho, int Wo,
                                                         int bits, int zero_point, int KR, int PW, int patch_words) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int KP = R * KR * 32;
  const int KPL = KP + 16;  // row pitch in LDS: 16 B of padding spreads the 32 rows over the banks
  int8_t *wl = reinterpret_cast<int8_t *>(lds);  // [64][KPL]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, g = lane >> 5;
  uint32_t *patch = reinterpret_cast<uint32_t *>(lds + 64 * KPL) + wave * patch_words;  // [R][PW] pixels
  const int co0 = blockIdx.y * 64;

  for (int i = tid; i < 64 * KP; i += 256) {
    const int co = co0 + i / KP, k = i % KP;
    const int r = k / (KR * 32), rem = k % (KR * 32);
    const int sx = rem >> 2, c = rem & 3;
    wl[(i / KP) * KPL + k] =
        (co < COUT && sx < S && c < C) ? Wt[(((long long)co * R + r) * S + sx) * C + c] : (int8_t)0;
  }

  __syncthreads();  // filter block staged once per work-group

  // Each wave walks over pixel groups (32 consecutive output pixels of one output row) with a
  // grid-wide stride; its patch is private, so no work-group barrier is needed inside the loop
  // (LDS operations of one wave complete in order).
  const int gpr = (Wo + 31) / 32;
  const long long ngroups = (long long)B * Ho * gpr;
  const int nt = (1 << bits) - 1;
  const long long rows_total = (long long)B * Ho * Wo;
  const int cw32 = COUT >> 5;
  int t0[2], t1[2], t2[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int co = co0 + nb * 32 + li;
    t0[nb] = t1[nb] = t2[nb] = 0x7fffffff;
    if (co < COUT && thr != nullptr && nt <= 3) {
      t0[nb] = thr[co * nt];
      if (nt > 1) t1[nb] = thr[co * nt + 1];
      if (nt > 2) t2[nb] = thr[co * nt + 2];
    }
  }
  for (long long group = (long long)blockIdx.x * 4 + wave; group < ngroups; group += (long long)gridDim.x * 4) {
    const int gx = (int)(group % gpr);
    const int oy = (int)((group / gpr) % Ho);
    const int b = (int)(group / ((long long)gpr * Ho));
    const int ox0 = gx * 32;
    // patch staging, eight pixels per lane at a time: all global byte loads of a batch are issued
    // before the first one is consumed (one memory round trip per batch, not per pixel)
    for (int base = 0; base < patch_words; base += 64 * 8) {
      uint8_t raw[8][4];
      bool inside[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int idx = base + j * 64 + lane;
        const int r = idx / PW, px = idx % PW;
        const int iy = oy * stride + r - pad;
        const int ix = ox0 * stride - pad + px;
        inside[j] = idx < patch_words && r < R && iy >= 0 && iy < H && ix >= 0 && ix < W;
        const int8_t *src = X + (((long long)b * H + (inside[j] ? iy : 0)) * W + (inside[j] ? ix : 0)) * C;
#pragma unroll
        for (int c = 0; c < 4; ++c) raw[j][c] = (c < C && inside[j]) ? (uint8_t)src[c] : (uint8_t)0;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int idx = base + j * 64 + lane;
        uint32_t word = 0;
        if (inside[j]) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (c < C) {
              const int v = zero_point ? (int)raw[j][c] - zero_point : (int)(int8_t)raw[j][c];
              word |= (uint32_t)(uint8_t)(int8_t)v << (8 * c);
            }
          }
        }
        if (idx < patch_words) patch[idx] = word;
      }
    }

    v16i_t acc[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[nb][r] = 0;
    for (int r = 0; r < R; ++r) {
      for (int h = 0; h < KR; ++h) {
        const uint32_t *ap = patch + r * PW + li * stride + h * 8 + g * 4;
        const v4i_t af = {(int)ap[0], (int)ap[1], (int)ap[2], (int)ap[3]};
        const int kb = (r * KR + h) * 32 + g * 16;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const v4i_t bf = *reinterpret_cast<const v4i_t *>(wl + (nb * 32 + li) * KPL + kb);
          acc[nb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, acc[nb], 0, 0, 0);
        }
      }
    }
    const long long row0 = ((long long)b * Ho + oy) * Wo;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int co = co0 + nb * 32 + li;
      const bool co_ok = co < COUT;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ox = ox0 + 8 * (r >> 2) + 4 * g + (r & 3);
        const bool ok = co_ok && ox < Wo;
        const long long o = (row0 + ox) * COUT + co;
        const int v = acc[nb][r];
        int code = 0;
        if (ok && thr != nullptr) {
          if (nt <= 3) {
            code = (v >= t0[nb] ? 1 : 0) + (v >= t1[nb] ? 1 : 0) + (v >= t2[nb] ? 1 : 0);
          } else {
            for (int k = 0; k < nt; ++k) code += v >= thr[co * nt + k] ? 1 : 0;
          }
        }
        if (ok && acc_out != nullptr) acc_out[o] = v;
        if (ok && codes != nullptr) codes[o] = (uint8_t)code;
        if (planes != nullptr) {
          for (int bit = 0; bit < bits; ++bit) {
            const unsigned long long mask = __ballot(ok && ((code >> bit) & 1));
            const uint32_t word = g ? __brev((uint32_t)(mask >> 32)) : __brev((uint32_t)mask);
            if (ok && li == 0) planes[bit * rows_total * cw32 + (row0 + ox) * cw32 + (co >> 5)] = word;
          }
        }
      }
    }
  }
}

template <int I, int N, class F>
__device__ __forceinline__ void static_for_n(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_n<I + 1, N>(f);
  }
}

// w = 16 w + four code bits, first value on top, for bit 1 and bit 0 of a 2-bit code: bit1 = v >= t1,
// bit0 = v >= (bit1 ? t2 : t0).  One block, because a vector instruction must not read a scalar register within
// two instructions of the vector instruction that wrote it, and the compiler does not see into assembly: each
// mask here is used at least three instructions after its compare.
__device__ __forceinline__ void append_int_codes(int v0, int v1, int v2, int v3, const v4i_t &a, const v4i_t &b,
                                                 const v4i_t &c, uint32_t &w1, uint32_t &w0) {
  unsigned long long s0, s1, s2, s3;
  int x0, x1, x2, x3;
  asm("v_cmp_ge_i32_e64 %[s0], %[v0], %[b0]\n\t"
      "v_cmp_ge_i32_e64 %[s1], %[v1], %[b1]\n\t"
      "v_cmp_ge_i32_e64 %[s2], %[v2], %[b2]\n\t"
      "v_cmp_ge_i32_e64 %[s3], %[v3], %[b3]\n\t"
      "v_cndmask_b32_e64 %[x0], %[a0], %[c0], %[s0]\n\t"
      "v_cndmask_b32_e64 %[x1], %[a1], %[c1], %[s1]\n\t"
      "v_cndmask_b32_e64 %[x2], %[a2], %[c2], %[s2]\n\t"
      "v_cndmask_b32_e64 %[x3], %[a3], %[c3], %[s3]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s0]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s1]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[w1], vcc, %[w1], %[w1], %[s3]\n\t"
      "v_cmp_ge_i32_e64 %[s0], %[v0], %[x0]\n\t"
      "v_cmp_ge_i32_e64 %[s1], %[v1], %[x1]\n\t"
      "v_cmp_ge_i32_e64 %[s2], %[v2], %[x2]\n\t"
      "v_cmp_ge_i32_e64 %[s3], %[v3], %[x3]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s0]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s1]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s2]\n\t"
      "v_addc_co_u32_e64 %[w0], vcc, %[w0], %[w0], %[s3]"
      : [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2), [s3] "=&s"(s3), [x0] "=&v"(x0), [x1] "=&v"(x1), [x2] "=&v"(x2),
        [x3] "=&v"(x3), [w1] "+v"(w1), [w0] "+v"(w0)
      : [v0] "v"(v0), [v1] "v"(v1), [v2] "v"(v2), [v3] "v"(v3), [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]),
        [a3] "v"(a[3]), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]), [c0] "v"(c[0]), [c1] "v"(c[1]),
        [c2] "v"(c[2]), [c3] "v"(c[3])
      : "vcc");
}

// ---- int8 first convolution for images, filter rows taken straight from the image bytes ------------
// In NHWC memory the S pixels x C channels under one filter row are S*C consecutive bytes, so K is laid
// out per filter row as that byte run, padded with zero weights to whole 16-byte halves (HPR halves per
// row); the halves of all R rows are numbered consecutively and k-step ks consumes halves 2ks (lane
// half 0) and 2ks+1 (lane half 1).  A wave works on a block of NSETS * 32 output pixels, 2^LW wide: its patch is
// the image-row segments under the block, copied to LDS as aligned dwords -- no per-pixel repacking -- with
// the zero point removed by an XOR (x - 128 == x ^ 0x80 as int8) and out-of-image dwords set to zero.
// A lane's 16 operand bytes start at byte lead + pixel*stride*C + 16*half of its row segment: five
// aligned dword reads and four v_alignbyte (one 16-byte read that is not aligned takes 48 clocks of the LDS, these
// about 20).  NKS > 0: the number of k-steps is known, the loop is unrolled and a lane keeps the patch address of each step.
// Weights are the first operand, so a lane of the accumulator owns one output pixel and its registers hold
// channels: code bits are appended to the lane's own words, thresholds come from a table in LDS.  Filter row
// 8q + 4h + j of a block of 32 holds channel 16h + 4q + j, which gives lane half h the channels 16h .. 16h + 15 in
// order; one half-wave swap joins the two halves of both planes' words.
// What bounds it: LDS reads, then vector issue (five operations per value: compare, select, compare, two appends).  Blocks
// instead of 32 pixels of a row (maps of 112 and 56 pixels left the fourth and second part of a row half empty, and a
// patch of R rows is loaded for 32 pixels), 64 pixels to every read of the filter and of the thresholds, patches of as many
// slots as they have, and a filter staged without vector work (a lane per channel: half, filter row and mask are scalar, all
// loads of a wave at once): us in graph replay at batch 8 / 64, 224x224x3, 7x7 stride 2 to 64 channels 10.4 -> 8.8 / 31.6
// -> 25.1, 3x3 stride 2 to 96 12.0 -> 7.7 / 41.9 -> 28.0, 11x11 stride 4 to 64 12.9 -> 9.8 / 25.9 -> 19.4.
// Two sets of 32 pixels from two blocks per unit (7x7 at batch 8 9.8 with one, 9.5 with two; 3x3 to 128 channels on 32x32 maps
// at batch 64 9.0 and 7.2), below that one, with the filter block in registers (7x7 at batch 8 10.6 without).
// Requires C <= 4, (W*C) % 4 == 0, X 4-byte aligned, bits <= 2, COUT % 32 == 0.
// NWAV waves per work-group share one filter block in LDS (each wave has its own patch and walks its
// own pixel blocks): eight waves where the filter block is large, so that its LDS cost per wave halves
// and four waves per SIMD stay resident (two work-groups per compute unit: the register budget of that
// variant is held to 128 by its launch bounds).
constexpr int kRowsTable = 3 * 64 * 4;  // bytes of thresholds in LDS, [3][64]
// bytes of a wave's patch of `dwords` dwords: the last pixel's last half may end 20 bytes past the segment
__host__ __device__ inline int rows_patch_bytes(int dwords) { return (4 * dwords + 32 + 15) & ~15; }

typedef v4i_t v4i_bytes __attribute__((aligned(1)));

template <int NKS, int NSETS, bool WREG, int NSLOT, int NWAV>
__global__ __launch_bounds__(64 * NWAV, WREG ? 3 : 4) void conv_i8_rows_kernel(const uint8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                           const int32_t *__restrict__ thr,
                                                           uint32_t *__restrict__ planes, int B, int H, int W, int C,
                                                           int COUT, int R, int S, int stride, int pad, int Ho, int Wo,
                                                           int bits, uint32_t xor_mask, int HPR, int PR, int NDW, int LW,
                                                           uint32_t magic_gpr, uint32_t magic_gpc, uint32_t magic_ndw,
                                                           uint32_t magic_hpr) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // n / d by multiply-high with ceil(2^32 / d) where the launcher found it exact (magic != 0)
  auto quot = [](uint32_t n, uint32_t d, uint32_t magic) { return magic != 0 ? __umulhi(n, magic) : (d == 1 ? n : n / d); };
  const int NH = R * HPR;
  const int nks = (NH + 1) / 2;
  const int KB = nks * 32, KPL = KB + 16;
  int *table = reinterpret_cast<int *>(lds);                  // [3][64]
  int8_t *wl = reinterpret_cast<int8_t *>(lds + kRowsTable);  // [64][KPL]
  // the wave index is the same in all 64 lanes: as a scalar it keeps the pixel-block arithmetic below
  // (block -> image, output row, image row addresses) on the scalar unit
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int npatch = PR * NDW;
  uint8_t *patch = lds + kRowsTable + 64 * KPL + wave * rows_patch_bytes(npatch);
  const int co0 = blockIdx.y * 64;
  const int SC = S * C;

  const int PX = 1 << LW, PY = 32 >> LW;  // of a set
  // filter block -> LDS: a lane per channel, a wave per 16-byte half, so that the half's place in the filter and the bytes
  // of it that hold weights are scalar.  The halves of a wave are requested before the first LDS store (all of them where
  // the number of k-steps is known).  Loads are unaligned; the filter's last 16 bytes are loaded instead of bytes past it.
  constexpr int NT = NKS > 0 ? (NKS * 2 + NWAV - 1) / NWAV : 4;
  {
    const int co = co0 + lane;
    const uint32_t live = co < COUT ? 0xffffffffu : 0u;
    const uint32_t top = (uint32_t)(COUT * R * SC) - 16u, base = (uint32_t)(min(co, COUT - 1) * R * SC);
    const int row = (lane & 0x23) | ((lane & 0xc) << 1) | ((lane & 0x10) >> 2);
    for (int h0 = wave; h0 < 2 * nks; h0 += NT * NWAV) {
      v4i_t w[NT];
      uint32_t past[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const int hh = h0 + u * NWAV;
        const int r = min((int)quot((uint32_t)hh, (uint32_t)HPR, magic_hpr), R - 1);
        const uint32_t off = min(base + (uint32_t)(r * SC + min(hh - r * HPR, HPR - 1) * 16), top + 15u), at = min(off, top);
        past[u] = off - at;
        w[u] = *reinterpret_cast<const v4i_bytes *>(Wt + at);
      }
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const int hh = h0 + u * NWAV;
        if (hh < 2 * nks) {
          const int r = (int)quot((uint32_t)hh, (uint32_t)HPR, magic_hpr);
          const int nvalid = r < R ? min(SC - (hh - r * HPR) * 16, 16) : 0;
          uint32_t v[5] = {(uint32_t)w[u][0], (uint32_t)w[u][1], (uint32_t)w[u][2], (uint32_t)w[u][3], 0u};
          if (__any(past[u] != 0)) {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const bool drop = (past[u] >> 2) > (uint32_t)i;
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = drop ? v[q + 1] : v[q];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = __builtin_amdgcn_alignbyte(v[q + 1], v[q], past[u] & 3u);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int nb = min(max(nvalid - 4 * q, 0), 4);
            v[q] &= live & (nb == 4 ? 0xffffffffu : (1u << (8 * nb)) - 1u);
          }
          *reinterpret_cast<uint4 *>(wl + row * KPL + hh * 16) = make_uint4(v[0], v[1], v[2], v[3]);
        }
      }
    }
  }
  const int nt = (1 << bits) - 1;
  if (tid < 3 * 64) {
    const int co = co0 + (tid & 63), k = tid >> 6;
    table[tid] = co < COUT ? thr[co * nt + (k < nt ? k : 0)] : 0x7fffffff;
  }
  __syncthreads();

  // this lane's pixel of set 0 (bytes into the patch) and the distance to the pixels of the next set
  const int px = li & (PX - 1), py = li >> LW;
  const int lead = (-pad * C) & 3;  // (a block's first byte is a multiple of 8 * stride * C beyond the padding)
  const int rowpitch = NDW * 4;
  const int first = lead + px * stride * C + py * stride * rowpitch;
  const uint32_t *mine = reinterpret_cast<const uint32_t *>(patch) + (first >> 2);
  const uint32_t sh = (uint32_t)first & 3u;
  const int set_bytes = PY * stride * rowpitch;
  constexpr int NW = NKS > 0 ? NKS : 1;
  v4i_t wreg[2][WREG ? NW : 1];
  int koff[NW];  // byte offset of this lane's half of k-step ks
  if (NKS > 0) {
#pragma unroll
    for (int ks = 0; ks < NW; ++ks) {
#pragma unroll
      for (int nb = 0; nb < (WREG ? 2 : 0); ++nb)
        wreg[nb][WREG ? ks : 0] = *reinterpret_cast<const v4i_t *>(wl + (nb * 32 + li) * KPL + ks * 32 + g * 16);
      const int hh = 2 * ks + g;
      const int r = min((int)quot((uint32_t)hh, (uint32_t)HPR, magic_hpr), R - 1);
      koff[ks] = r * rowpitch + (hh - (int)quot((uint32_t)hh, (uint32_t)HPR, magic_hpr) * HPR) * 16;
    }
  }

  const int gpr = (Wo + PX - 1) >> LW, gpc = (Ho + NSETS * PY - 1) / (NSETS * PY);
  const long long rows_total = (long long)B * Ho * Wo;
  const int cw32 = COUT >> 5;
  const int rowbytes = W * C;

  // Patch element idx = slot * 64 + lane is dword d of row segment r, the same for every block:
  // (r, d) is decoded once.  The raw dwords of the next block are requested before the current
  // one is computed (patches of up to 64 * NSLOT dwords; larger ones are staged in place, chunk by chunk).
  const bool prefetch = npatch <= 64 * NSLOT;
  // rd[j]: row segment r in the upper half-word, byte offset 4*d in the lower one; r = NO_ROW marks a
  // slot past the end of the patch (it then fails the row test of every block)
  constexpr int NO_ROW = 0x7fff;
  auto slot_code = [&](int idx) {
    const int r = (int)quot((uint32_t)idx, (uint32_t)NDW, magic_ndw);
    return idx < npatch ? ((r << 16) | (4 * (idx - r * NDW))) : (NO_ROW << 16);
  };
  int rd[NSLOT];
#pragma unroll
  for (int j = 0; j < NSLOT; ++j) rd[j] = slot_code(j * 64 + lane);
  // Loads go through a descriptor of the image (the launcher checks H * W * C < 2^31, W * C < 2^24 and H + pad < NO_ROW),
  // a dword outside the image has the offset 0xffffffff; raw_ok[j]: slot j lies inside.  A load whose value is used inside
  // a branch on its predicate would make the compiler wait for it there, one memory round trip per slot.
  uint32_t raw[NSLOT];
  bool raw_ok[NSLOT];
  struct Origin {
    int b, oy0, ox0;
  };
  auto origin = [&](uint32_t blk) {
    const uint32_t t = quot(blk, (uint32_t)gpr, magic_gpr);
    Origin o;
    o.ox0 = (int)(blk - t * (uint32_t)gpr) << LW;
    o.b = (int)quot(t, (uint32_t)gpc, magic_gpc);
    o.oy0 = (int)(t - (uint32_t)o.b * (uint32_t)gpc) * (NSETS * PY);
    return o;
  };
  auto image = [&](const Origin &o) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(X + (long long)o.b * H * rowbytes), 0, H * rowbytes, 0x00020000);
  };
  auto load_slot = [&](__amdgpu_buffer_rsrc_t img, int ybase, int sbase, int code, uint32_t &word, bool &inside) {
    const int iy = ybase + (code >> 16);
    const int sb = sbase + (code & 0xffff);
    inside = (uint32_t)iy < (uint32_t)H && (uint32_t)sb < (uint32_t)rowbytes;
    const int off = iy * rowbytes + sb;
    word = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(img, inside ? off : -1, 0, 0);
  };
  auto request = [&](uint32_t blk) {
    const Origin o = origin(blk);
    const auto img = image(o);
    const int sbase = ((o.ox0 * stride - pad) * C) & ~3;  // two's complement: rounds towards minus infinity
    const int ybase = o.oy0 * stride - pad;
#pragma unroll
    for (int j = 0; j < NSLOT; ++j) load_slot(img, ybase, sbase, rd[j], raw[j], raw_ok[j]);
  };
  uint32_t *pdw = reinterpret_cast<uint32_t *>(patch) + lane;
  auto publish = [&]() {
#pragma unroll
    for (int j = 0; j < NSLOT; ++j)
      if (j * 64 + 64 <= npatch || j * 64 + lane < npatch) pdw[j * 64] = raw_ok[j] ? raw[j] ^ xor_mask : 0u;
  };
  // patches larger than the slots: staged in place, one dword per lane and round trip
  auto stage_in_place = [&](uint32_t blk) {
    const Origin o = origin(blk);
    const auto img = image(o);
    const int sbase = ((o.ox0 * stride - pad) * C) & ~3, ybase = o.oy0 * stride - pad;
#pragma unroll 1
    for (int idx = lane; idx < npatch; idx += 64) {
      uint32_t word;
      bool inside;
      load_slot(img, ybase, sbase, slot_code(idx), word, inside);
      reinterpret_cast<uint32_t *>(patch)[idx] = inside ? word ^ xor_mask : 0u;
    }
  };

  // (the launcher keeps the number of blocks below 2^31: 32-bit index arithmetic)
  const uint32_t gstep = gridDim.x * (uint32_t)NWAV, ng = (uint32_t)B * (uint32_t)(gpr * gpc);
  uint32_t block = blockIdx.x * (uint32_t)NWAV + (uint32_t)wave;
  if (prefetch && block < ng) request(block);
  for (; block < ng; block += gstep) {
    if (prefetch) {
      publish();
      if (block + gstep < ng) request(block + gstep);
    } else {
      stage_in_place(block);
    }

    v16i_t acc[NSETS][2];
#pragma unroll
    for (int st = 0; st < NSETS; ++st)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[st][nb][r] = 0;
    auto k_step = [&](int ks, int off, int rs) {
      v4i_t w[2], af[NSETS];
#pragma unroll
      for (int st = 0; st < NSETS; ++st) {
        const uint32_t *wp = mine + ((off + st * set_bytes) >> 2);
        const uint32_t w0 = wp[0], w1 = wp[1], w2 = wp[2], w3 = wp[3], w4 = wp[4];
        af[st][0] = (int)__builtin_amdgcn_alignbyte(w1, w0, sh);
        af[st][1] = (int)__builtin_amdgcn_alignbyte(w2, w1, sh);
        af[st][2] = (int)__builtin_amdgcn_alignbyte(w3, w2, sh);
        af[st][3] = (int)__builtin_amdgcn_alignbyte(w4, w3, sh);
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        if constexpr (WREG) w[nb] = wreg[nb][rs];
        else w[nb] = *reinterpret_cast<const v4i_t *>(wl + (nb * 32 + li) * KPL + ks * 32 + g * 16);
      }
#pragma unroll
      for (int st = 0; st < NSETS; ++st)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) acc[st][nb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[nb], af[st], acc[st][nb], 0, 0, 0);
    };
    if (NKS > 0) {
#pragma unroll
      for (int ks = 0; ks < NW; ++ks) k_step(ks, koff[ks], ks);
    } else {
      int r = 0, h = g;  // half index 2ks + g = r * HPR + h
      for (int ks = 0; ks < nks; ++ks) {
        while (h >= HPR) {
          h -= HPR;
          ++r;
        }
        k_step(ks, min(r, R - 1) * rowpitch + h * 16, 0);
        h += 2;
      }
    }

    // ---- thresholds -> bit-plane words: lane half 0 ends with the pixel's word of plane 0, half 1 of plane 1 ----
    // wait states between the last matrix instruction and a vector instruction that reads its result (19 for sixteen
    // passes): the compiler adds them for instructions it can see, not for the assembly of append_int_codes
#pragma unroll
    for (int st = 0; st < NSETS; ++st) asm volatile("" : "+v"(acc[st][0]), "+v"(acc[st][1]));
    asm volatile("s_nop 15\n\ts_nop 7");
#pragma unroll
    for (int st = 0; st < NSETS; ++st) asm volatile("" : "+v"(acc[st][0]), "+v"(acc[st][1]));
    __builtin_amdgcn_sched_barrier(0);  // (keeps the threshold reads from piling up in registers)
    const int *tab = table + 16 * g;
    uint32_t word[NSETS][2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      uint32_t w0[NSETS], w1[NSETS];
#pragma unroll
      for (int st = 0; st < NSETS; ++st) w0[st] = w1[st] = 0;
      static_for_n<0, 4>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const v4i_t a = *reinterpret_cast<const v4i_t *>(tab + nb * 32 + 4 * q);
        const v4i_t b1 = *reinterpret_cast<const v4i_t *>(tab + 64 + nb * 32 + 4 * q);
        const v4i_t c2 = *reinterpret_cast<const v4i_t *>(tab + 128 + nb * 32 + 4 * q);
#pragma unroll
        for (int st = 0; st < NSETS; ++st)
          append_int_codes(acc[st][nb][4 * q], acc[st][nb][4 * q + 1], acc[st][nb][4 * q + 2], acc[st][nb][4 * q + 3], a, b1, c2,
                           w1[st], w0[st]);
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int st = 0; st < NSETS; ++st) {
        const auto s = __builtin_amdgcn_permlane32_swap(w0[st], w1[st], false, false);
        word[st][nb] = (s[0] << 16) | s[1];
      }
    }
    const Origin o = origin(block);
    const int plane = g;
#pragma unroll
    for (int st = 0; st < NSETS; ++st) {
      const int ox = o.ox0 + px, oy = o.oy0 + st * PY + py;
      if (ox < Wo && oy < Ho && plane < bits) {
        uint32_t *dst = planes + plane * rows_total * cw32 + (((long long)o.b * Ho + oy) * Wo + ox) * cw32 + (co0 >> 5);
        if ((cw32 & 1) == 0) {
          *reinterpret_cast<uint2 *>(dst) = make_uint2(word[st][0], word[st][1]);
        } else {
          dst[0] = word[st][0];
          if (co0 + 32 < COUT) dst[1] = word[st][1];
        }
      }
    }
  }
}

// ---- max-pool directly on bit-planes ----------------------------------------------------------------
// in: [bits][B*H*W][cw] -> out: [bits][B*Ho*Wo][cw]; the maximum of two multi-bit codes is computed for
// 32 channels at once with bitwise logic (compare from the top plane down).
// NB: planes held in registers (2 for the usual one- and two-bit codes, else 8).  VEC: channel words per
// thread; 2 (64-bit loads and stores, an even number of channel words, 3x3 windows on at most two planes)
// halves the number of load instructions, which is what bounds this kernel.
template <int NB, int VEC = 1>
__global__ __launch_bounds__(256) void pool_planes_kernel(const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
                                                          int B, int H, int W, int cw, int bits, int win, int stride,
                                                          int pad, int Ho, int Wo) {
  const long long rows_in = (long long)B * H * W, rows_out = (long long)B * Ho * Wo;
  const int cwv = cw / VEC;  // threads per output pixel
  const long long total = rows_out * cwv;
  const bool small = total < 0x7fffffffLL;  // 32-bit index arithmetic (64-bit divisions cost ~100 instructions)
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    int wi, ox, oy, b;
    long long row;
    if (small) {
      const uint32_t iu = (uint32_t)i, r32 = iu / (uint32_t)cwv;
      wi = (int)(iu - r32 * (uint32_t)cwv) * VEC;
      const uint32_t t = r32 / (uint32_t)Wo;
      ox = (int)(r32 - t * (uint32_t)Wo);
      b = (int)(t / (uint32_t)Ho);
      oy = (int)(t - (uint32_t)b * (uint32_t)Ho);
      row = r32;
    } else {
      wi = (int)(i % cwv) * VEC;
      row = i / cwv;
      ox = (int)(row % Wo);
      oy = (int)((row / Wo) % Ho);
      b = (int)(row / ((long long)Wo * Ho));
    }
    if constexpr (VEC == 2) {
      // two channel words per thread: the same window logic on both halves of 64-bit loads
      uint2 v[9][2];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int iy = oy * stride + t / 3 - pad, ix = ox * stride + t % 3 - pad;
        const bool ok = iy >= 0 && iy < H && ix >= 0 && ix < W;
        const long long rin = ((long long)b * H + iy) * W + ix;
#pragma unroll
        for (int p = 0; p < 2; ++p)
          v[t][p] = (ok && p < bits) ? *reinterpret_cast<const uint2 *>(in + p * rows_in * cw + rin * cw + wi)
                                     : make_uint2(0u, 0u);
      }
      uint32_t m0x = 0, m0y = 0, m1x = 0, m1y = 0;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const uint32_t ltx = (v[t][1].x & ~m1x) | (~(v[t][1].x ^ m1x) & v[t][0].x & ~m0x);
        const uint32_t lty = (v[t][1].y & ~m1y) | (~(v[t][1].y ^ m1y) & v[t][0].y & ~m0y);
        m0x = (m0x & ~ltx) | (v[t][0].x & ltx);
        m1x = (m1x & ~ltx) | (v[t][1].x & ltx);
        m0y = (m0y & ~lty) | (v[t][0].y & lty);
        m1y = (m1y & ~lty) | (v[t][1].y & lty);
      }
      *reinterpret_cast<uint2 *>(out + row * cw + wi) = make_uint2(m0x, m0y);
      if (bits > 1) *reinterpret_cast<uint2 *>(out + rows_out * cw + row * cw + wi) = make_uint2(m1x, m1y);
      continue;
    }
    uint32_t m[NB];
#pragma unroll
    for (int p = 0; p < NB; ++p) m[p] = 0;
    if (NB == 2 && win == 3) {
      // the usual 3x3 window on one- or two-bit codes: all eighteen loads are requested before the
      // first compare (out-of-image taps read as code 0, the identity of the maximum)
      uint32_t v[9][2];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int iy = oy * stride + t / 3 - pad, ix = ox * stride + t % 3 - pad;
        const bool ok = iy >= 0 && iy < H && ix >= 0 && ix < W;
        const long long rin = ((long long)b * H + iy) * W + ix;
#pragma unroll
        for (int p = 0; p < 2; ++p) v[t][p] = (ok && p < bits) ? in[p * rows_in * cw + rin * cw + wi] : 0u;
      }
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        // per channel: v > m  <=>  (v1 & ~m1) | (~(v1 ^ m1) & v0 & ~m0)
        const uint32_t lt = (v[t][1] & ~m[1]) | (~(v[t][1] ^ m[1]) & v[t][0] & ~m[0]);
        m[0] = (m[0] & ~lt) | (v[t][0] & lt);
        m[1] = (m[1] & ~lt) | (v[t][1] & lt);
      }
    } else
    for (int r = 0; r < win; ++r) {
      const int iy = oy * stride + r - pad;
      if (iy < 0 || iy >= H) continue;
      for (int sx = 0; sx < win; ++sx) {
        const int ix = ox * stride + sx - pad;
        if (ix < 0 || ix >= W) continue;
        const long long rin = ((long long)b * H + iy) * W + ix;
        uint32_t v[NB];
#pragma unroll
        for (int p = 0; p < NB; ++p) v[p] = p < bits ? in[p * rows_in * cw + rin * cw + wi] : 0u;
        uint32_t gt = 0, lt = 0;  // per channel: m > v decided / m < v decided
#pragma unroll
        for (int p = NB - 1; p >= 0; --p) {
          const uint32_t diff = m[p] ^ v[p], open = ~(gt | lt);
          gt |= open & diff & m[p];
          lt |= open & diff & v[p];
        }
#pragma unroll
        for (int p = 0; p < NB; ++p) m[p] = (m[p] & ~lt) | (v[p] & lt);
      }
    }
#pragma unroll
    for (int p = 0; p < NB; ++p)
      if (p < bits) out[p * rows_out * cw + row * cw + wi] = m[p];
  }
}

// ---- max-pool on codes + bit-plane packing ---------------------------------------------------------
// codes: [B][H][W][C] uint8 -> planes [bits][B*Ho*Wo][cpad/32], window win x win, stride, pad
// (out-of-image taps ignored).  One wave per (pixel, 64-channel group).
__global__ __launch_bounds__(256) void pool_pack_kernel(const uint8_t *__restrict__ codes, uint32_t *__restrict__ planes,
                                                        int B, int H, int W, int C, int cpad, int bits, int win,
                                                        int stride, int pad, int Ho, int Wo) {
  const int lane = threadIdx.x & 63;
  const int cw = cpad >> 5;
  const int groups = (cpad + 63) >> 6;
  const long long rows = (long long)B * Ho * Wo;
  const long long total = rows * groups;
  for (long long gidx = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); gidx < total; gidx += (long long)gridDim.x * 4) {
    const long long row = gidx / groups;
    const int c = (int)(gidx % groups) * 64 + lane;
    const int ox = (int)(row % Wo), oy = (int)((row / Wo) % Ho), b = (int)(row / ((long long)Wo * Ho));
    int v = 0;
    if (c < C) {
      for (int r = 0; r < win; ++r) {
        const int iy = oy * stride + r - pad;
        if (iy < 0 || iy >= H) continue;
        for (int s = 0; s < win; ++s) {
          const int ix = ox * stride + s - pad;
          if (ix < 0 || ix >= W) continue;
          v = max(v, (int)codes[(((long long)b * H + iy) * W + ix) * C + c]);
        }
      }
    }
    for (int bit = 0; bit < bits; ++bit) {
      const unsigned long long mask = __ballot((v >> bit) & 1);
      const uint32_t word = (lane < 32) ? __brev((uint32_t)mask) : __brev((uint32_t)(mask >> 32));
      const int wi = c >> 5;
      if ((lane & 31) == 0 && wi < cw) planes[bit * rows * cw + row * cw + wi] = word;
    }
  }
}

// ---- packed codes -> int8 values (optionally summed over `group` consecutive rows) ---------------
// planes: [bits][rows][cpad/32];  out[r][c] = (sum_{j<group} code[r*group + j][c]) >> shift, int8.
// group = 1, shift = 0: plain unpacking.  group = H*W: global pooling of a feature map.
// JP (a power of two <= 64) consecutive lanes share one output element and split its `group` rows;
// their partial sums meet in a butterfly reduction.
__global__ __launch_bounds__(256) void unpack_sum_kernel(const uint32_t *__restrict__ planes, int8_t *__restrict__ out,
                                                         long long rows_out, int group, int C, int cpad, int bits,
                                                         int shift, int JP) {
  const int cw = cpad >> 5;
  const long long rows_in = rows_out * group;
  const long long total = rows_out * C;
  const int part = threadIdx.x & (JP - 1);
  const long long nthreads = (long long)gridDim.x * blockDim.x;
  // every lane of a JP-group runs the same number of iterations (the shuffles need all of them)
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t / JP < total; t += nthreads) {
    const long long i = t / JP;
    long long r;
    int c;
    if (total < 0x7fffffffLL) {
      const uint32_t r32 = (uint32_t)i / (uint32_t)C;
      c = (int)((uint32_t)i - r32 * (uint32_t)C);
      r = r32;
    } else {
      r = i / C;
      c = (int)(i % C);
    }
    const int sh = 31 - (c & 31);
    int sum = 0;
    for (int j = part; j < group; j += JP) {
      const long long rin = r * group + j;
      int code = 0;
      for (int b = 0; b < bits; ++b) code |= (int)((planes[b * rows_in * cw + rin * cw + (c >> 5)] >> sh) & 1u) << b;
      sum += code;
    }
    for (int off = JP >> 1; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (part == 0) out[i] = (int8_t)min(127, sum >> shift);
  }
}

// Pooled variant of the above for group >= 8 (global pooling of a feature map): one wave per (output
// row, 32-channel word).  Lane j holds pixel j of the group (64 pixels per pass): one load per plane
// and lane, all in flight together; the sum over the pixels of channel c's bit in plane b is the
// population count of a wave-wide compare, accumulated in scalar registers.  Lane c stores channel c.
__global__ __launch_bounds__(256) void pool_sum_kernel(const uint32_t *__restrict__ planes, int8_t *__restrict__ out,
                                                       long long rows_out, int group, int C, int cpad, int bits,
                                                       int shift) {
  const int lane = threadIdx.x & 63;
  const int cw = cpad >> 5;
  const long long task = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (task >= rows_out * cw) return;  // the whole wave
  const long long r = task / cw;
  const int w = (int)(task - r * cw);
  const long long rows_in = rows_out * group;
  int cnt[32];
#pragma unroll
  for (int c = 0; c < 32; ++c) cnt[c] = 0;
  for (int j0 = 0; j0 < group; j0 += 64) {
    const int j = j0 + lane;
    uint32_t wv[8];
#pragma unroll
    for (int b = 0; b < 8; ++b)
      wv[b] = (b < bits && j < group) ? planes[(long long)b * rows_in * cw + (r * group + j) * cw + w] : 0u;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (b < bits) {  // same for the whole wave
        static_for_n<0, 32>([&](auto cc) {
          constexpr int c = decltype(cc)::value;
          cnt[c] += __popcll(__ballot((wv[b] >> (31 - c)) & 1u)) << b;
        });
      }
    }
  }
  int mine = 0;
  static_for_n<0, 32>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    if (lane == c) mine = cnt[c];
  });
  const int ch = w * 32 + lane;
  if (lane < 32 && ch < C) out[r * C + ch] = (int8_t)min(127, mine >> shift);
}

// ---- int8 classifier: out[b][n] = scale[n] * sum_k X[b][k] * Wt[n][k] + bias[n] -----------------
// One wave per (group of NN output features, group of four batch rows): lanes stride over K in dwords
// (v_dot4_i32_i8 on four int8 pairs), every operand dword is used NN or four times, then wave64
// butterfly reductions.  K % 4 != 0 (or unaligned rows) falls back to byte loads.
// NN output features x 4 batch rows per wave (NN = 4 when the batch is large enough to make operand
// re-reads the cost, else 1: more waves for small batches).
template <int NN>
__global__ __launch_bounds__(256) void fc_i8_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                    const float *__restrict__ scale, const float *__restrict__ bias,
                                                    float *__restrict__ out, int32_t *__restrict__ acc_out, int Bn,
                                                    int N, int K, int vec_ok) {
  const int lane = threadIdx.x & 63;
  const int bgroups = (Bn + 3) >> 2, ngroups = (N + NN - 1) / NN;
  const long long wid = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= (long long)ngroups * bgroups) return;
  const int n0 = (int)(wid % ngroups) * NN;
  const int b0 = (int)(wid / ngroups) * 4;
  int acc[NN][4];
#pragma unroll
  for (int i = 0; i < NN; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0;
  // the affine map of this wave's features, requested before the K loop (clamped index, no branch) so
  // that the epilogue does not pay a memory round trip per output
  float sc[NN], bi[NN];
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    const int n = min(n0 + i, N - 1);
    sc[i] = scale[n];
    bi[i] = bias[n];
  }
  if (vec_ok) {
    // four independent iterations in flight: a long K would otherwise be one memory round trip per step
#pragma unroll 4
    for (int k4 = lane; k4 < (K >> 2); k4 += 64) {
      int wv[NN], xv[4];
#pragma unroll
      for (int i = 0; i < NN; ++i)
        wv[i] = n0 + i < N ? reinterpret_cast<const int *>(Wt + (long long)(n0 + i) * K)[k4] : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xv[j] = b0 + j < Bn ? reinterpret_cast<const int *>(X + (long long)(b0 + j) * K)[k4] : 0;
#pragma unroll
      for (int i = 0; i < NN; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_sdot4(xv[j], wv[i], acc[i][j], false);
    }
  } else {
    for (int k = lane; k < K; k += 64) {
#pragma unroll
      for (int i = 0; i < NN; ++i) {
        const int wv = n0 + i < N ? (int)Wt[(long long)(n0 + i) * K + k] : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (b0 + j < Bn) acc[i][j] += (int)X[(long long)(b0 + j) * K + k] * wv;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NN; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) acc[i][j] += __shfl_xor(acc[i][j], off, 64);
      if (lane == 0 && b0 + j < Bn && n0 + i < N) {
        const long long o = (long long)(b0 + j) * N + n0 + i;
        if (acc_out != nullptr) acc_out[o] = acc[i][j];
        out[o] = (float)acc[i][j] * sc[i] + bi[i];
      }
    }
}

hipError_t launch_conv_i8_bn(const int8_t *X, const int8_t *Wt, const int32_t *thr, uint8_t *codes, int32_t *acc_out,
                             uint32_t *planes, int B, int H, int W, int C, int COUT, int R, int S, int stride, int pad,
                             int bits, int zero_point, hipStream_t s) {
  const int Ho = (H + 2 * pad - R) / stride + 1, Wo = (W + 2 * pad - S) / stride + 1;
  const long long npix = (long long)B * Ho * Wo;
  const long long groups = (long long)B * Ho * ((Wo + 31) / 32);
  dim3 grid((unsigned)((groups + 3) / 4), (unsigned)((COUT + 63) / 64));
  if (C <= 4 && planes != nullptr && codes == nullptr && acc_out == nullptr && bits <= 2 && (COUT % 32) == 0 &&
      groups < 0x7fffffffLL && (long long)H * W * C < 0x7fffffffLL && (long long)W * C < (1 << 24) &&
      (long long)H + pad < 0x7fff && (long long)COUT * R * S * C < 0x7fffffffLL && ((W * C) % 4) == 0 && (reinterpret_cast<uintptr_t>(X) & 3u) == 0 && (zero_point == 0 || zero_point == 128) &&
      thr != nullptr) {
    // image rows consumed as bytes (no repacking): see conv_i8_rows_kernel
    const int HPR = (S * C + 15) / 16;
    const int nks = (R * HPR + 1) / 2;
    int cus = 0, dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    if (cus <= 0) cus = 256;
    // pixel blocks 16 or 8 wide, whichever needs fewer of them, then the smaller patch
    struct Shape {
      int lw, pr, ndw, gpr, gpc;
    };
    auto shape = [&](int sets, int lw) {
      const int px = 1 << lw, py = sets * (32 >> lw);
      return Shape{lw, (py - 1) * stride + R, (3 + ((px - 1) * stride + S) * C + 3) / 4, (Wo + px - 1) / px, (Ho + py - 1) / py};
    };
    auto best = [&](int sets) {
      const Shape w = shape(sets, 4), n = shape(sets, 3);
      const long long bw = (long long)w.gpr * w.gpc, bn = (long long)n.gpr * n.gpc;
      return bw < bn || (bw == bn && w.pr * w.ndw <= n.pr * n.ndw) ? w : n;
    };
    const bool wide_patch = nks > 8;
    const int nwav = wide_patch ? 8 : 4;
    auto patch_of = [](const Shape &c) { return c.pr * c.ndw; };
    auto blocks_of = [&](const Shape &c) { return (long long)B * c.gpr * c.gpc; };
    auto lds_of = [&](const Shape &c) { return kRowsTable + (size_t)64 * (nks * 32 + 16) + (size_t)nwav * rows_patch_bytes(patch_of(c)); };
    const size_t lds_limit = wide_patch ? 82 * 1024 : 64 * 1024;
    Shape sh = best(2);
    const bool two = !wide_patch && patch_of(sh) <= 64 * (nks == 2 ? 4 : 6) && blocks_of(sh) >= 2 * cus;
    if (!two) sh = best(1);
    // A patch beyond the slots of the form for the number of k-steps is staged in place, and strides beyond the filter put rows
    // and pixels that no output reads between those of a block.  The shape that stages least, 32 pixels of a row among them, and a
    // form of 8 or 18 slots, where that is less by more than the form for the number of k-steps saves (a wave's patch, times the
    // rounds of sixteen waves a unit; 7x7 stride 32 on one channel, 96x96 at batch 64: 54 us in blocks of 16x2 pixels, 12 in
    // rows; 4x4 stride 4 on four channels at batch 64, 516 dwords of 520: 15.3 so, 11.6 in place), or where only it fits the LDS.
    const int own_slots = 64 * (wide_patch ? 12 : nks == 7 || nks == 2 ? 6 : 8);
    bool more = false;
    if (!two && patch_of(sh) > own_slots) {
      auto cost = [&](const Shape &c) { return std::max(blocks_of(c), 16LL * cus) * patch_of(c); };
      auto staged = [&](const Shape &c) { return (blocks_of(c) + 16 * cus - 1) / (16 * cus) * patch_of(c); };
      Shape least = sh;
      for (const Shape &c : {shape(1, 3), shape(1, 4), shape(1, 5)})
        if (lds_of(c) <= lds_limit && (lds_of(least) > lds_limit || cost(c) < cost(least))) least = c;
      const int percent = nks == 2 ? 70 : nks == 7 ? 90 : nks == 17 ? 85 : 95;
      if (lds_of(sh) > lds_limit || 100 * staged(least) <= percent * staged(sh)) {
        sh = least;
        more = patch_of(sh) > own_slots;
      }
    }
    const long long blocks = blocks_of(sh);
    const size_t all = lds_of(sh);
    if (all <= lds_limit && blocks < 0x7fffffffLL) {
      auto kern = !more ? (wide_patch && nks == 17 ? conv_i8_rows_kernel<17, 1, false, 12, 8>
                           : wide_patch ? conv_i8_rows_kernel<0, 1, false, 12, 8>
                           : two && nks == 7 ? conv_i8_rows_kernel<7, 2, false, 6, 4>
                           : two && nks == 2 ? conv_i8_rows_kernel<2, 2, false, 4, 4>
                           : two             ? conv_i8_rows_kernel<0, 2, false, 6, 4>
                           : nks == 7        ? conv_i8_rows_kernel<7, 1, true, 6, 4>
                           : nks == 2        ? conv_i8_rows_kernel<2, 1, true, 6, 4>
                                             : conv_i8_rows_kernel<0, 1, false, 8, 4>)
                  : wide_patch                ? conv_i8_rows_kernel<0, 1, false, 18, 8>
                  : patch_of(sh) <= 8 * 64    ? conv_i8_rows_kernel<0, 1, false, 8, 4>
                                              : conv_i8_rows_kernel<0, 1, false, 18, 4>;
      // persistent grid: exactly as many work-groups as the device holds at once
      int per_cu = 0;
      if (wide_patch) {
        static std::atomic<unsigned long long> raised[3];
        e = raise_lds_limit(raised[more ? 2 : nks == 17], reinterpret_cast<const void *>(kern), lds_limit);
      }
      if (e == hipSuccess)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kern), 64 * nwav, all);
      if (e != hipSuccess) return e;
      unsigned resident = (unsigned)(per_cu > 0 ? per_cu : 1) * (unsigned)cus;
      const unsigned slices = (unsigned)((COUT + 63) / 64);
      resident = resident / slices > 0 ? resident / slices : 1;
      const unsigned want = (unsigned)((blocks + nwav - 1) / nwav);
      dim3 g2(want > resident ? resident : want, slices);
      const uint32_t xm = zero_point == 128 ? 0x80808080u : 0u;
      const uint8_t *Xu = reinterpret_cast<const uint8_t *>(X);
      // multiply-high quotients for the block decode, where they are exact (n * d < 2^32)
      auto magic = [&](unsigned long long d) {
        return (d >= 2 && (unsigned long long)blocks * d < (1ull << 32)) ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u;
      };
      const uint32_t mg = magic((unsigned long long)sh.gpr), mh = magic((unsigned long long)sh.gpc);
      // small dividends (patch slots, filter tasks below 2^16): always exact
      auto small_magic = [](int d) { return d >= 2 ? (uint32_t)(((1ull << 32) + (unsigned)d - 1) / (unsigned)d) : 0u; };
      const uint32_t mn = small_magic(sh.ndw), mp = small_magic(HPR);
      hipLaunchKernelGGL(kern, g2, dim3(64 * nwav), all, s, Xu, Wt, thr, planes, B, H, W, C, COUT, R, S, stride, pad, Ho,
                         Wo, bits, xm, HPR, sh.pr, sh.ndw, sh.lw, mg, mh, mn, mp);
      return hipGetLastError();
    }
  }
  if (C <= 4) {
    // dword-per-pixel patch kernel, persistent over pixel groups: the filter block is staged once
    // per work-group
    if (grid.x > 1024) grid.x = 1024;
    const int KR = (S * 4 + 31) / 32;
    const int PW = 31 * stride + KR * 8;
    const int patch_words = (R * PW + 15) / 16 * 16;
    const size_t lds = (size_t)64 * (R * KR * 32 + 16) + 4 * (size_t)patch_words * 4;
    if (lds <= 160 * 1024) {
      if (lds > 64 * 1024) {
        static std::atomic<unsigned long long> raised;
        const hipError_t e = raise_lds_limit(raised, reinterpret_cast<const void *>(conv_i8_c4_kernel), 160 * 1024);
        if (e != hipSuccess) return e;
      }
      hipLaunchKernelGGL(conv_i8_c4_kernel, grid, dim3(256), lds, s, X, Wt, thr, codes, acc_out, planes, B, H, W, C,
                         COUT, R, S, stride, pad, Ho, Wo, bits, zero_point, KR, PW, patch_words);
      return hipGetLastError();
    }
  }
  if (planes != nullptr) return hipErrorNotSupported;  // plane output is produced by the C <= 4 kernel only
  // general C: byte-gather matrix-core kernel whenever its LDS footprint (filter block, k table, 4 patches) fits
  const int T = (R * S * C + 31) / 32;
  const int rowlen = (31 * stride + S) * C;
  const int patch_bytes = (R * rowlen + 15) / 16 * 16;
  const size_t mfma_lds = (size_t)64 * T * 32 + 2 * T * 32 + 4 * (size_t)patch_bytes;
  if (mfma_lds <= 64 * 1024 && R * rowlen < 0xFFFF) {
    hipLaunchKernelGGL(conv_i8_mfma_kernel, grid, dim3(256), mfma_lds, s, X, Wt, thr, codes, acc_out, B, H, W, C, COUT,
                       R, S, stride, pad, Ho, Wo, bits, zero_point, T, rowlen, patch_bytes);
    return hipGetLastError();
  }
  const size_t lds = (size_t)64 * R * S * C;
  dim3 grid2((unsigned)((npix + 63) / 64), (unsigned)((COUT + 63) / 64));
  hipLaunchKernelGGL(conv_i8_bn_kernel<64>, grid2, dim3(256), lds, s, X, Wt, thr, codes, acc_out, B, H, W, C, COUT, R,
                     S, stride, pad, Ho, Wo, bits, zero_point);
  return hipGetLastError();
}

hipError_t launch_pool_planes(const uint32_t *in, uint32_t *out, int B, int H, int W, int cw, int bits, int win,
                              int stride, int pad, hipStream_t s) {
  const int Ho = (H + 2 * pad - win) / stride + 1, Wo = (W + 2 * pad - win) / stride + 1;
  long long blocks = ((long long)B * Ho * Wo * cw + 255) / 256;
  if (blocks > 262144) blocks = 262144;
  // 64-bit accesses need 8-byte aligned rows: an even number of channel words and 8-byte aligned buffers
  const bool vec2 = bits <= 2 && win == 3 && (cw & 1) == 0 &&
                    ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 7) == 0;
  if (vec2)
    hipLaunchKernelGGL((pool_planes_kernel<2, 2>), dim3((unsigned)((blocks + 1) / 2)), dim3(256), 0, s, in, out, B, H, W, cw,
                       bits, win, stride, pad, Ho, Wo);
  else if (bits <= 2)
    hipLaunchKernelGGL(pool_planes_kernel<2>, dim3((unsigned)blocks), dim3(256), 0, s, in, out, B, H, W, cw, bits, win,
                       stride, pad, Ho, Wo);
  else
    hipLaunchKernelGGL(pool_planes_kernel<8>, dim3((unsigned)blocks), dim3(256), 0, s, in, out, B, H, W, cw, bits, win,
                       stride, pad, Ho, Wo);
  return hipGetLastError();
}

hipError_t launch_pool_pack(const uint8_t *codes, uint32_t *planes, int B, int H, int W, int C, int cpad, int bits,
                            int win, int stride, int pad, hipStream_t s) {
  const int Ho = (H + 2 * pad - win) / stride + 1, Wo = (W + 2 * pad - win) / stride + 1;
  const long long total = (long long)B * Ho * Wo * ((cpad + 63) / 64);
  long long blocks = (total + 3) / 4;
  if (blocks > 262144) blocks = 262144;
  hipLaunchKernelGGL(pool_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, s, codes, planes, B, H, W, C, cpad, bits,
                     win, stride, pad, Ho, Wo);
  return hipGetLastError();
}

hipError_t launch_unpack_sum(const uint32_t *planes, int8_t *out, long long rows_out, int group, int C, int cpad,
                             int bits, int shift, hipStream_t s) {
  if (group >= 8) {
    const long long waves = rows_out * (cpad >> 5);
    if ((waves + 3) / 4 <= 0x7fffffffLL) {
      hipLaunchKernelGGL(pool_sum_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, planes, out, rows_out,
                         group, C, cpad, bits, shift);
      return hipGetLastError();
    }
  }
  int JP = 1;
  while (JP < 16 && JP * 2 <= group) JP *= 2;
  long long blocks = (rows_out * C * JP + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(unpack_sum_kernel, dim3((unsigned)blocks), dim3(256), 0, s, planes, out, rows_out, group, C, cpad,
                     bits, shift, JP);
  return hipGetLastError();
}

// Larger batches: one wave per 8 output features x 8 batch rows (every operand dword is used eight times, so
// the waves re-read half as many bytes from L2 as with 4 x 4).  The 64 per-lane partial sums are reduced
// by a transposing butterfly: at step s a lane keeps the accumulator whose index has bit s equal to its own
// lane bit s and hands the other one to its partner lane, so the number of live accumulators halves at every
// step (63 exchanges in all instead of 6 x 64) and lane l ends up with the complete sum of accumulator l.
// Requires K % 4 == 0 and 4-byte aligned rows.
__global__ __launch_bounds__(256) void fc_i8_tile_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                         const float *__restrict__ scale, const float *__restrict__ bias,
                                                         float *__restrict__ out, int32_t *__restrict__ acc_out, int Bn,
                                                         int N, int K) {
  const int lane = threadIdx.x & 63;
  const int bgroups = (Bn + 7) >> 3, ngroups = (N + 7) >> 3;
  const long long wid = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= (long long)ngroups * bgroups) return;
  const int n0 = (int)(wid % ngroups) * 8;
  const int b0 = (int)(wid / ngroups) * 8;
  int acc[64];
#pragma unroll
  for (int a = 0; a < 64; ++a) acc[a] = 0;
  // the affine map of this lane's output feature, requested before the K loop
  const int nf = min(n0 + (lane >> 3), N - 1);
  const float out_scale = scale[nf], out_bias = bias[nf];
  const int *wrow[8], *xrow[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    wrow[i] = reinterpret_cast<const int *>(Wt + (long long)min(n0 + i, N - 1) * K);
    xrow[i] = reinterpret_cast<const int *>(X + (long long)min(b0 + i, Bn - 1) * K);
  }
#pragma unroll 2
  for (int k4 = lane; k4 < (K >> 2); k4 += 64) {
    int wv[8], xv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      wv[i] = wrow[i][k4];
      xv[i] = xrow[i][k4];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i * 8 + j] = __builtin_amdgcn_sdot4(xv[j], wv[i], acc[i * 8 + j], false);
  }
  static_for_n<0, 6>([&](auto sc) {
    constexpr int st = decltype(sc)::value;
    constexpr int n = 64 >> st;  // live accumulators before this step
    const bool hi = (lane >> st) & 1;
#pragma unroll
    for (int t = 0; t < n / 2; ++t) {
      const int keep = hi ? acc[2 * t + 1] : acc[2 * t];
      const int send = hi ? acc[2 * t] : acc[2 * t + 1];
      acc[t] = keep + __shfl_xor(send, 1 << st, 64);
    }
  });
  // lane l = 8 * feature + batch row (rows / features past the end were clamped duplicates: dropped here)
  const int i = lane >> 3, j = lane & 7;
  if (n0 + i < N && b0 + j < Bn) {
    const long long o = (long long)(b0 + j) * N + n0 + i;
    if (acc_out != nullptr) acc_out[o] = acc[0];
    out[o] = (float)acc[0] * out_scale + out_bias;
  }
}

hipError_t launch_fc_i8(const int8_t *X, const int8_t *Wt, const float *scale, const float *bias, float *out,
                        int32_t *acc_out, int Bn, int N, int K, hipStream_t s) {
  const int vec_ok = (K % 4 == 0) && ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Wt)) & 3u) == 0;
  if (vec_ok && Bn >= 32 && (long long)((N + 7) / 8) * ((Bn + 7) / 8) >= 512) {
    const long long waves = (long long)((N + 7) / 8) * ((Bn + 7) / 8);
    hipLaunchKernelGGL(fc_i8_tile_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, X, Wt, scale, bias, out,
                       acc_out, Bn, N, K);
    return hipGetLastError();
  }
  if ((long long)N * ((Bn + 3) / 4) >= 8192) {  // plenty of waves: four features per wave cut the re-reads of X
    const long long waves = (long long)((N + 3) / 4) * ((Bn + 3) / 4);
    hipLaunchKernelGGL(fc_i8_kernel<4>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, X, Wt, scale, bias, out,
                       acc_out, Bn, N, K, vec_ok);
  } else {
    const long long waves = (long long)N * ((Bn + 3) / 4);
    hipLaunchKernelGGL(fc_i8_kernel<1>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, X, Wt, scale, bias, out,
                       acc_out, Bn, N, K, vec_ok);
  }
  return hipGetLastError();
}

}  // namespace apnn
