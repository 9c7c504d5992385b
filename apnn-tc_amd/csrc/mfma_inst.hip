// One translation unit per (INST_CORE, INST_PA, INST_PB, INST_CONV): tile-shape instantiations of
// the MFMA kernel.  INST_CORE 0 = int8 operands, 1 = FP4 operands.
#include "mfma_kernel.h"
#if INST_CORE == 1
#include "async_kernel.h"
#if !INST_CONV
#include "ksplit_kernel.h"
#endif
#endif

#ifndef INST_PA
#error "compile with -DINST_PA=.. -DINST_PB=.. -DINST_CONV=0|1"
#endif

#if INST_CORE == 1
#define APNN_PFX(n) mfma4_##n
#else
#define APNN_PFX(n) mfma_##n
#endif
#define APNN_CAT2(a, b, c, d) a##b##_##c##_##d
#define APNN_CAT(a, b, c, d) APNN_CAT2(a, b, c, d)

namespace apnn {

#if INST_CONV
hipError_t APNN_CAT(APNN_PFX(conv_), INST_PA, INST_PB, x)(int vw, int tile, const KParams &p, hipStream_t s) {
#if INST_CORE == 1
  if constexpr (async_built(INST_PA, INST_PB)) {
    if (vw == 4 && tile == MT_128x256) return launch_async<INST_PA, INST_PB, 2, 4, 2, 2, true, 2>(p, s);
    if (vw == 4 && tile == MT_128x128) return launch_async<INST_PA, INST_PB, 2, 2, 2, 2, true, 2>(p, s);
  }
#endif
  switch (vw) {
    case 4: return launch_mfma_tile<INST_CORE, INST_PA, INST_PB, 4, true>(tile, p, s);
    case 2: return launch_mfma_tile<INST_CORE, INST_PA, INST_PB, 2, true>(tile, p, s);
    default: return launch_mfma_tile<INST_CORE, INST_PA, INST_PB, 1, true>(tile, p, s);
  }
}
#else
hipError_t APNN_CAT(APNN_PFX(gemm_), INST_PA, INST_PB, x)(int vw, int tile, const KParams &p, hipStream_t s) {
  (void)vw;
#if INST_CORE == 1
  if constexpr (async_built(INST_PA, INST_PB)) {
    if (tile == MT_256x128) return launch_async<INST_PA, INST_PB, 4, 2, 2, 2, false, 2>(p, s);
  }
#endif
#if INST_CORE == 1
  if constexpr (ksplit_built(CORE_F4, false, MT_128x64_K4, INST_PA, INST_PB)) {
    if (tile == MT_128x64_K4) return launch_ksplit<INST_PA, INST_PB, 2, 2, 2, 4>(p, s);
  }
  if constexpr (ksplit_built(CORE_F4, false, MT_64x96_K8, INST_PA, INST_PB)) {
    if (tile == MT_64x96_K8) return launch_ksplit<INST_PA, INST_PB, 2, 3, 1, 8>(p, s);
  }
#endif
  return launch_mfma_tile<INST_CORE, INST_PA, INST_PB, 4, false>(tile, p, s);
}
#endif

}  // namespace apnn
