// One translation unit per (INST_PA, INST_PB): the 128x128 tile of the patch-resident convolution with packed weights.
#include "wide_patch_kernel.h"

#ifndef INST_PA
#error "compile with -DINST_PA=.. -DINST_PB=.."
#endif
#define APNN_CAT2(a, b, c, d) a##b##_##c##_##d
#define APNN_CAT(a, b, c, d) APNN_CAT2(a, b, c, d)

namespace apnn {

hipError_t APNN_CAT(wide_patch_, INST_PA, INST_PB, x)(const KParams &p, hipStream_t s) {
  return launch_wide_patch<INST_PA, INST_PB>(p, s);
}

}  // namespace apnn
