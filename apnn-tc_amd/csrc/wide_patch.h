// Sizes of the patch-resident convolution with packed weights (wide_patch_kernel.h), for its launcher and the dispatch.
#pragma once
#include <cstddef>

namespace apnn {

constexpr int kWidePatchPixels = 384;  // three half pixels a thread
constexpr int wide_patch_units(int pa) { return pa > 2 ? 2 : 3; }  // work-groups per compute unit (registers)
// LDS words of a patch pixel: eight operands of 16 or, FP6, 24 bytes; sums of two weight planes
constexpr int wide_pixel_words(int pa, int pb) { return 8 * (pa > 2 ? 6 : 4) + (pb > 1 ? 2 : 0); }
constexpr size_t wide_stage_words(int pa, int pb, int tb, int cap) {
  const size_t words = (size_t)2 * pb * tb * 8 + (size_t)wide_pixel_words(pa, pb) * cap;
  return ((words > 4096 ? words : 4096) + 3) & ~(size_t)3;  // the output stage uses 16 KB
}

}  // namespace apnn
