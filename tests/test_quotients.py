"""Quotients of the patch-resident convolutions: exact on maps of any height and width."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle_lib as O
import pkg

A = pkg.load()
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include "quotient.h"
#include <cstdio>
using namespace apnn;
template <bool SHORT> static bool bad(uint32_t d, uint32_t m, uint32_t n) {
  if (quotient<SHORT>(n, d, m) == n / d) return false;
  printf("%u / %u\n", n, d);
  return true;
}
// a quotient a little above n / d is wrong first for the largest n of a remainder d - 1, and at whole multiples where it is below
template <bool SHORT> static bool bad(uint32_t d) {
  const uint32_t m = quotient_magic(d, SHORT), top = SHORT ? d + 1024 : 0x80000000u, last = top / d * d;
  for (uint32_t k = 1; k <= 1024 / d + 2 && (unsigned long long)k * d <= top; ++k)
    if (bad<SHORT>(d, m, k * d - 1) || bad<SHORT>(d, m, k * d)) return true;
  return bad<SHORT>(d, m, 0) || bad<SHORT>(d, m, last) || bad<SHORT>(d, m, last - 1) || bad<SHORT>(d, m, top);
}
int main() {
  for (uint32_t d = 1; d <= kShortDivisor; ++d)
    if (bad<true>(d)) return 1;
  for (uint32_t d = 1; d < (1u << 22); ++d)
    if (bad<false>(d)) return 1;
  for (int b = 22; b < 31; ++b)
    for (int k = -300; k <= 300; ++k)
      if (bad<false>((1u << b) + k)) return 1;
  for (uint32_t d = 4194319, i = 0; i < 2000000; ++i, d = (d * 1664525u + 1013904223u) & 0x7fffffffu)
    if (d > 0 && bad<false>(d)) return 1;
  return 0;
}
"""


def test_exact_for_every_divisor(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "apnn-tc_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, "quotient is not exact: " + r.stdout


# heights at which the padded frame or the row grid passes 65536, and widths (a single row under the filter: more rows of such
# maps exceed any patch); 100000 rows, whose multiply-high without a shift fails too
WIDE_MAPS = [(1, 65535, 1, 3, 3, 1), (1, 65536, 1, 3, 3, 1), (2, 65537, 1, 3, 3, 1), (1, 100000, 1, 3, 3, 1), (1, 65536, 2, 3, 3, 1),
             (2, 1, 65539, 1, 3, 0), (1, 1, 100001, 1, 3, 0), (2, 3, 65537, 1, 1, 0)]


def _tall(G, path, tile, wb, xb, B, H, W, C, cout, R, S, pad):
    rng = np.random.default_rng(9300 + H + W + 10 * wb + xb)
    X, Wt = O.random_planes(rng, xb, B * H * W, C // 32), O.random_planes(rng, wb, cout * R * S, C // 32)
    kw = dict(batch=B, H=H, W=W, cout=cout, R=R, S=S, stride=1, pad=pad, halo=0, wb=wb, xb=xb)
    expect = O.conv(Wt, X, cwords=C // 32, sym_w=1, nthreads=8, **kw).reshape(-1)
    return np.array_equal(G.run_conv(Wt, X, cin_pad=C, sym=1, path=path, tile=tile, **kw), expect)


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", [(1, 2), (1, 4), (2, 2)])
@pytest.mark.parametrize("B,H,W,R,S,pad", WIDE_MAPS)
def test_packed_weights_patch_on_tall_and_wide_maps(B, H, W, R, S, pad, wb, xb):
    import gpu_util as G
    assert _tall(G, A.PATH_MFMA, 12, wb, xb, B, H, W, 256, 32, R, S, pad)


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", [(1, 2), (1, 4), (2, 2)])
@pytest.mark.parametrize("tile,C", [(1, 64), (3, 96), (4, 64)])
@pytest.mark.parametrize("B,H,W,R,S,pad", WIDE_MAPS)
def test_expanded_patch_on_tall_and_wide_maps(B, H, W, R, S, pad, tile, C, wb, xb):
    import gpu_util as G
    assert _tall(G, A.PATH_MFMA_PATCH, tile, wb, xb, B, H, W, C, 32, R, S, pad)


@pytest.mark.gpu
def test_auto_on_a_tall_map():
    """A layer that AUTO gives to the 128x128 tile over a patch; the last rows are those a rounded quotient misplaces."""
    import gpu_util as G
    plan = A.Plan()
    d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=1, H=65537, Wd=4, cin_pad=256, COUT=128, R=3, S=3, stride=1, pad=1, halo=0, wb=1,
                   xb=2, path=A.PATH_AUTO)
    assert A.lib().apnn_conv_plan(ctypes.byref(d), ctypes.byref(plan)) == 0 and plan.tile == 12
    assert _tall(G, A.PATH_AUTO, None, 1, 2, 1, 65537, 4, 256, 128, 3, 3, 1)
