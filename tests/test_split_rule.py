"""Where AUTO takes the 32x32 and where the 32x64 split-K tile for convolutions of few outputs."""
import ctypes

import pytest

import pkg

A = pkg.load()


@pytest.mark.parametrize("B,H,C,cout,blocks", [(8, 13, 384, 256, 344), (2, 16, 512, 512, 256), (12, 7, 512, 512, 304), (5, 16, 512, 512, 640),
                                               (8, 14, 128, 256, 392), (8, 13, 320, 256, 344)])
def test_split_tiles_beyond_one_block_a_unit(B, H, C, cout, blocks):
    """The 32x32 split-K tile serves up to one block per unit; beyond, 32x64 over 72 words and more in 128-bit loads."""
    assert -(-B * H * H // 32) * (cout // 32) == blocks
    for wb, xb in [(1, 3), (1, 4), (2, 2)]:
        plan = A.Plan()
        d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=B, H=H, Wd=H, cin_pad=C, COUT=cout, R=3, S=3, stride=1, pad=1, halo=0,
                       wb=wb, xb=xb, path=A.PATH_AUTO)
        assert A.lib().apnn_conv_plan(ctypes.byref(d), ctypes.byref(plan)) == 0
        assert plan.kernel == A.KERNEL_MFMA_FP4
        assert (plan.tile_rows, plan.tile_cols) == ((32, 64) if blocks > 256 and 9 * C // 32 >= 72 and C % 128 == 0 else (32, 32))


@pytest.mark.parametrize("B,H,C,cout,wb,xb,cols", [
    (50, 14, 512, 32, 1, 4, 32), (22, 14, 512, 96, 1, 3, 32),                               # a second 32x64 tile for a unit
    (15, 14, 512, 96, 1, 3, 64), (15, 14, 512, 96, 2, 2, 64), (7, 14, 512, 224, 1, 4, 64),  # none, a quarter or an eighth empty
    (7, 14, 512, 416, 1, 3, 64), (30, 14, 512, 96, 1, 4, 64), (90, 14, 512, 32, 1, 4, 32),  # up to 2.5 blocks: little, a quarter, half empty
    (12, 14, 256, 256, 1, 4, 64), (12, 14, 256, 256, 2, 2, 32),                             # 72 words there
    (29, 13, 768, 128, 2, 2, 64), (29, 13, 1024, 128, 2, 2, 32), (6, 14, 512, 544, 2, 2, 32),
    (8, 14, 256, 256, 1, 3, 32),                                                            # 72 words
])
def test_split_tiles_by_rounds(B, H, C, cout, wb, xb, cols):
    """32x64 where it leaves every unit one tile, or up to 2.5 blocks of 32x32 a unit where its columns are filled."""
    plan = A.Plan()
    d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=B, H=H, Wd=H, cin_pad=C, COUT=cout, R=3, S=3, stride=1, pad=1, halo=0,
                   wb=wb, xb=xb, path=A.PATH_AUTO)
    assert A.lib().apnn_conv_plan(ctypes.byref(d), ctypes.byref(plan)) == 0
    assert plan.kernel == A.KERNEL_MFMA_FP4 and (plan.tile_rows, plan.tile_cols) == (32, cols)
