"""First layer on blocks of pixels: one and two sets of 32, blocks 8, 16 and 32 wide, maps that end inside a block, every number of
k-steps with a form of its own, half a block of channels, filters whose last 16 bytes are loaded from before their place."""
import numpy as np
import pytest
import torch

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


@pytest.mark.parametrize("B,H,W,C,cout,R,stride,pad", [
    (1, 11, 12, 3, 32, 3, 1, 1), (40, 33, 36, 3, 96, 3, 1, 1), (24, 61, 64, 3, 32, 3, 2, 0),      # 2 k-steps, one and two sets
    (2, 17, 20, 3, 64, 7, 2, 3), (40, 65, 68, 3, 96, 7, 2, 3), (70, 45, 48, 3, 64, 7, 1, 0),      # 7
    (2, 37, 40, 3, 64, 11, 4, 5), (30, 63, 64, 3, 32, 11, 4, 0),                                  # 17, eight waves
    (3, 20, 16, 1, 64, 7, 2, 3), (60, 40, 44, 1, 32, 7, 1, 3), (50, 31, 32, 4, 96, 5, 1, 2), (2, 40, 40, 3, 32, 9, 3, 4),  # other numbers
    (3, 40, 44, 4, 64, 11, 2, 5), (1, 8, 8, 2, 32, 1, 1, 0),
    # strides beyond the filter: 32 pixels of a row, also where no other block fits the LDS
    (2, 64, 64, 1, 64, 16, 16, 0), (1, 96, 96, 1, 32, 11, 24, 5), (3, 100, 100, 3, 64, 4, 32, 2), (40, 69, 72, 3, 96, 5, 16, 2),
    (2, 64, 64, 4, 64, 4, 4, 0), (1, 70, 72, 3, 32, 7, 7, 0), (40, 64, 64, 1, 32, 14, 7, 0), (3, 80, 84, 4, 64, 11, 5, 2),  # in place
    (1, 9, 1100, 1, 64, 7, 32, 3), (2, 40, 700, 4, 32, 2, 8, 1), (1, 16, 1056, 3, 64, 3, 16, 1),
])
@pytest.mark.parametrize("bits,zero", [(2, 128), (1, 128), (2, 0)])
def test_first_layer_blocks(G, B, H, W, C, cout, R, stride, pad, bits, zero):
    rng = np.random.default_rng(9900 + B + H + R + bits + zero)
    X = rng.integers(0, 256, size=(B, H, W, C)).astype(np.uint8)
    Wt = rng.integers(-128, 128, size=(cout, R, R, C)).astype(np.int8)
    signed = (X.astype(np.int16) - 128).astype(np.int8) if zero else X.view(np.int8)
    acc = O.conv_i8(Wt, signed, stride, pad).reshape(-1, cout)
    rows = acc.shape[0]
    thr = np.sort(rng.integers(acc.min(), acc.max() + 1, size=(cout, 2 ** bits - 1)), axis=1).astype(np.int32)
    dX, dW, dT = torch.from_numpy(X).cuda(), G.to_dev(Wt), G.to_dev(thr)
    planes = G.dev_empty_i32(bits * rows * cout // 32, fill=-7)
    G.A.check(G.A.lib().apnn_conv_i8_bn_pack(G.ptr(dX), G.ptr(dW), G.ptr(dT), G.ptr(planes), B, H, W, C, cout, R, R, stride, pad,
                                             bits, zero, None), "conv_i8_bn_pack")
    expect = O.pack_bits(O.bn_quantize(acc, None, thr, None, bits).astype(np.uint32), rows, cout, cout, bits)
    assert np.array_equal(G.to_host(planes, np.uint32).reshape(expect.shape), expect)
