"""Edges of the kernels' tiles and of the dispatch rules: remainders, smallest and largest sizes, each against
the oracle or an exact integer / fp32 reference (integers and packed words: equality, no tolerance)."""
import numpy as np
import pytest
import torch

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# Packers: one wave owns 8 words of a small tensor and 64 of a large one (from 131072 words); rows with padding
# (C < cpad) and without; one-word rows, where the two halves of a wave work on different rows.
@pytest.mark.parametrize("rows,C,cpad", [(1, 32, 32), (7, 1, 32), (9, 31, 32), (33, 33, 64), (5, 96, 96), (131071, 32, 32),
                                         (131075, 30, 32), (26216, 160, 160), (26219, 129, 160), (65537, 64, 64)])
@pytest.mark.parametrize("bits,lo,hi", [(2, -10.0, 10.0), (5, -0.3, 0.7), (1, 0.0, 3.0), (3, -1e-20, 3e-20)])
def test_float_packer_edges(G, rows, C, cpad, bits, lo, hi):
    """Every operation of the quantizer is one fp32 rounding, so numpy's fp32 arithmetic is the exact reference; the
    last range is below 2^-60 and takes the kernel's dividing form."""
    rng = np.random.default_rng(8100 + rows + bits)
    lo, hi = np.float32(lo), np.float32(hi)
    span = np.float32(hi - lo)
    x = rng.uniform(float(lo) - 0.2 * float(span), float(hi) + 0.2 * float(span), size=(rows, C)).astype(np.float32)
    flat = x.reshape(-1)
    ties = (lo + span * (np.arange(min(flat.size, 64)) + 0.5).astype(np.float32) / np.float32(2 ** bits)).astype(np.float32)
    flat[:ties.size] = ties
    if flat.size > 70:
        flat[64:70] = [np.nan, np.inf, -np.inf, lo, hi, -0.0]
    d = torch.from_numpy(x).cuda()
    planes = G.dev_empty_i32(bits * rows * cpad // 32, fill=-7)
    G.A.check(G.A.lib().apnn_quantize_pack(G.ptr(d), G.ptr(planes), rows, C, cpad, bits, float(lo), float(hi), None), "quantize_pack")
    c = np.where(np.isnan(x), lo, np.clip(x, lo, hi)).astype(np.float32)
    q = (((c - lo) * np.float32(2 ** bits)) / span).astype(np.float32)
    codes = np.minimum(np.rint(q), 2 ** bits - 1).astype(np.uint32)
    expect = O.pack_bits(codes, rows, C, cpad, bits)
    assert np.array_equal(G.to_host(planes, np.uint32).reshape(expect.shape), expect)


# Precisions beyond five planes (FP6 digits of four planes) and w1a1 on every tile that is built: one row past a
# tile, one short of it, reductions that end inside a chunk.
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 9])
@pytest.mark.parametrize("wb,xb", [(1, 1), (1, 8), (2, 8), (4, 4)])
@pytest.mark.parametrize("M,N,K,sym", [(129, 255, 640, 1), (31, 33, 128, 0), (257, 129, 1152, 0)])
def test_wide_precision_gemm_tiles(G, wb, xb, tile, M, N, K, sym):
    rng = np.random.default_rng(8200 + M + 10 * wb + xb)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=sym, path=2, tile=tile).reshape(M, N)
    assert np.array_equal(got, O.gemm(W, X, M, N, K, wb, xb, sym_w=sym))


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("wb,xb", [(1, 5), (2, 6), (1, 8), (2, 8)])
@pytest.mark.parametrize("H,C,cout,R,sym", [(13, 128, 96, 3, 1), (5, 256, 33, 1, 0)])
def test_wide_precision_conv_tiles(G, wb, xb, tile, H, C, cout, R, sym):
    rng = np.random.default_rng(8300 + H + 10 * wb + xb)
    W, X = O.random_planes(rng, wb, cout * R * R, C // 32), O.random_planes(rng, xb, 2 * H * H, C // 32)
    kw = dict(batch=2, H=H, W=H, cout=cout, R=R, S=R, stride=1, pad=R // 2, halo=0, wb=wb, xb=xb)
    got = G.run_conv(W, X, cin_pad=C, sym=sym, path=2, tile=tile, **kw)
    assert np.array_equal(got.reshape(-1, cout), O.conv(W, X, cwords=C // 32, sym_w=sym, **kw).reshape(-1, cout))


@pytest.mark.parametrize("wb,xb,M,N,K", [(1, 1, 111, 67, 1792), (1, 1, 1, 1, 128), (2, 8, 52, 72, 128), (4, 4, 3, 5, 256), (1, 8, 16, 1, 8192)])
def test_small_products_of_precisions_without_popcount_kernel(G, wb, xb, M, N, K):
    """AUTO takes the matrix cores for these at every size (the any-precision popcount kernel is 5-16 times slower)."""
    rng = np.random.default_rng(8400 + M + wb + xb)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    assert np.array_equal(G.run_gemm(W, X, M, N, K, wb, xb).reshape(M, N), O.gemm(W, X, M, N, K, wb, xb))


# The convolution output stage with pixels in the lanes: codes of one to four bits, flip flags, shortcut scales that
# are one or two terms m * 2^j (m up to 15) and one that is not, pixel rows and channels that end inside a tile.
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("xb,ob,scale", [(2, 2, 43), (2, 1, -171), (2, 3, 0), (3, 3, 203), (4, 4, 1365), (3, 2, 0), (4, 1, 15)])
@pytest.mark.parametrize("sym", [0, 1])
def test_conv_codes_flips_and_shortcuts(G, tile, xb, ob, scale, sym):
    rng = np.random.default_rng(8500 + tile + 10 * xb + ob)
    batch, H, C, cout = 3, 7, 128, 96
    W, X = O.random_planes(rng, 1, cout * 9, C // 32), O.random_planes(rng, xb, batch * H * H, C // 32)
    kw = dict(batch=batch, H=H, W=H, cout=cout, R=3, S=3, stride=1, pad=1, halo=0, wb=1, xb=xb)
    v = O.conv(W, X, cwords=C // 32, sym_w=sym, **kw).reshape(-1, cout).astype(np.int64)
    extra = {}
    if scale:
        short = rng.integers(0, 4, size=v.shape).astype(np.uint32)
        v = v + scale * short.astype(np.int64)
        d_short = G.to_dev(O.pack_bits(short, v.shape[0], cout, cout, 2))
        extra = dict(resid_planes=d_short, resid_bits=2, resid_scale=scale)
    thr = np.sort(rng.integers(v.min() - 5, v.max() + 6, size=(cout, 2 ** ob - 1)), axis=1).astype(np.int32)
    thr[0, :] = np.iinfo(np.int32).min
    thr[1, :] = np.iinfo(np.int32).max
    flip = rng.integers(0, 2, size=cout).astype(np.uint8)
    thr[flip != 0] = np.sort(-thr[flip != 0].astype(np.int64), axis=1).clip(-2 ** 31, 2 ** 31 - 1).astype(np.int32)
    d_thr, d_flip = G.to_dev(thr), G.to_dev(flip)
    epi = G.epilogue(mode=G.A.EPI_BN, out_bits=ob, thr=d_thr, flip=d_flip, **extra)
    got = G.run_conv(W, X, cin_pad=C, sym=sym, epi=epi, path=2, tile=tile, **kw).view(np.uint32).reshape(ob, -1, cout // 32)
    q = O.bn_quantize(v.astype(np.int32), None, thr, flip, ob)
    assert np.array_equal(got, O.lowbits_pack(q, v.shape[0], cout, ob))


# GEMM tile 256x128 (operands loaded straight to LDS): rows and columns around the tile, reductions of half a group,
# one group, one chunk and a few words more; -1 / +1, unsigned and two-plane weights.
@pytest.mark.parametrize("wb,xb", [(1, 1), (1, 2), (1, 3), (1, 4), (2, 2)])
@pytest.mark.parametrize("sym", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (255, 127, 256), (257, 129, 384), (256, 128, 512), (300, 130, 640),
                                   (511, 257, 1024), (513, 96, 1152), (40, 300, 2176)])
def test_async_gemm_tile(G, wb, xb, sym, M, N, K):
    rng = np.random.default_rng(8400 + M + 10 * wb + xb)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=sym, path=2, tile=6).reshape(M, N)
    assert np.array_equal(got, O.gemm(W, X, M, N, K, wb, xb, sym_w=sym))


# Convolution tiles 128x256 and 128x128 (operands loaded straight to LDS): images smaller and larger than a tile,
# channel words that are and are not a power of two, taps that straddle a chunk, stride, padding, int32 results,
# thresholds and a shortcut (the other output forms: test_conv_output_forms).
@pytest.mark.parametrize("tile", [1, 7])
@pytest.mark.parametrize("wb,xb", [(1, 2), (1, 3), (1, 4), (2, 2)])
@pytest.mark.parametrize("batch,H,C,cout,R,stride,pad", [(1, 5, 128, 32, 3, 1, 1), (2, 9, 384, 288, 3, 1, 1),
                                                         (3, 13, 256, 160, 3, 2, 1), (1, 16, 640, 256, 1, 1, 0),
                                                         (2, 8, 128, 96, 5, 1, 2)])
@pytest.mark.parametrize("sym,mode", [(0, "int32"), (1, "int32"), (1, "bn"), (0, "shortcut")])
def test_async_conv_tiles(G, wb, xb, tile, batch, H, C, cout, R, stride, pad, sym, mode):
    rng = np.random.default_rng(8500 + C + cout + 10 * wb + xb)
    Ho = (H + 2 * pad - R) // stride + 1
    rows = batch * Ho * Ho
    X = O.random_planes(rng, xb, batch * H * H, C // 32)
    Wt = O.random_planes(rng, wb, cout * R * R, C // 32)
    kw = dict(batch=batch, H=H, W=H, cout=cout, R=R, S=R, stride=stride, pad=pad, halo=0, wb=wb, xb=xb)
    acc = O.conv(Wt, X, cwords=C // 32, sym_w=sym, **kw).reshape(-1, cout)
    if mode == "int32":
        got = G.run_conv(Wt, X, cin_pad=C, sym=sym, path=2, tile=tile, **kw).reshape(rows, cout)
        assert np.array_equal(got, acc)
        return
    lo, hi = int(acc.min()), int(acc.max())
    thr = np.sort(rng.integers(lo, hi + 1, size=(cout, (1 << xb) - 1)), axis=1).astype(np.int32)
    keep = [G.to_dev(thr)]
    extra, value = {}, acc
    if mode == "shortcut":
        codes = rng.integers(0, 4, size=(rows, cout)).astype(np.uint32)
        keep.append(G.to_dev(O.pack_bits(codes, rows, cout, cout, 2)))
        extra = dict(resid_planes=keep[1], resid_bits=2, resid_scale=5)
        value = acc + 5 * codes.astype(np.int32)
    epi = G.epilogue(mode=G.A.EPI_BN, out_bits=xb, thr=keep[0], **extra)
    got = G.run_conv(Wt, X, cin_pad=C, sym=sym, epi=epi, path=2, tile=tile, **kw).view(np.uint32).reshape(xb, rows, cout // 32)
    q = O.bn_quantize(value, None, thr, None, xb)
    assert np.array_equal(got, O.lowbits_pack(q, rows, cout, xb))


# First layer on image rows: seven k-steps with the filter in registers and (beyond 4096 pixel groups) in LDS, two, three
# and seventeen k-steps; an odd number of channel words, one and two bits, thresholds at the ends of int32.
@pytest.mark.parametrize("B,H,W,C,cout,R,stride,pad", [(2, 30, 36, 3, 96, 7, 2, 3), (42, 200, 8, 3, 96, 7, 2, 3), (3, 9, 36, 3, 64, 3, 1, 1),
                                                       (1, 12, 72, 4, 160, 3, 2, 0), (2, 13, 40, 3, 32, 5, 1, 2),
                                                       (2, 33, 64, 3, 96, 11, 4, 5)])
@pytest.mark.parametrize("bits", [1, 2])
def test_first_layer_filter_supply(G, B, H, W, C, cout, R, stride, pad, bits):
    rng = np.random.default_rng(8600 + H + R + bits)
    X = rng.integers(0, 256, size=(B, H, W, C)).astype(np.uint8)
    Wt = rng.integers(-128, 128, size=(cout, R, R, C)).astype(np.int8)
    acc = O.conv_i8(Wt, (X.astype(np.int16) - 128).astype(np.int8), stride, pad).reshape(-1, cout)
    rows = acc.shape[0]
    thr = np.sort(rng.integers(acc.min(), acc.max() + 1, size=(cout, 2 ** bits - 1)), axis=1).astype(np.int32)
    thr[0, :], thr[17, :] = np.iinfo(np.int32).min, np.iinfo(np.int32).max
    dX, dW, dT = torch.from_numpy(X).cuda(), G.to_dev(Wt), G.to_dev(thr)
    planes = G.dev_empty_i32(bits * rows * cout // 32, fill=-7)
    G.A.check(G.A.lib().apnn_conv_i8_bn_pack(G.ptr(dX), G.ptr(dW), G.ptr(dT), G.ptr(planes), B, H, W, C, cout, R, R, stride, pad,
                                             bits, 128, None), "conv_i8_bn_pack")
    expect = O.pack_bits(O.bn_quantize(acc, None, thr, None, bits).astype(np.uint32), rows, cout, cout, bits)
    assert np.array_equal(G.to_host(planes, np.uint32).reshape(expect.shape), expect)


# A packed shortcut beside sums near the 2^24 limit of fp32: with symmetric weights the matrix cores may hold the raw sum of
# unsigned products, worth two results, and an odd shortcut term is half a unit of it.  All-ones operands make every
# result K * wmax * amax (raw sums between 2^23 and 2^24 units), so the codes equal the shortcut's codes exactly when
# no half unit was rounded away.
_LARGE_SUMS = [(2, 8, 12800), (2, 6, 51200), (2, 2, 1024000), (4, 4, 41600), (1, 8, 64000), (1, 4, 640000), (1, 2, 3200000)]


@pytest.mark.parametrize("gemm,path,tile,wb,xb,K", [
    (gemm, path, tile, wb, xb, K) for gemm in (0, 1) for path, tile in ((0, None), (2, 1), (2, 2), (2, 4), (2, 5), (2, 9), (5, 2))
    for wb, xb, K in _LARGE_SUMS
    # precisions that the expand-while-staging kernel (path 5) and the GEMM matrix-core kernels are built for
    if (path != 5 or (wb, xb) in ((1, 2), (1, 4), (2, 2))) and not (gemm and (wb, xb) == (2, 6))])
def test_shortcut_beside_large_sums(G, gemm, path, tile, wb, xb, K):
    wmax, amax, rows, cols = 2 ** wb - 1, 2 ** xb - 1, 32, 32
    assert 2 ** 23 < K * wmax * amax < 2 ** 24 - 64
    v = K * wmax * amax
    rng = np.random.default_rng(8700 + wb + 10 * xb)
    codes = rng.integers(0, 4, size=(rows, cols)).astype(np.uint32)
    d_short = G.to_dev(O.pack_bits(codes, rows, cols, cols, 2))
    W, X = np.full((wb, cols, K // 32), 0xFFFFFFFF, np.uint32), np.full((xb, rows, K // 32), 0xFFFFFFFF, np.uint32)
    for scale in (1, -3):
        thr = np.sort(v + scale * np.repeat(np.arange(1, 4, dtype=np.int64)[None, :], cols, axis=0), axis=1)
        d_thr = G.to_dev((thr + (scale < 0)).astype(np.int32))
        expect = codes if scale > 0 else 3 - codes
        epi = G.epilogue(mode=G.A.EPI_BN, out_bits=2, thr=d_thr, resid_planes=d_short, resid_bits=2, resid_scale=scale)
        if gemm:
            got = G.run_gemm(W, X, rows, cols, K, wb, xb, sym=1, epi=epi, path=path, tile=tile)
        else:
            got = G.run_conv(W, X, batch=1, H=4, W=8, cin_pad=K, cout=cols, R=1, S=1, stride=1, pad=0, halo=0, wb=wb, xb=xb,
                             sym=1, epi=epi, path=path, tile=tile)
        assert np.array_equal(got.view(np.uint32).reshape(2, rows, cols // 32), O.lowbits_pack(expect, rows, cols, 2)), scale


# Unsigned one-plane weights are plain digits: the shortcut folds while the raw sum and the terms stay below 2^24.
@pytest.mark.parametrize("tile", [None, 1, 2, 4, 5, 9])
@pytest.mark.parametrize("xb", [2, 4, 8])
def test_unsigned_shortcut_beside_large_sums(G, tile, xb):
    amax, rows, cols = 2 ** xb - 1, 32, 32
    K = 1 << (((2 ** 24 - 64) // amax).bit_length() - 1)
    v = K * amax
    rng = np.random.default_rng(8800 + xb)
    codes = rng.integers(0, 4, size=(rows, cols)).astype(np.uint32)
    d_short = G.to_dev(O.pack_bits(codes, rows, cols, cols, 2))
    W, X = np.full((1, cols, K // 32), 0xFFFFFFFF, np.uint32), np.full((xb, rows, K // 32), 0xFFFFFFFF, np.uint32)
    thr = v + np.repeat(np.arange(1, 4, dtype=np.int32)[None, :], cols, axis=0)
    d_thr = G.to_dev(thr.astype(np.int32))
    epi = G.epilogue(mode=G.A.EPI_BN, out_bits=2, thr=d_thr, resid_planes=d_short, resid_bits=2, resid_scale=1)
    got = G.run_conv(W, X, batch=1, H=4, W=8, cin_pad=K, cout=cols, R=1, S=1, stride=1, pad=0, halo=0, wb=1, xb=xb, sym=0,
                     epi=epi, path=0 if tile is None else 2, tile=tile)
    assert np.array_equal(got.view(np.uint32).reshape(2, rows, cols // 32), O.lowbits_pack(codes, rows, cols, 2))


# int32 results pass LDS into rows of 128 bytes: channels that end inside a block and inside a 16-byte unit, pixel rows that
# end inside a tile, output rows that do not start on 16 bytes.
@pytest.mark.parametrize("tile", [1, 2, 3, 7, 9])
@pytest.mark.parametrize("wb,xb,C", [(1, 2, 128), (2, 2, 256), (1, 4, 64), (2, 8, 128)])
@pytest.mark.parametrize("H,cout", [(3, 1), (7, 31), (9, 34), (13, 130), (8, 256)])
def test_conv_int32_rows(G, tile, wb, xb, C, H, cout):
    if C == 64 and tile == 9:
        pytest.skip("two wave groups need 128-bit loads")
    rng = np.random.default_rng(8900 + cout + wb)
    W, X = O.random_planes(rng, wb, cout, C // 32), O.random_planes(rng, xb, 3 * H * H, C // 32)
    kw = dict(batch=3, H=H, W=H, cout=cout, R=1, S=1, stride=1, pad=0, halo=0, wb=wb, xb=xb)
    got = G.run_conv(W, X, cin_pad=C, sym=1, path=2, tile=tile, **kw)
    assert np.array_equal(got.reshape(-1, cout), O.conv(W, X, cwords=C // 32, sym_w=1, **kw).reshape(-1, cout))


# Every output form of the convolutions that is not a plain threshold code, on every tile: low bits, pooled averages and
# maxima, flip flags, codes of one to eight bits, a shortcut scale the matrix cores do not take, an int32 map with the sums
# saved.
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("wb,xb,ob", [(1, 2, 2), (1, 2, 3), (1, 4, 4), (2, 2, 1), (1, 5, 5), (2, 8, 8)])
@pytest.mark.parametrize("bn,pool", [(0, 0), (0, 1), (0, 2), (1, 0), (1, 1), (1, 2)])
def test_conv_output_forms(G, tile, wb, xb, ob, bn, pool):
    rng = np.random.default_rng(9000 + 100 * tile + 10 * xb + ob + 3 * bn + pool)
    batch, H, C, cout = 3, 6, 128, 96
    W, X = O.random_planes(rng, wb, cout * 9, C // 32), O.random_planes(rng, xb, batch * H * H, C // 32)
    kw = dict(batch=batch, H=H, W=H, cout=cout, R=3, S=3, stride=1, pad=1, halo=0, wb=wb, xb=xb)
    v = O.conv(W, X, cwords=C // 32, sym_w=1, **kw).reshape(-1, cout).astype(np.int64)
    extra, keep = {}, []
    if pool == 0 and ob != 3:
        short = rng.integers(0, 4, size=v.shape).astype(np.uint32)
        v = v + 1365 * short.astype(np.int64)
        keep.append(G.to_dev(O.pack_bits(short, v.shape[0], cout, cout, 2)))
        extra = dict(resid_planes=keep[-1], resid_bits=2, resid_scale=1365)
    elif pool == 0:
        res = rng.integers(-500, 500, size=v.shape).astype(np.int32)
        v = v + res
        keep += [G.to_dev(res), G.dev_empty_i32(v.size, fill=-7)]
        extra = dict(resid=keep[0], save=keep[1])
    if pool:  # windows in raster order, four values each
        v = v.reshape(batch, H // 2, 2, H // 2, 2, cout).transpose(0, 1, 3, 2, 4, 5).reshape(-1, 4, cout)
    if pool == 1:
        s = v.sum(axis=1)
        v = np.where(s < 0, -(-s // 4), s // 4)[:, None, :]
    v = v.reshape(-1, cout)
    if bn:
        thr = np.sort(rng.integers(v.min() - 5, v.max() + 6, size=(cout, 2 ** ob - 1)), axis=1).astype(np.int32)
        thr[0, :], thr[1, :] = np.iinfo(np.int32).min, np.iinfo(np.int32).max
        flip = rng.integers(0, 2, size=cout).astype(np.uint8)
        thr[flip != 0] = np.sort(-thr[flip != 0].astype(np.int64), axis=1).clip(-2 ** 31, 2 ** 31 - 1).astype(np.int32)
        keep += [G.to_dev(thr), G.to_dev(flip)]
        epi = G.epilogue(mode=G.A.EPI_BN, out_bits=ob, pool=pool, thr=keep[-2], flip=keep[-1], **extra)
        q = O.bn_quantize(v.astype(np.int32), None, thr, flip, ob)
    else:
        epi = G.epilogue(mode=G.A.EPI_LOWBITS, out_bits=ob, pool=pool, **extra)
        q = v & (2 ** ob - 1)
    q = np.asarray(q).astype(np.uint32).reshape(-1, cout)
    if pool == 2:
        q = np.ascontiguousarray(q.reshape(-1, 4, cout).max(axis=1))
    got = G.run_conv(W, X, cin_pad=C, sym=1, epi=epi, path=2, tile=tile, **kw).view(np.uint32).reshape(ob, -1, cout // 32)
    assert np.array_equal(got, O.lowbits_pack(q, q.shape[0], cout, ob))
    if "save" in extra:
        assert np.array_equal(G.to_host(keep[1]).reshape(v.shape), v)


def test_packer_beyond_one_grid(G):
    """More than 2^32 words: the packers' grid of one wave per 64 words would exceed the threads one launch may have."""
    rows, words = (2 ** 32 + 3 * 4096) // 3, 3
    if torch.cuda.mem_get_info()[0] < 40 * 2 ** 30:
        pytest.skip("needs 40 GB of device memory")
    x = torch.randint(0, 256, (rows,), dtype=torch.uint8, device="cuda")
    planes = torch.full((rows, words), -7, dtype=torch.int32, device="cuda")
    G.A.check(G.A.lib().apnn_quantize_pack_u8(G.ptr(x), G.ptr(planes), rows, 1, 32 * words, 1, None), "quantize_pack_u8")
    step = 1 << 28
    for r in range(0, rows, step):
        got = planes[r:r + step]
        assert torch.equal(got[:, 0] != 0, x[r:r + step] >= 128) and bool(((got[:, 0] == 0) | (got[:, 0] == -2 ** 31)).all())
        assert not bool(got[:, 1:].any())


# Sums just below 2^24 on the kernels that load straight to LDS, on convolutions and with FP6 digits: all-ones operands
# give the largest value the host admits, random ones are checked with the oracle.
@pytest.mark.parametrize("wb,xb", [(1, 2), (1, 4), (2, 2), (2, 8), (4, 4)])
@pytest.mark.parametrize("gemm,tile", [(1, 6), (1, 2), (0, 1), (0, 7), (0, 2), (0, 9)])
@pytest.mark.parametrize("sym", [0, 1])
def test_exact_just_below_the_limit(G, gemm, tile, wb, xb, sym):
    span = (2 ** wb - 1) * (2 ** xb - 1)
    K = 128 * (1 << ((2 ** 24 - 1) // span // 128).bit_length() - 1)  # words per pixel a power of two
    rows = cols = 32
    rng = np.random.default_rng(9100 + 10 * wb + xb)
    for W, X in ((np.full((wb, cols, K // 32), 0xFFFFFFFF, np.uint32), np.full((xb, rows, K // 32), 0xFFFFFFFF, np.uint32)),
                 (O.random_planes(rng, wb, cols, K // 32), O.random_planes(rng, xb, rows, K // 32))):
        if gemm:
            got = G.run_gemm(W, X, cols, rows, K, wb, xb, sym=sym, path=2, tile=tile).reshape(cols, rows)
        else:
            got = G.run_conv(W, X, batch=1, H=4, W=8, cin_pad=K, cout=cols, R=1, S=1, stride=1, pad=0, halo=0, wb=wb, xb=xb,
                             sym=sym, path=2, tile=tile).reshape(rows, cols).T
        assert np.array_equal(got, O.gemm(W, X, cols, rows, K, wb, xb, sym_w=sym, nthreads=8))


@pytest.mark.parametrize("path,tile", [(0, None), (1, 0), (1, 2), (2, 1), (2, 2), (2, 4), (2, 7), (2, 9), (3, 2), (5, 2)])
def test_very_long_single_tap(G, path, tile):
    """A 1x1 filter over 174760 words per pixel: the multiply-high that finds a word's tap is exact up to 65536 words."""
    K, rows, cols = 32 * 174760, 32, 32
    W, X = np.full((1, cols, K // 32), 0xFFFFFFFF, np.uint32), np.full((2, rows, K // 32), 0xFFFFFFFF, np.uint32)
    got = G.run_conv(W, X, batch=1, H=4, W=8, cin_pad=K, cout=cols, R=1, S=1, stride=1, pad=0, halo=0, wb=1, xb=2, sym=0,
                     path=path, tile=tile)
    assert np.all(got == 3 * K)


@pytest.mark.parametrize("path,tile", [(0, None), (1, 0), (1, 1), (1, 3)])
@pytest.mark.parametrize("words", [92820, 66466, 46779])
def test_taps_of_very_long_filters(G, path, tile, words):
    """Two taps of 128-, 64- and 32-bit loads over more channels than the multiply-high finds the tap of exactly."""
    rows, cols = 8, 32
    rng = np.random.default_rng(words)
    W, X = O.random_planes(rng, 1, cols * 2, words), O.random_planes(rng, 2, rows + 1, words)
    kw = dict(batch=1, H=1, W=rows + 1, cout=cols, R=1, S=2, stride=1, pad=0, halo=0, wb=1, xb=2)
    got = G.run_conv(W, X, cin_pad=32 * words, sym=0, path=path, tile=tile, **kw)
    assert np.array_equal(got.reshape(rows, cols), O.conv(W, X, cwords=words, sym_w=0, **kw).reshape(rows, cols))


# Patch-resident convolution: the forms of its kernel (any filter; 3x3 over an odd and over an even number of channel words; 5x5
# over an even one, run on the narrow tiles), one chunk of 64 channels and several, rows one past a tile and one short of it, a last column tile that is
# mostly empty, raw sums and codes with flips.
@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("wb,xb", [(1, 2), (1, 3), (1, 4), (2, 2)])
@pytest.mark.parametrize("H,Wd,C,cout,R,S,stride,sym", [
    (3, 43, 64, 96, 3, 3, 1, 1),     # 129 rows
    (15, 17, 192, 64, 3, 3, 1, 0),   # 255 rows, three chunks
    (11, 12, 96, 160, 3, 3, 1, 1),   # an odd last word
    (4, 16, 32, 32, 3, 3, 1, 0),     # one word
    (9, 14, 160, 64, 4, 2, 1, 1),    # general form, odd words
    (10, 10, 128, 32, 1, 1, 1, 1),   # one tap
    (12, 15, 64, 96, 5, 5, 1, 1),    # 130 rows
    (7, 9, 192, 64, 5, 5, 1, 0),     # three chunks
    (9, 60, 64, 96, 5, 5, 1, 1),     # patches of 640 (128x64) and 776 (256x64) pixels: they fit with the one digit of two planes
    (10, 58, 96, 64, 5, 5, 1, 0),    # the same over an odd number of words
])
def test_patch_conv_forms(G, wb, xb, tile, H, Wd, C, cout, R, S, stride, sym):
    if R == 5 and tile not in ((1, 3, 4) if xb == 2 else (3, 4)) or Wd > 50 and xb > 2:
        pytest.skip("the patch and the filter block of 25 taps do not fit")
    rng = np.random.default_rng(8700 + H + 10 * C + tile)
    pad = 1 if R > 1 else 0
    X, W = O.random_planes(rng, xb, H * Wd, C // 32), O.random_planes(rng, wb, cout * R * S, C // 32)
    kw = dict(batch=1, H=H, W=Wd, cout=cout, R=R, S=S, stride=stride, pad=pad, halo=0, wb=wb, xb=xb)
    acc = O.conv(W, X, cwords=C // 32, sym_w=sym, **kw).reshape(-1, cout)
    got = G.run_conv(W, X, cin_pad=C, sym=sym, path=G.A.PATH_MFMA_PATCH, tile=tile, **kw).reshape(acc.shape)
    assert np.array_equal(got, acc)
    sigma = max(int(acc.std()), 2)
    thr = np.sort(rng.integers(-sigma, sigma, size=(cout, (1 << xb) - 1)) + int(acc.mean()), axis=1).astype(np.int32)
    flip = rng.integers(0, 2, size=cout).astype(np.uint8)
    d_thr, d_flip = G.to_dev(thr), G.to_dev(flip)
    epi = G.epilogue(mode=G.A.EPI_BN, out_bits=xb, thr=d_thr, flip=d_flip)
    got = G.run_conv(W, X, cin_pad=C, sym=sym, epi=epi, path=G.A.PATH_MFMA_PATCH, tile=tile, **kw).view(np.uint32)
    expect = O.lowbits_pack(O.bn_quantize(acc, None, thr, flip, xb), acc.shape[0], cout, xb)
    assert np.array_equal(got.reshape(expect.shape), expect)


# Every output of the patch-resident convolution, in each form of its kernel: low bits, pooled averages and maxima, searched and
# compared codes of one to four bits, flips, a shortcut that the matrix cores add (with one and two digits a pixel, with
# weight operands of -1 / +1, of 0 / 1 and of two planes) and one that they do not, an int32 map with the sums saved.
@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("wb,xb,ob,sym", [(1, 2, 2, 1), (1, 2, 3, 0), (1, 3, 3, 1), (1, 4, 4, 1), (1, 4, 2, 0), (2, 2, 1, 0), (2, 2, 2, 1)])
@pytest.mark.parametrize("batch,H,C,R", [(3, 6, 128, 3), (2, 10, 96, 3), (3, 8, 64, 5), (2, 6, 160, 2)])
@pytest.mark.parametrize("out", ["low", "low_avg", "low_max", "near", "far", "map", "avg", "max"])
def test_patch_conv_output_forms(G, tile, wb, xb, ob, sym, batch, H, C, R, out):
    if R == 5 and tile not in ((1, 3, 4) if xb == 2 else (3, 4)):
        pytest.skip("the patch and the filter block of 25 taps do not fit")
    cout, pad, far = 96, R // 2, 1365
    rng = np.random.default_rng(9300 + 100 * tile + 10 * xb + ob + 3 * C + len(out))
    Ho = H + 2 * pad - R + 1
    if out[-3:] in ("avg", "max") and Ho % 2:
        H, Ho = H + 1, Ho + 1
    W, X = O.random_planes(rng, wb, cout * R * R, C // 32), O.random_planes(rng, xb, batch * H * H, C // 32)
    kw = dict(batch=batch, H=H, W=H, cout=cout, R=R, S=R, stride=1, pad=pad, halo=0, wb=wb, xb=xb)
    v = O.conv(W, X, cwords=C // 32, sym_w=sym, **kw).reshape(-1, cout).astype(np.int64)
    extra, keep, pool = {}, [], {"avg": 1, "max": 2}.get(out[-3:], 0)
    if out in ("near", "far"):
        scale = 12 if out == "near" else far
        short = rng.integers(0, 4, size=v.shape).astype(np.uint32)
        v = v + scale * short.astype(np.int64)
        keep.append(G.to_dev(O.pack_bits(short, v.shape[0], cout, cout, 2)))
        extra = dict(resid_planes=keep[-1], resid_bits=2, resid_scale=scale)
    elif out == "map":
        res = rng.integers(-500, 500, size=v.shape).astype(np.int32)
        v = v + res
        keep += [G.to_dev(res), G.dev_empty_i32(v.size, fill=-7)]
        extra = dict(resid=keep[0], save=keep[1])
    if pool:  # windows in raster order, four values each
        v = v.reshape(batch, Ho // 2, 2, Ho // 2, 2, cout).transpose(0, 1, 3, 2, 4, 5).reshape(-1, 4, cout)
    if pool == 1:
        s = v.sum(axis=1)
        v = np.where(s < 0, -(-s // 4), s // 4)[:, None, :]
    v = v.reshape(-1, cout)
    if out.startswith("low"):
        epi = G.epilogue(mode=G.A.EPI_LOWBITS, out_bits=ob, pool=pool)
        q = v & (2 ** ob - 1)
    else:
        thr = np.sort(rng.integers(v.min() - 5, v.max() + 6, size=(cout, 2 ** ob - 1)), axis=1).astype(np.int32)
        thr[0, :], thr[1, :] = np.iinfo(np.int32).min, np.iinfo(np.int32).max
        flip = rng.integers(0, 2, size=cout).astype(np.uint8)
        thr[flip != 0] = np.sort(-thr[flip != 0].astype(np.int64), axis=1).clip(-2 ** 31, 2 ** 31 - 1).astype(np.int32)
        keep += [G.to_dev(thr), G.to_dev(flip)]
        epi = G.epilogue(mode=G.A.EPI_BN, out_bits=ob, pool=pool, thr=keep[-2], flip=keep[-1], **extra)
        q = O.bn_quantize(v.astype(np.int32), None, thr, flip, ob)
    q = np.asarray(q).astype(np.uint32).reshape(-1, cout)
    if pool == 2:
        q = np.ascontiguousarray(q.reshape(-1, 4, cout).max(axis=1))
    got = G.run_conv(W, X, cin_pad=C, sym=sym, epi=epi, path=G.A.PATH_MFMA_PATCH, tile=tile, **kw).view(np.uint32)
    assert np.array_equal(got.reshape(ob, -1, cout // 32), O.lowbits_pack(q, q.shape[0], cout, ob))
    if out == "map":
        assert np.array_equal(G.to_host(keep[1]).reshape(v.shape), v)
