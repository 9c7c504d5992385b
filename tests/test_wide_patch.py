"""The 128x128 convolution tile over a patch of expanded activations with packed weights: edges of tiles, passes of 256 channels
and weight chunks, every result form, and the layers at which AUTO takes it."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O
import pkg

A = pkg.load()
TILE = 12
COMBOS = [(1, 2), (1, 3), (1, 4), (2, 2)]


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# images smaller than a tile and several tiles long, one to three passes, one tap to 25, rectangular frames and filters, no
# padding, a stored halo, channels that end inside a tile
GEOMS = [(1, 5, 5, 256, 32, 3, 3, 1, 0), (2, 9, 9, 512, 160, 3, 3, 1, 0), (3, 14, 14, 768, 128, 3, 3, 1, 0), (2, 8, 8, 256, 96, 5, 5, 2, 0),
         (2, 7, 11, 512, 256, 3, 2, 1, 0), (40, 3, 3, 256, 32, 3, 3, 1, 0), (1, 20, 30, 256, 288, 3, 3, 0, 0), (2, 16, 12, 512, 96, 3, 3, 1, 1),
         (1, 16, 9, 768, 64, 1, 1, 0, 0), (1, 6, 25, 256, 32, 2, 2, 0, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", COMBOS)
@pytest.mark.parametrize("B,H,Wd,C,cout,R,S,pad,halo", GEOMS)
@pytest.mark.parametrize("sym,mode", [(0, "int32"), (1, "int32"), (1, "bn"), (0, "shortcut"), (1, "shortcut")])
def test_wide_patch_geometry(G, wb, xb, B, H, Wd, C, cout, R, S, pad, halo, sym, mode):
    rng = np.random.default_rng(9900 + C + cout + 10 * wb + xb)
    grow = 2 * pad if halo else 0
    X = O.random_planes(rng, xb, B * (H + grow) * (Wd + grow), C // 32)
    Wt = O.random_planes(rng, wb, cout * R * S, C // 32)
    kw = dict(batch=B, H=H, W=Wd, cout=cout, R=R, S=S, stride=1, pad=pad, halo=halo, wb=wb, xb=xb)
    acc = O.conv(Wt, X, cwords=C // 32, sym_w=sym, nthreads=8, **kw).reshape(-1, cout)
    rows = acc.shape[0]
    if mode == "int32":
        assert np.array_equal(G.run_conv(Wt, X, cin_pad=C, sym=sym, path=2, tile=TILE, **kw).reshape(rows, cout), acc)
        return
    thr = np.sort(rng.integers(acc.min(), acc.max() + 1, size=(cout, (1 << xb) - 1)), axis=1).astype(np.int32)
    keep, extra, value = [G.to_dev(thr)], {}, acc
    if mode == "shortcut":
        codes = rng.integers(0, 4, size=(rows, cout)).astype(np.uint32)
        keep.append(G.to_dev(O.pack_bits(codes, rows, cout, cout, 2)))
        extra = dict(resid_planes=keep[1], resid_bits=2, resid_scale=5)
        value = acc + 5 * codes.astype(np.int32)
    epi = G.epilogue(mode=A.EPI_BN, out_bits=xb, thr=keep[0], **extra)
    got = G.run_conv(Wt, X, cin_pad=C, sym=sym, epi=epi, path=2, tile=TILE, **kw).view(np.uint32).reshape(xb, rows, cout // 32)
    assert np.array_equal(got, O.lowbits_pack(O.bn_quantize(value, None, thr, None, xb), rows, cout, xb))


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", COMBOS)
@pytest.mark.parametrize("B,H,Wd,R,S,stride", [(90, 3, 1, 3, 1, 2), (40, 12, 1, 4, 1, 2), (90, 2, 3, 1, 1, 2), (60, 9, 1, 3, 1, 3), (9, 39, 3, 1, 1, 2)])
def test_wide_patch_strides(G, wb, xb, B, H, Wd, R, S, stride):
    """A tile's patch is sized for 128 pixels anywhere: only maps a few pixels wide fit one of stride 2 or 3."""
    rng = np.random.default_rng(9920 + H + 10 * wb + xb)
    C, cout = 512, 96
    X, Wt = O.random_planes(rng, xb, B * H * Wd, C // 32), O.random_planes(rng, wb, cout * R * S, C // 32)
    kw = dict(batch=B, H=H, W=Wd, cout=cout, R=R, S=S, stride=stride, pad=0, halo=0, wb=wb, xb=xb)
    acc = O.conv(Wt, X, cwords=C // 32, sym_w=1, nthreads=8, **kw).reshape(-1)
    assert np.array_equal(G.run_conv(Wt, X, cin_pad=C, sym=1, path=2, tile=TILE, **kw), acc)


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", COMBOS)
@pytest.mark.parametrize("B,H,cout", [(20, 30, 160), (6, 28, 1000)])
def test_wide_patch_bands(G, wb, xb, B, H, cout):
    """At least 256 tiles, a multiple of eight, in two columns and more: the order of the bands of an XCD, with a last band
    that is not full (132 rows of tiles; 35)."""
    rows = B * (H - 1) ** 2
    assert (-(-rows // 128) * -(-cout // 128)) % 8 == 0 and -(-rows // 128) * -(-cout // 128) >= 256
    rng = np.random.default_rng(9940 + H + 10 * wb + xb)
    C, R = 256, 2
    X, Wt = O.random_planes(rng, xb, B * H * H, C // 32), O.random_planes(rng, wb, cout * R * R, C // 32)
    kw = dict(batch=B, H=H, W=H, cout=cout, R=R, S=R, stride=1, pad=0, halo=0, wb=wb, xb=xb)
    acc = O.conv(Wt, X, cwords=C // 32, sym_w=1, nthreads=8, **kw).reshape(-1)
    assert np.array_equal(G.run_conv(Wt, X, cin_pad=C, sym=1, path=2, tile=TILE, **kw), acc)


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb", COMBOS)
@pytest.mark.parametrize("bits,pool,save", [(1, 0, 1), (2, 0, 1), (4, 0, 0), (5, 0, 0), (2, 1, 0), (2, 2, 0), (3, 2, 0)])
@pytest.mark.parametrize("low", [0, 1])
def test_wide_patch_outputs(G, wb, xb, bits, pool, save, low):
    """Low bits and threshold codes, pooled windows (pixels in pool order) and int32 maps added and saved."""
    rng = np.random.default_rng(9950 + 10 * xb + bits + pool)
    B, H, C, cout = 3, 10, 512, 160
    Wt, X = O.random_planes(rng, wb, cout * 9, C // 32), O.random_planes(rng, xb, B * H * H, C // 32)
    kw = dict(batch=B, H=H, W=H, cout=cout, R=3, S=3, stride=1, pad=1, halo=0, wb=wb, xb=xb)
    v = O.conv(Wt, X, cwords=C // 32, sym_w=1, nthreads=8, **kw).reshape(-1, cout)
    keep, extra = [], {}
    if save:
        res = rng.integers(-500, 500, size=v.shape).astype(np.int32)
        v = v + res
        keep = [G.to_dev(res), G.dev_empty_i32(v.size, fill=-7)]
        extra = dict(resid=keep[0], save=keep[1])
    full = v
    if pool:
        v = v.reshape(B, H // 2, 2, H // 2, 2, cout).transpose(0, 1, 3, 2, 4, 5).reshape(-1, 4, cout)
        if pool == 1:
            s = v.astype(np.int64).sum(axis=1)
            v = np.where(s < 0, -(-s // 4), s // 4)[:, None, :]
        v = np.ascontiguousarray(v.reshape(-1, cout)).astype(np.int32)
    if low:
        epi, q = G.epilogue(mode=A.EPI_LOWBITS, out_bits=bits, pool=pool, **extra), v & (2 ** bits - 1)
    else:
        thr = np.sort(rng.integers(v.min(), v.max() + 1, size=(cout, 2 ** bits - 1)), axis=1).astype(np.int32)
        flip = rng.integers(0, 2, size=cout).astype(np.uint8)
        keep += [G.to_dev(thr), G.to_dev(flip)]
        epi = G.epilogue(mode=A.EPI_BN, out_bits=bits, pool=pool, thr=keep[-2], flip=keep[-1], **extra)
        q = O.bn_quantize(v, None, thr, flip, bits)
    q = np.asarray(q).astype(np.uint32).reshape(-1, cout)
    if pool == 2:
        q = np.ascontiguousarray(q.reshape(-1, 4, cout).max(axis=1))
    got = G.run_conv(Wt, X, cin_pad=C, sym=1, epi=epi, path=2, tile=TILE, **kw).view(np.uint32).reshape(bits, -1, cout // 32)
    assert np.array_equal(got, O.lowbits_pack(q, q.shape[0], cout, bits))
    if save:
        assert np.array_equal(G.to_host(keep[1]).reshape(full.shape), full)


@pytest.mark.gpu
@pytest.mark.parametrize("wb,xb,K", [(2, 2, 1024000), (1, 4, 640000), (1, 2, 3200000)])
def test_wide_patch_shortcut_beside_large_sums(G, wb, xb, K):
    """Raw sums between 2^23 and 2^24: all-ones operands make the codes the shortcut's when no half unit is rounded away."""
    v, rows, cols = K * (2 ** wb - 1) * (2 ** xb - 1), 32, 32
    codes = np.random.default_rng(9970 + xb).integers(0, 4, size=(rows, cols)).astype(np.uint32)
    W, X = np.full((wb, cols, K // 32), 0xFFFFFFFF, np.uint32), np.full((xb, rows, K // 32), 0xFFFFFFFF, np.uint32)
    thr = (v + np.repeat(np.arange(1, 4, dtype=np.int64)[None, :], cols, axis=0)).astype(np.int32)
    keep = [G.to_dev(thr), G.to_dev(O.pack_bits(codes, rows, cols, cols, 2))]
    epi = G.epilogue(mode=A.EPI_BN, out_bits=2, thr=keep[0], resid_planes=keep[1], resid_bits=2, resid_scale=1)
    got = G.run_conv(W, X, batch=1, H=4, W=8, cin_pad=K, cout=cols, R=1, S=1, stride=1, pad=0, halo=0, wb=wb, xb=xb, sym=1,
                     epi=epi, path=2, tile=TILE)
    assert np.array_equal(got.view(np.uint32).reshape(2, rows, cols // 32), O.lowbits_pack(codes, rows, cols, 2))


def _plan(batch, H, W, C, cout, R, S, stride, pad, wb, xb, path=A.PATH_AUTO, pool=0):
    plan, epi = A.Plan(), A.Epilogue()
    if pool:
        epi.mode, epi.out_bits, epi.pool = A.EPI_LOWBITS, 2, pool
    d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=batch, H=H, Wd=W, cin_pad=C, COUT=cout, R=R, S=S, stride=stride,
                   pad=pad, halo=0, wb=wb, xb=xb, epi=epi, path=path)
    return A.lib().apnn_conv_plan(ctypes.byref(d), ctypes.byref(plan)), plan


@pytest.mark.parametrize("B,H,C,cout,R,stride,combos", [
    (64, 14, 512, 512, 3, 1, COMBOS), (64, 28, 512, 512, 3, 1, COMBOS), (12, 28, 512, 512, 3, 1, COMBOS), (64, 14, 512, 512, 5, 1, COMBOS),
    (48, 28, 512, 512, 3, 1, COMBOS),
    (64, 14, 512, 1024, 3, 1, []), (40, 28, 512, 512, 3, 1, []),    # 784, 980 tiles: a second round
    (56, 28, 512, 512, 3, 1, [(1, 4), (2, 2)]), (30, 56, 512, 256, 3, 1, []),      # 686, 735 tiles of 128x256: most of a round
    (56, 28, 512, 416, 3, 1, [(1, 4), (2, 2)]), (56, 28, 512, 384, 3, 1, COMBOS),           # their columns mostly and half filled
    (64, 28, 512, 512, 1, 1, []), (64, 28, 512, 512, 3, 2, []),     # nothing to keep; a patch of 636 pixels and more
    (64, 56, 256, 256, 3, 1, [(1, 2)]), (64, 14, 384, 512, 3, 1, []),   # two work-groups a unit or a large patch; a pass and a half
    (32, 14, 512, 512, 3, 1, COMBOS), (8, 28, 512, 512, 3, 1, COMBOS), (64, 7, 512, 1024, 3, 1, COMBOS),  # three tiles to four units
    (31, 14, 512, 512, 3, 1, []), (16, 16, 1024, 1024, 3, 1, []), (64, 7, 512, 512, 3, 1, []),    # the split tiles keep theirs
    (35, 28, 768, 32, 3, 1, []), (33, 28, 256, 64, 3, 1, []), (50, 16, 512, 160, 3, 1, []),       # columns mostly empty
    (31, 28, 512, 96, 3, 1, []), (40, 28, 512, 96, 3, 1, COMBOS),                                 # three quarters full, below and above
    (18, 28, 1024, 160, 3, 1, COMBOS), (18, 28, 768, 160, 3, 1, [(2, 2)]), (12, 28, 768, 288, 5, 1, COMBOS[:3]),  # 1323 and 1470 blocks of 32x64: by the reduction
])
def test_wide_patch_rule(B, H, C, cout, R, stride, combos):
    for wb, xb in COMBOS + [(1, 8), (2, 8), (1, 1), (4, 4)]:
        rc, plan = _plan(B, H, H, C, cout, R, R, stride, R // 2, wb, xb)
        assert rc == 0 and (plan.kernel == A.KERNEL_MFMA_FP4 and plan.tile == TILE) == ((wb, xb) in combos), (wb, xb, plan.tile)
        if (wb, xb) in combos:  # the plan's own pin repeats it
            assert 0 < plan.patch_pixels <= 384 and (plan.tile_rows, plan.tile_cols, plan.split_k) == (128, 128, 1)
            rc, pinned = _plan(B, H, H, C, cout, R, R, stride, R // 2, wb, xb, path=plan.path | ((TILE + 1) << 8))
            assert rc == 0 and (pinned.tile, pinned.patch_pixels) == (TILE, plan.patch_pixels)


@pytest.mark.parametrize("C,xb,tile", [(512, 3, 5), (768, 3, 5), (1024, 3, TILE), (512, 2, TILE), (512, 4, TILE)])
def test_wide_patch_rule_general_results(C, xb, tile):
    """w1a3 maxima of three-bit codes stay on the 32x64 split-K tile over up to 216 words (33x28x28, 203 tiles)."""
    plan, epi = A.Plan(), A.Epilogue()
    epi.mode, epi.out_bits, epi.pool, epi.thresholds = A.EPI_BN, xb, A.POOL_MAX2X2, 0x1000
    d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=33, H=28, Wd=28, cin_pad=C, COUT=128, R=3, S=3, stride=1, pad=1, halo=0, wb=1,
                   xb=xb, epi=epi, path=A.PATH_AUTO)
    assert A.lib().apnn_conv_plan(ctypes.byref(d), ctypes.byref(plan)) == 0 and plan.kernel == A.KERNEL_MFMA_FP4 and plan.tile == tile


@pytest.mark.parametrize("B,H,W,R,S,stride,pad,pool", [
    (3, 16, 16, 3, 3, 1, 1, 0), (2, 28, 28, 3, 3, 1, 1, 0), (5, 7, 7, 3, 3, 1, 1, 0), (2, 13, 11, 5, 5, 1, 2, 0), (2, 12, 20, 3, 3, 1, 1, 1),
    (9, 5, 6, 3, 3, 1, 1, 0), (7, 6, 6, 3, 3, 1, 1, 1), (70, 3, 3, 3, 3, 1, 1, 0), (1, 40, 6, 1, 5, 1, 2, 0), (3, 9, 8, 2, 2, 2, 0, 0),
    (1, 2, 90, 3, 3, 1, 1, 0), (2, 8, 64, 3, 3, 1, 1, 2), (2, 14, 14, 3, 3, 2, 1, 0)])
def test_wide_patch_span(B, H, W, R, S, stride, pad, pool):
    """No tile of consecutive output pixels reads more of the padded frame than the host sizes the patch for, nor more than
    three half pixels a thread; a larger patch is refused."""
    Ho, Wo = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - S) // stride + 1
    PH, PW = H + pad, W + pad  # the padding after a row or an image is that before the next
    b, y, x = np.meshgrid(np.arange(B), np.arange(Ho), np.arange(Wo), indexing="ij")
    base = (b * PH + y * stride) * PW + x * stride
    if pool:
        base = base.reshape(B, Ho // 2, 2, Wo // 2, 2).transpose(0, 1, 3, 2, 4)
    base = base.reshape(-1)
    rc, plan = _plan(B, H, W, 256, 64, R, S, stride, pad, 1, 2, path=A.PATH_MFMA | ((TILE + 1) << 8), pool=pool)
    spans = [int(t.max() - t.min()) + (R - 1) * PW + S for t in np.split(base, range(128, base.size, 128))]
    if rc == A.EUNSUPPORTED:
        assert plan.patch_pixels == 0
        return
    assert rc == 0 and np.all(np.diff(base.reshape(-1, 4)[:, 0] if pool else base) > 0) and max(spans) <= plan.patch_pixels <= 384


@pytest.mark.parametrize("C,wb,xb,path", [(384, 1, 2, A.PATH_MFMA), (128, 1, 4, A.PATH_MFMA), (256, 1, 8, A.PATH_MFMA), (256, 4, 4, A.PATH_MFMA),
                                          (256, 1, 2, A.PATH_MFMA_I8)])
def test_wide_patch_refuses(C, wb, xb, path):
    assert _plan(2, 8, 8, C, 64, 3, 3, 1, 1, wb, xb, path=path | ((TILE + 1) << 8))[0] == A.EUNSUPPORTED
