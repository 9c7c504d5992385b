"""GEMM tiles whose eight waves split K (128x64 by four, 64x96 by eight): edges of the tiles and of the 1024-bit chunks, every
result form, and the sizes at which AUTO takes them."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O
import pkg

A = pkg.load()
K4, K8 = 10, 11
BUILT = [(K4, 1, 2), (K4, 1, 3), (K4, 1, 4), (K4, 2, 2), (K4, 1, 8), (K4, 4, 4), (K8, 4, 4)]


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


@pytest.mark.gpu
@pytest.mark.parametrize("sym", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (129, 65, 1152), (63, 97, 1024), (128, 192, 896), (257, 31, 3200)])
@pytest.mark.parametrize("tile,wb,xb", BUILT)
def test_ksplit_int32(G, tile, wb, xb, M, N, K, sym):
    """One row past a tile and one short of it; reductions that end inside, at and just past a chunk."""
    rng = np.random.default_rng(9700 + M + 10 * wb + xb + tile)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=sym, path=A.PATH_MFMA, tile=tile).reshape(M, N)
    assert np.array_equal(got, O.gemm(W, X, M, N, K, wb, xb, sym_w=sym))


@pytest.mark.gpu
@pytest.mark.parametrize("tile,wb,xb", BUILT)
@pytest.mark.parametrize("columns", [2, 24])
def test_ksplit_bands(G, tile, wb, xb, columns):
    """At least 256 tiles, a multiple of eight, in two columns and more: the order of the bands of an XCD, with a last band that is
    not full (132 rows of tiles; 11)."""
    ta, tb = (128, 64) if tile == K4 else (64, 96)
    M, N, K = (132 if columns == 2 else 11) * ta - 5, columns * tb - 7, 128
    rng = np.random.default_rng(9770 + 10 * wb + xb + tile)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=1, path=A.PATH_MFMA, tile=tile).reshape(M, N)
    assert np.array_equal(got, O.gemm(W, X, M, N, K, wb, xb, sym_w=1))


@pytest.mark.gpu
@pytest.mark.parametrize("sym", [0, 1])
@pytest.mark.parametrize("K", list(range(128, 1025, 128)) + list(range(1152, 3073, 128)))
@pytest.mark.parametrize("tile,wb,xb", BUILT)
def test_ksplit_last_chunk(G, tile, wb, xb, K, sym):
    """Every number of words in the last chunk, which up to half of them are spread over the waves, alone and behind one and two
    full ones; all-ones operands and ones with a single word set show a word that is counted twice or left out."""
    M, N = 97, 70
    rng = np.random.default_rng(9750 + K + 10 * wb + xb + tile)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    W[:, :4], X[:, :3] = 0xFFFFFFFF, 0xFFFFFFFF
    for n in range(K // 32):
        if 8 + n < M:
            W[:, 8 + n] = 0
            W[:, 8 + n, n] = 0xFFFFFFFF
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=sym, path=A.PATH_MFMA, tile=tile).reshape(M, N)
    assert np.array_equal(got, O.gemm(W, X, M, N, K, wb, xb, sym_w=sym))


@pytest.mark.gpu
@pytest.mark.parametrize("tile,wb,xb", BUILT)
@pytest.mark.parametrize("bits,form", [(2, "low"), (1, "bn"), (2, "bn"), (4, "bn"), (5, "bn"), (2, "near"), (2, "far"), (2, "map")])
def test_ksplit_packed(G, tile, wb, xb, bits, form):
    """Low bits, threshold codes, shortcuts that fold into the matrix cores (near) or not (far), int32 maps with saved sums."""
    M, N, K, sym = 141, 160, 1152, int(form != "low")
    rng = np.random.default_rng(9800 + 10 * wb + xb + tile + bits)
    W, X = O.random_planes(rng, wb, M, K // 32), O.random_planes(rng, xb, N, K // 32)
    acc = O.gemm(W, X, M, N, K, wb, xb, sym_w=sym)
    if form == "low":
        got = G.run_gemm(W, X, M, N, K, wb, xb, epi=G.epilogue(mode=A.EPI_LOWBITS, out_bits=bits), path=A.PATH_MFMA, tile=tile)
        assert np.array_equal(got.view(np.uint32).reshape(bits, M, N // 32), O.lowbits_pack(acc, M, N, bits))
        return
    spread = int(acc.std()) + 1
    thr = np.sort(rng.integers(-2 * spread, 2 * spread, size=(N, 2 ** bits - 1)), axis=1).astype(np.int32)
    flip = rng.integers(0, 2, size=N).astype(np.uint8)
    kw, keep, resid = {}, [G.to_dev(thr), G.to_dev(flip)], None
    if form == "map":
        resid = rng.integers(-spread, spread, size=(M, N)).astype(np.int32)
        keep += [G.to_dev(resid), G.dev_empty_i32(M * N, fill=-7)]
        kw = dict(resid=keep[2], save=keep[3])
    elif form in ("near", "far"):
        scale = 12 if form == "near" else 1365
        codes = rng.integers(0, 4, size=(M, N)).astype(np.uint32)
        resid = (codes * scale).astype(np.int32)
        keep.append(G.to_dev(O.pack_bits(codes, M, N, N, 2)))
        kw = dict(resid_planes=keep[2], resid_bits=2, resid_scale=scale)
    epi = G.epilogue(mode=A.EPI_BN, out_bits=bits, thr=keep[0], flip=keep[1], **kw)
    got = G.run_gemm(W, X, M, N, K, wb, xb, sym=sym, epi=epi, path=A.PATH_MFMA, tile=tile).view(np.uint32).reshape(bits, M, N // 32)
    assert np.array_equal(got, O.lowbits_pack(O.bn_quantize(acc, resid, thr, flip, bits), M, N, bits))
    if form == "map":
        assert np.array_equal(G.to_host(keep[3]).reshape(M, N), acc + resid)


@pytest.mark.parametrize("M,N,K,wb,xb,tile", [
    (1000, 2016, 1024, 1, 2, K4), (1000, 2016, 896, 1, 2, None), (1000, 2016, 1024, 2, 2, None), (1000, 2016, 2048, 2, 2, K4),
    (1024, 768, 2048, 1, 4, K4), (512, 1024, 2048, 1, 4, None), (1000, 1000, 2048, 2, 2, None), (2304, 1024, 2048, 1, 2, None),
    (2048, 2048, 2048, 1, 8, K4), (4096, 4096, 2048, 1, 8, None), (1000, 2016, 2048, 2, 8, None), (1000, 2016, 2048, 1, 1, None),
    (4096, 333, 4096, 4, 4, K8), (4096, 333, 1024, 4, 4, K4), (1000, 1000, 4096, 4, 4, K8), (1000, 2016, 4096, 4, 4, K4),
    (8192, 16, 2048, 1, 2, None), (16, 8192, 2048, 1, 2, None),
    # up to half a tile per unit a begun chunk costs w1a2 and w1a3 more than it gains
    (1024, 768, 1024, 1, 2, K4), (1024, 768, 1152, 1, 2, None), (1000, 1000, 1920, 1, 2, None), (1000, 1000, 4224, 1, 2, None),
    (1024, 768, 2048, 1, 3, K4), (1024, 768, 1152, 1, 3, None), (1000, 1000, 2304, 1, 3, None), (1000, 1000, 2432, 1, 3, K4),
    (1000, 1000, 1152, 1, 4, K4), (768, 1536, 1152, 1, 2, K4), (768, 1536, 1152, 1, 3, K4),
    # a little more than half a tile per unit, partly empty: the 32x64 tile has 512 blocks at most
    (408, 2272, 2304, 2, 2, None), (898, 1044, 1152, 4, 4, None), (348, 2720, 1152, 1, 2, None), (348, 2720, 2048, 1, 2, K4),
    (1000, 1152, 1152, 4, 4, K4), (1000, 1152, 2048, 2, 2, K4),
])
def test_ksplit_rule(M, N, K, wb, xb, tile):
    """Where AUTO takes these tiles: one round of at least 3/8 (1/2) of the units, 1024 bits, tiles mostly filled."""
    plan = A.Plan()
    d = A.GemmDesc(W=0x1000, X=0x1000, D=0x1000, M=M, N=N, K=K, wb=wb, xb=xb, path=A.PATH_AUTO)
    assert A.lib().apnn_gemm_plan(ctypes.byref(d), ctypes.byref(plan)) == 0
    assert plan.kernel == A.KERNEL_MFMA_FP4
    assert (plan.tile if plan.tile in (K4, K8) else None) == tile
    if tile is not None:
        assert (plan.tile_rows, plan.tile_cols, plan.split_k) == ((128, 64, 4) if tile == K4 else (64, 96, 8))
