"""The work that performance is judged on: what a user of this library has it do, through its public entry
points, over the sizes and precisions that its benchmark, tests and networks use.

  gemm      apnn_gemm: bit-plane matrix products.  From the M = 64 products of one small batch (one launch, a
            few microseconds) to 8192 x 8192 x 8192; int32 results or low-bit packed ones; weights of -1 / +1
            (symmetric) or unsigned planes; every precision that has a named entry point.
  conv      apnn_conv and the named apconv_* entry points: 1x1, 3x3 and 5x5 filters on 7x7 .. 56x56 maps,
            batch 1 .. 64, int32 results or the fused threshold quantizer, with max-pooling or a packed shortcut.
  net       apnn_net_forward: a whole forward pass, images in and logits out, batch 1 .. 64.
  quantize  apnn_quantize_pack: float activations to bit-planes, the way into the low-bit path.

run() enqueues on torch's current stream and returns the output buffers of the state, as a serving loop does.
"""
import ctypes
import importlib.util
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "apnn-tc_amd")
_NETS = {"alexnet": 0, "resnet18": 1, "vgg": 2}
_GEMM_BITS = ((1, 2), (1, 2), (1, 2), (1, 3), (1, 4), (2, 2), (1, 1), (1, 8), (2, 8), (4, 4))
_CONV_BITS = ((1, 2), (1, 2), (1, 2), (1, 3), (1, 4), (2, 2), (1, 5), (2, 6), (1, 8), (2, 8))  # (weights, activations)
_TOP = 8192 ** 3  # products of the largest GEMM (at two plane pairs)


def _package():
    """This repository's package: its folder name has a hyphen, so it is loaded by path."""
    if "apnn_tc_amd" not in sys.modules:
        pkg = os.path.join(os.getcwd(), "apnn-tc_amd")
        pkg = pkg if os.path.isdir(pkg) else _PKG
        spec = importlib.util.spec_from_file_location("apnn_tc_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["apnn_tc_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["apnn_tc_amd"]


def _gemm(M, N, K, wb, xb, sym=1, out="int32", name=None):
    c = {"kind": "gemm", "M": M, "N": N, "K": K, "wb": wb, "xb": xb, "sym": sym, "out": out}
    return dict(c, name=name) if name else c


def _conv(batch, H, C, cout, R, stride, wb, xb, out, named=0, name=None):
    c = {"kind": "conv", "batch": batch, "H": H, "C": C, "cout": cout, "R": R, "stride": stride, "wb": wb, "xb": xb,
         "out": out, "named": named}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one small batch against a square layer: the reference's headline product, all launch and latency
        _gemm(64, 1024, 1024, 1, 2, name="gemm_w1a2_m64"),
        # ragged middle sizes with the low bits of the result packed for a next product (apmm_w2a2_decompose)
        _gemm(1000, 2016, 2048, 2, 2, sym=0, out="lowbits", name="gemm_w2a2_ragged_packed"),
        # a 4096-wide layer over a few hundred rows of 4-bit activations and weights
        _gemm(4096, 333, 4096, 4, 4, sym=0, name="gemm_w4a4_rows"),
        # large square products: four-bit activations, and the main precision at the largest size
        _gemm(4096, 4096, 4096, 1, 4, name="gemm_w1a4_4096"),
        _gemm(8192, 8192, 8192, 1, 2, name="gemm_w1a2_8192"),
        # 3x3 convolution of one image on a stored halo through the named entry point (the reference's sweep)
        _conv(1, 16, 512, 512, 3, 1, 1, 2, "int32", named=1, name="conv_w1a2_b1"),
        # a batched hidden layer with its threshold quantizer fused
        _conv(16, 16, 512, 512, 3, 1, 1, 3, "bn", name="conv_w1a3_b16_bn"),
        # whole networks: small batches, where 10 to 20 launches of a few microseconds follow each other, and large ones
        {"kind": "net", "net": "alexnet", "batch": 8, "name": "alexnet_b8"},
        {"kind": "net", "net": "resnet18", "batch": 8, "name": "resnet18_b8"},
        {"kind": "net", "net": "resnet18", "batch": 64, "name": "resnet18_b64"},
        {"kind": "net", "net": "vgg", "batch": 64, "name": "vgg_b64"},
        # float activations of a 56x56x64 map, batch 64, to two-bit planes: memory traffic only
        {"kind": "quantize", "rows": 200704, "C": 64, "bits": 2, "name": "quantize_56x56x64_b64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "conv", "conv", "net", "quantize"))
    if kind == "gemm":
        wb, xb = rng.choice(_GEMM_BITS)
        out = rng.choice(("int32", "int32", "lowbits"))
        K = 128 * _log(rng, 1, 64)
        while True:
            M, N = _log(rng, 16, 8192), _log(rng, 16, 8192)
            if out == "lowbits":
                N = 32 * max(1, N // 32)
            if M * N * K * max(1, wb * xb // 2) <= _TOP:
                break
        return _gemm(M, N, K, wb, xb, sym=rng.choice((0, 1)), out=out)
    if kind == "conv":
        wb, xb = rng.choice(_CONV_BITS)
        R = rng.choice((1, 3, 3, 3, 5))
        out = rng.choice(("int32", "bn", "bn", "bn_pool", "bn_shortcut"))
        while True:
            H, batch = rng.choice((7, 13, 14, 16, 27, 28, 32, 56)), _log(rng, 1, 64)
            C, cout = 32 * _log(rng, 1, 16 if R == 5 else 32), 32 * _log(rng, 1, 32)
            stride = 1 if out == "bn_pool" else rng.choice((1, 1, 1, 2))
            if out == "bn_pool" and H % 2:
                continue
            if batch * H * H * R * R * C * cout * max(1, wb * xb // 2) <= _TOP // 4:
                break
        return _conv(batch, H, C, cout, R, stride, wb, xb, out)
    if kind == "net":
        return {"kind": "net", "net": rng.choice(("alexnet", "resnet18", "resnet18", "vgg")), "batch": _log(rng, 1, 64)}
    while True:
        rows, C = _log(rng, 64, 400000), _log(rng, 16, 1024)
        if rows * C <= 200704 * 64 * 2:
            return {"kind": "quantize", "rows": rows, "C": C, "bits": rng.choice((1, 2, 2, 3, 4, 8))}


class _Net:
    """A network handle that is destroyed with its state."""

    def __init__(self, kind, batch, seed):
        A = _package()
        self._lib = A.nn_lib()
        self.handle = self._lib.apnn_net_create(kind, batch, seed, A.PATH_AUTO)
        if not self.handle:
            raise RuntimeError("apnn_net_create failed")

    def __del__(self):
        if getattr(self, "handle", None):
            torch.cuda.synchronize()
            self._lib.apnn_net_destroy(self.handle)
            self.handle = None


def _planes(gen, planes, words):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, (planes, words), dtype=torch.int32, device="cuda", generator=gen)


def _thresholds(gen, channels, bits, sigma, center=0.0):
    """Ascending thresholds that give every code about the same share of values of that spread."""
    steps = (1 << bits) - 1
    q = (torch.arange(1, steps + 1, device="cuda", dtype=torch.float64) / (steps + 1)) * 2 - 1
    mid = center + sigma * math.sqrt(2.0) * torch.erfinv(q)
    jitter = 0.1 * sigma * torch.randn((channels, 1), dtype=torch.float64, device="cuda", generator=gen)
    return (mid[None, :] + jitter).round().to(torch.int32).contiguous()


def _sigma(n, wb, xb):
    """Spread of a sum of n products of uniform symmetric weights and uniform activation codes."""
    a, w = (1 << xb) - 1, (1 << wb) - 1
    return math.sqrt(n * (a * (2 * a + 1) / 6.0) * ((w * w + 2 * w) / 3.0))


def _out_bits(case):
    return min(case["xb"], 8)


def prepare(case, seed):
    A = _package()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    s = {"kind": case["kind"], "A": A}
    if case["kind"] == "gemm":
        M, N, K, wb, xb = (case[k] for k in ("M", "N", "K", "wb", "xb"))
        W, X = _planes(gen, wb, M * K // 32), _planes(gen, xb, N * K // 32)
        epi = A.Epilogue()
        if case["out"] == "lowbits":
            epi.mode, epi.out_bits = A.EPI_LOWBITS, _out_bits(case)
            out = torch.zeros((epi.out_bits, M, N // 32), dtype=torch.int32, device="cuda")
        else:
            out = torch.zeros((M, N), dtype=torch.int32, device="cuda")
        desc = A.GemmDesc(W=W.data_ptr(), X=X.data_ptr(), D=out.data_ptr(), M=M, N=N, K=K, wb=wb, xb=xb,
                          weight_mode=case["sym"], epi=epi, path=A.PATH_AUTO)
        s.update(fn=A.lib().apnn_gemm, desc=desc, ref=ctypes.byref(desc), out=out, keep=(W, X))
    elif case["kind"] == "conv":
        batch, H, C, cout, R, stride, wb, xb = (case[k] for k in ("batch", "H", "C", "cout", "R", "stride", "wb", "xb"))
        pad = (R - 1) // 2
        Ho = (H + 2 * pad - R) // stride + 1
        rows, W = batch * Ho * Ho, _planes(gen, wb, cout * R * R * C // 32)
        if case["named"]:  # halo stored, contents of the halo zero
            X = torch.zeros((xb, batch, H + 2 * pad, H + 2 * pad, C // 32), dtype=torch.int32, device="cuda")
            X[:, :, pad:H + pad, pad:H + pad] = _planes(gen, xb, batch * H * H * C // 32).view(xb, batch, H, H, C // 32)
            out = torch.zeros((rows, cout), dtype=torch.int32, device="cuda")
            fn = getattr(A.lib(), "apconv_w%da%d" % (wb, xb))
            args = (W.data_ptr(), X.data_ptr(), out.data_ptr(), H, H, C, cout)
            s.update(fn=fn, args=args, out=out, keep=(W, X))
            return s
        X = _planes(gen, xb, batch * H * H * C // 32)
        epi, keep = A.Epilogue(), [W, X]
        if case["out"] == "int32":
            out = torch.zeros((rows, cout), dtype=torch.int32, device="cuda")
        else:
            epi.mode, epi.out_bits = A.EPI_BN, _out_bits(case)
            sigma, center = _sigma(R * R * C, wb, xb), 0.0
            if case["out"] == "bn_shortcut":  # packed codes of an earlier layer at half a standard deviation
                keep.append(_planes(gen, min(xb, 2), rows * cout // 32))
                epi.residual_planes, epi.residual_bits = keep[-1].data_ptr(), min(xb, 2)
                top = (1 << epi.residual_bits) - 1
                epi.residual_scale = max(1, int(round(sigma / (2.0 * top))))
                center = epi.residual_scale * top / 2.0
            elif case["out"] == "bn_pool":
                epi.pool = A.POOL_MAX2X2
            keep.append(_thresholds(gen, cout, epi.out_bits, sigma, center))
            epi.thresholds = keep[-1].data_ptr()
            out = torch.zeros((epi.out_bits, rows // (4 if epi.pool else 1), cout // 32), dtype=torch.int32, device="cuda")
        desc = A.ConvDesc(W=W.data_ptr(), X=X.data_ptr(), O=out.data_ptr(), batch=batch, H=H, Wd=H, cin_pad=C, COUT=cout,
                          R=R, S=R, stride=stride, pad=pad, halo=0, wb=wb, xb=xb, weight_mode=A.WEIGHT_SYMMETRIC,
                          epi=epi, path=A.PATH_AUTO)
        s.update(fn=A.lib().apnn_conv, desc=desc, ref=ctypes.byref(desc), out=out, keep=keep)
    elif case["kind"] == "net":
        net = _Net(_NETS[case["net"]], case["batch"], int(seed) + 1)
        images = torch.randint(0, 256, (case["batch"], 224, 224, 3), dtype=torch.uint8, device="cuda", generator=gen)
        out = torch.zeros((case["batch"], 1000), dtype=torch.float32, device="cuda")
        s.update(fn=A.nn_lib().apnn_net_forward, net=net, args=(net.handle, images.data_ptr(), out.data_ptr()), out=out,
                 keep=images)
    else:
        rows, C, bits = case["rows"], case["C"], case["bits"]
        cpad = -(-C // 32) * 32
        # activations of about the range the quantizer clips to
        x = 4.0 * torch.randn((rows, C), dtype=torch.float32, device="cuda", generator=gen)
        out = torch.zeros((bits, rows, cpad // 32), dtype=torch.int32, device="cuda")
        s.update(fn=A.lib().apnn_quantize_pack, args=(x.data_ptr(), out.data_ptr(), rows, C, cpad, bits, -10.0, 10.0),
                 out=out, keep=x)
    return s


def run(s):
    stream = torch.cuda.current_stream().cuda_stream
    if "ref" in s:
        rc = s["fn"](s["ref"], stream)
    else:
        rc = s["fn"](*s["args"], stream)
    if rc != 0:
        s["A"].check(rc, s["kind"])
    return s["out"]


def _net_layers(net):
    """(output height, input channels, output channels, filter) of every layer that holds weights, the layer's
    bits per weight, and whether its input is the image."""
    if net == "alexnet":
        convs = [(56, 3, 64, 11, 8), (28, 64, 192, 5, 1), (14, 192, 384, 3, 1), (14, 384, 256, 3, 1), (14, 256, 256, 3, 1)]
        return convs + [(1, 12544, 4096, 1, 1), (1, 4096, 4096, 1, 1), (1, 4096, 1000, 1, 8)]
    if net == "vgg":
        convs = [(112, 3, 96, 3, 8), (56, 96, 256, 3, 1)] + [(56, 256, 256, 3, 1)] * 2 + [(28, 256, 512, 3, 1)]
        convs += [(28, 512, 512, 3, 1)] * 2 + [(14, 512, 512, 3, 1)] * 3
        return convs + [(1, 25088, 4096, 1, 1), (1, 4096, 4096, 1, 1), (1, 4096, 1000, 1, 8)]
    layers = [(112, 3, 64, 7, 8)] + [(56, 64, 64, 3, 1)] * 4
    for i, ch in enumerate((128, 256, 512)):
        h = 28 >> i
        layers += [(h, ch // 2, ch, 3, 1), (h, ch // 2, ch, 1, 1)] + [(h, ch, ch, 3, 1)] * 3
    return layers + [(1, 512, 1000, 1, 8)]


def work(case):
    if case["kind"] == "gemm":
        M, N, K, wb, xb = (case[k] for k in ("M", "N", "K", "wb", "xb"))
        out = 4 * M * N if case["out"] == "int32" else _out_bits(case) * M * N // 8
        return {"bytes": (wb * M * K + xb * N * K) // 8 + out, "flops": 2 * M * N * K}
    if case["kind"] == "conv":
        batch, H, C, cout, R, wb, xb = (case[k] for k in ("batch", "H", "C", "cout", "R", "wb", "xb"))
        pad = (R - 1) // 2
        Ho = (H + 2 * pad - R) // case["stride"] + 1
        rows = batch * Ho * Ho
        if case["out"] == "int32":
            out = 4 * rows * cout
        else:
            out = _out_bits(case) * rows * cout // (32 if case["out"] == "bn_pool" else 8)
            out += 4 * cout * ((1 << _out_bits(case)) - 1)
            out += min(xb, 2) * rows * cout // 8 if case["out"] == "bn_shortcut" else 0
        return {"bytes": xb * batch * H * H * C // 8 + wb * cout * R * R * C // 8 + out, "flops": 2 * rows * cout * R * R * C}
    if case["kind"] == "net":
        # images, weights and logits; the activations between layers need not leave the chip
        layers, batch = _net_layers(case["net"]), case["batch"]
        weights = sum(cin * cout * r * r * bits for _, cin, cout, r, bits in layers) // 8
        ops = sum(2 * h * h * cin * cout * r * r for h, cin, cout, r, _ in layers)
        return {"bytes": batch * (224 * 224 * 3 + 4000) + weights, "flops": batch * ops}
    cpad = -(-case["C"] // 32) * 32
    return {"bytes": 4 * case["rows"] * case["C"] + case["bits"] * case["rows"] * cpad // 8, "flops": 0}


def tolerance(case):
    # Integer sums, codes and packed words are exact at every precision.  A network's logits are one fp32
    # multiply and add of an exact integer: another order of the two roundings moves them by 3e-8 (measured
    # against the same affine map in 64 bits: 3e-8 relative).
    return {"rel": 2e-7} if case["kind"] == "net" else "exact"
