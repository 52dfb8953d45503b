"""The work a user has this library do, as timed cases: single core convolutions, Tucker operators and whole Tucker
networks, fp32 NCHW inference, from one latency-bound launch to batches that fill the device.

Sizes are those of the benchmark sweep (3x3 cores, H = W in {7, 14, 28, 56}, ranks 16 to 128), of the four Tucker blocks
and the two networks the library builds (Tucker ResNet-18, Tucker DenseNet-121), of the reference's 224x224 core layer,
and serving batches and ragged shapes of the same ranges.  Everything runs with the library's default settings.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "ppopp23-tdc_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tdc_amd import Conv2dPlan, TKConv2dC, TKConvOp, nets, ranks_dict  # noqa: E402

SWEEP_H = (7, 14, 28, 56)
SWEEP_RANKS = ((16, 16), (32, 32), (64, 64), (96, 96), (128, 128), (32, 64), (64, 128))


def _conv(name, batch, C, N, H, W, stride=1, bias=False, relu=False, residual=False):
    c = {"kind": "conv", "batch": batch, "C": C, "N": N, "H": H, "W": W, "stride": stride, "bias": bias, "relu": relu,
         "residual": residual}
    return {"name": name, **c} if name else c


def _tkconv(name, batch, C, R1, R2, N, H, W, stride=1, module=False, bias=False, relu=False, residual=False):
    c = {"kind": "tkconv", "batch": batch, "C": C, "R1": R1, "R2": R2, "N": N, "H": H, "W": W, "stride": stride,
         "module": module, "bias": bias, "relu": relu, "residual": residual}
    return {"name": name, **c} if name else c


def _net(name, net, batch, H=224, W=224):
    c = {"kind": "net", "net": net, "batch": batch, "H": H, "W": W}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One small core convolution for one image: nothing but launch and latency.
        _conv("conv_32x32_7_b1", 1, 32, 32, 7, 7),
        # The benchmark's pass: all 28 core shapes of the sweep, one image, one launch each.
        {"name": "core_sweep_b1", "kind": "sweep"},
        # A large single image: the 224x224 core layer the reference times.
        _conv("conv_64x32_224_b1", 1, 64, 32, 224, 224),
        # A core of no round size for a handful of images, with the whole epilogue (bias, residual, ReLU).
        _conv("conv_60x84_35_b5_ragged", 5, 60, 84, 35, 35, bias=True, relu=True, residual=True),
        # The sweep's largest core for a full serving batch: the largest single launch.
        _conv("conv_128x128_56_b64", 64, 128, 128, 56, 56),
        # A Tucker block through the drop-in module, one image: a layer swapped into an existing model.
        _tkconv("tkconv_256_64_56_b1", 1, 256, 64, 64, 256, 56, 56, module=True, bias=True),
        # The same kind of block for a batch: the first and last factors carry most of the traffic.
        _tkconv("tkconv_512_128_28_b32", 32, 512, 128, 128, 512, 28, 28, bias=True, relu=True, residual=True),
        # The deepest block, 7x7 pixels and 2048 channels, for a large batch.
        _tkconv("tkconv_2048_256_7_b64", 64, 2048, 256, 256, 2048, 7, 7),
        # Whole networks: one image (latency) and batches (throughput).
        _net("resnet18_b1", "resnet18", 1),
        _net("resnet18_b32", "resnet18", 32),
        _net("densenet121_b1", "densenet121", 1),
        _net("densenet121_b8", "densenet121", 8),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


_MAX_FLOPS = 55e9     # below the largest listed case (conv_128x128_56_b64: 59 GFLOP, 206 MB)
_MAX_BYTES = 200e6


def draw(rng):
    kind = rng.choice(("conv", "conv", "conv", "tkconv", "tkconv", "net"))
    if kind == "net":
        net = rng.choice(("resnet18", "densenet121"))
        batch = _log(rng, 1, 32 if net == "resnet18" else 8)
        H, W = _log(rng, 96, 224), _log(rng, 96, 224)
        if rng.random() < 0.5:          # crops in whole steps of 32 are the ordinary ones
            H = W = (H + 31) // 32 * 32
        return _net(None, net, batch, H, W)
    while True:
        stride = rng.choice((1, 1, 1, 2))
        bias, relu, residual = rng.choice(((0, 0, 0), (0, 0, 0), (1, 0, 0), (1, 1, 0), (1, 1, 1)))
        flags = {"bias": bool(bias), "relu": bool(relu), "residual": bool(residual)}
        batch = _log(rng, 1, 64)
        if kind == "conv":
            c = _conv(None, batch, _log(rng, 16, 256), _log(rng, 16, 256), _log(rng, 7, 112), _log(rng, 7, 112), stride, **flags)
            if rng.random() < 0.5:      # channel counts in whole steps of 16 and square images are the ordinary ones
                c.update(C=(c["C"] + 15) // 16 * 16, N=(c["N"] + 15) // 16 * 16, W=c["H"])
        else:
            r1, r2 = _log(rng, 16, 256), _log(rng, 16, 256)
            c = _tkconv(None, batch, _log(rng, r1, 2048), r1, r2, _log(rng, r2, 2048), _log(rng, 7, 56), _log(rng, 7, 56), stride,
                        module=rng.random() < 0.5, **flags)
            if rng.random() < 0.5:
                c.update({k: (c[k] + 15) // 16 * 16 for k in ("C", "R1", "R2", "N")}, W=c["H"])
            if c["module"]:             # (the module has no ReLU and no residual)
                c.update(relu=False, residual=False)
        w = work(c)
        if w["flops"] <= _MAX_FLOPS and w["bytes"] <= _MAX_BYTES:
            return c


def _out(n, stride):
    return (n - 1) // stride + 1     # 3x3, pad 1


def _conv_work(batch, C, N, H, W, K, stride, pad):
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    return {"bytes": 4.0 * (batch * (C * H * W + N * Ho * Wo) + K * K * C * N), "flops": 2.0 * batch * Ho * Wo * C * N * K * K}


def _half(n):
    return (n - 1) // 2 + 1     # stride 2: 3x3 / pad 1, 7x7 / pad 3 and 1x1 / pad 0 alike


def _resnet18_convs(H, W):
    """(C, N, K, output pixels) of every convolution of the Tucker ResNet-18 (ranks = half the width)."""
    h, w = _half(H), _half(W)
    out, cin = [(3, 64, 7, h * w)], 64
    h, w = _half(h), _half(w)
    for planes, stride in nets.RESNET18_STAGES:
        r = planes // 2
        for b in range(2):
            before = h * w
            if b == 0 and stride == 2:
                h, w = _half(h), _half(w)
                out.append((cin, planes, 1, h * w))
            out += [(cin, r, 1, before), (r, r, 3, h * w), (r, planes, 1, h * w)]
            out += [(planes, r, 1, h * w), (r, r, 3, h * w), (r, planes, 1, h * w)]
            cin = planes
    return out + [(512, 1000, 1, 1)]


def _densenet121_convs(H, W):
    h, w = _half(H), _half(W)
    out, c = [(3, 64, 7, h * w)], 64
    h, w = _half(h), _half(w)
    for b, layers in enumerate(nets.DENSENET121_BLOCKS):
        for _ in range(layers):
            out += [(c, 128, 1, h * w), (128, 64, 1, h * w), (64, 16, 3, h * w), (16, 32, 1, h * w)]
            c += 32
        if b < 3:
            out.append((c, c // 2, 1, h * w))
            c, h, w = c // 2, h // 2, w // 2
    return out + [(c, 1000, 1, 1)]


def work(case):
    b = case.get("batch", 1)
    if case["kind"] == "sweep":
        ws = [_conv_work(1, r1, r2, h, h, 3, 1, 1) for h in SWEEP_H for r1, r2 in SWEEP_RANKS]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    if case["kind"] == "conv":
        w = _conv_work(b, case["C"], case["N"], case["H"], case["W"], 3, case["stride"], 1)
        if case["residual"]:
            w["bytes"] += 4.0 * b * case["N"] * _out(case["H"], case["stride"]) * _out(case["W"], case["stride"])
        return w
    if case["kind"] == "tkconv":
        # the intermediates of ranks R1 and R2 need never reach memory
        C, R1, R2, N, H, W, s = (case[k] for k in ("C", "R1", "R2", "N", "H", "W", "stride"))
        po = _out(H, s) * _out(W, s)
        return {"bytes": 4.0 * (b * (C * H * W + N * po * (2 if case["residual"] else 1)) + C * R1 + 9 * R1 * R2 + R2 * N),
                "flops": 2.0 * b * (C * R1 * H * W + 9 * R1 * R2 * po + R2 * N * po)}
    H, W = case["H"], case["W"]
    convs = _resnet18_convs(H, W) if case["net"] == "resnet18" else _densenet121_convs(H, W)
    return {"bytes": 4.0 * (b * (3 * H * W + 1000) + sum(C * N * K * K for C, N, K, _ in convs)),
            "flops": sum(2.0 * b * p * C * N * K * K for C, N, K, p in convs)}


def tolerance(case):
    # Against the same layers in 64 bits: one convolution 1.0e-7 to 3.5e-7 (largest difference 2.6e-6 of the rms: Winograd
    # at batch 64), fp32 on a CPU 1.7e-7 to 2.4e-7; through three of them or a network up to 7.3e-7 (3.4e-6: the sums of
    # 2048 and 2304 products of the 7x7 block).  About four times that:
    if case["kind"] in ("conv", "sweep"):
        return {"rel": 1.5e-6, "max": 1.2e-5}
    return {"rel": 3e-6, "max": 1.5e-5}


def _gen(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed))


def _uniform(g, *shape):
    """Activations ~ U[-1, 1] on the device."""
    return torch.empty(*shape, device="cuda").uniform_(-1.0, 1.0, generator=g)


def _kaiming(g, n, c, k):
    return torch.empty(n, c, k, k).normal_(0.0, math.sqrt(2.0 / (c * k * k)), generator=g)


def _orthonormal(g, rows, cols):
    """A rows x cols matrix with orthonormal columns (rows >= cols), or orthonormal rows."""
    q, _ = torch.linalg.qr(torch.randn(max(rows, cols), min(rows, cols), generator=g))
    return (q if rows >= cols else q.t()).contiguous()


def _make_conv(case, gc, gd):
    b, C, N, H, W, s = (case[k] for k in ("batch", "C", "N", "H", "W", "stride"))
    plan = Conv2dPlan(b, C, N, H, W, 3, 3, stride=s, pad=1, bias=case["bias"], relu=case["relu"])
    plan.set_weights(_kaiming(gc, N, C, 3), torch.randn(N, generator=gc) * 0.1 if case["bias"] else None)
    x = _uniform(gd, b, C, H, W)
    res = _uniform(gd, b, N, _out(H, s), _out(W, s)) if case["residual"] else None
    return plan, x, res


def _make_tkconv(case, gc, gd):
    b, C, R1, R2, N, H, W, s = (case[k] for k in ("batch", "C", "R1", "R2", "N", "H", "W", "stride"))
    # orthonormal factors and a Gaussian core, as a Tucker decomposition of a trained layer leaves them
    first = _orthonormal(gc, C, R1).t().contiguous().reshape(R1, C, 1, 1)
    core = torch.empty(R2, R1, 3, 3).normal_(0.0, 0.02, generator=gc)
    last = _orthonormal(gc, N, R2).reshape(N, R2, 1, 1)
    bias = torch.randn(N, generator=gc) * 0.1 if case["bias"] else None
    x = _uniform(gd, b, C, H, W)
    res = _uniform(gd, b, N, _out(H, s), _out(W, s)) if case["residual"] else None
    if case["module"]:
        op = TKConv2dC(C, N, 3, stride=s, padding=1, bias=case["bias"], hp_dict=ranks_dict(layer=[R2, R1]), name="layer")
        op.load_kernels(first, core, last, bias)
        op(x)      # a module builds its operator for a shape on the first call: a program's warm-up
        return op, x, None
    op = TKConvOp(b, C, R1, R2, N, H, W, 3, stride=s, pad=1, bias=case["bias"], relu=case["relu"])
    op.set_weights(first, core, last, bias)
    return op, x, res


def prepare(case, seed):
    gc, gd = _gen(seed, "cpu"), _gen(seed, "cuda")
    kind = case["kind"]
    if kind == "sweep":
        layers = [_conv(None, 1, r1, r2, h, h) for h in SWEEP_H for r1, r2 in SWEEP_RANKS]
        return {"calls": [_make_conv(c, gc, gd) for c in layers]}
    if kind == "conv":
        return {"calls": [_make_conv(case, gc, gd)]}
    if kind == "tkconv":
        op, x, res = _make_tkconv(case, gc, gd)
        return {"module": op, "x": x} if case["module"] else {"calls": [(op, x, res)]}
    b, H, W = case["batch"], case["H"], case["W"]
    if case["net"] == "resnet18":
        net = nets.build_tucker_resnet18(nets.resnet18_params(seed=int(seed)), batch=b, H=H, W=W)
    else:
        net = nets.build_tucker_densenet121(nets.densenet121_params(seed=int(seed)), batch=b, H=H, W=W)
    return {"module": net, "x": torch.empty(b, 3, H, W, device="cuda").normal_(generator=gd)}


def run(state):
    if "module" in state:
        return state["module"](state["x"])
    return [op.forward(x, res) for op, x, res in state["calls"]]
