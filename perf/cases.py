"""The work a user of borch_amd has it do, as measurable cases, each through the package's
public entry points on one GPU:

* ``linear``: one ``nn.Linear`` called eagerly, W8A8 (per-row dynamic activations) or weight-only
  W8A32 (f32 activations), with a bias: one layer of somebody's own model;
* ``chain``: decode steps, a stack of ``LinearReLU`` blocks on a few rows, in a HIP graph
  (``compiled(graph=True)``), W8A8 or W8A32;
* ``attention``: the f32 softmax attention between a transformer's int8 projections;
* ``encoder``: one ViT encoder layer (LayerNorm, qkv, attention, proj, MLP), called eagerly;
* ``conv``: one fused convolution block (bias, optional residual, ReLU) with dynamic scales;
* ``resnet18`` / ``efficientnet_b0``: a whole int8 forward in a HIP graph, with dynamic or
  calibrated scales, to the logits;
* ``stream``: host-resident int8 weights streamed through a bounded device window.

Sizes are those of the repository's workloads and tests (4096-wide Linears, ViT-B/16's layers,
CIFAR ResNet-18, EfficientNet-B0 at 224²) and, in ``draw``, the ranges around them, ragged ones
included. Kernels are chosen by the library's shape rules (``tune=False``), so that every
process runs the same ones."""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import borch_amd
from borch_amd import int8, nets, nn, streaming
from borch_amd.nn import intrinsic

# (expand ratio, kernel, stride, in, out, repeats): EfficientNet-B0's stages
_B0 = [(1, 3, 1, 32, 16, 1), (6, 3, 2, 16, 24, 2), (6, 5, 2, 24, 40, 2), (6, 3, 2, 40, 80, 3),
       (6, 5, 1, 80, 112, 3), (6, 5, 2, 112, 192, 4), (6, 3, 1, 192, 320, 1)]
# (in, out, stride): CIFAR ResNet-18's blocks
_R18 = [(64, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 1), (128, 256, 2), (256, 256, 1), (256, 512, 2),
        (512, 512, 1)]


def listed():
    return [
        # the smallest call: a 512-wide layer on 16 rows, where the launches and the host count
        {"name": "linear_16x512x512", "kind": "linear", "mode": "w8a8", "M": 16, "K": 512, "N": 512},
        # the large square product of the repository's benchmark
        {"name": "linear_4096", "kind": "linear", "mode": "w8a8", "M": 4096, "K": 4096, "N": 4096},
        # a layer of somebody's own sizes: nothing divides a tile or a 16-byte load
        {"name": "linear_ragged", "kind": "linear", "mode": "w8a8", "M": 1000, "K": 1555, "N": 2999},
        # a transformer MLP's first projection with weight-only quantization, 32 images of 197 tokens
        {"name": "w8a32_6304x768x3072", "kind": "linear", "mode": "w8a32", "M": 6304, "K": 768, "N": 3072},
        # weight-only prefill of a short prompt
        {"name": "w8a32_256x4096x4096", "kind": "linear", "mode": "w8a32", "M": 256, "K": 4096, "N": 4096},
        # single-row decode through eight 4096-wide layers
        {"name": "decode_w8a8_m1", "kind": "chain", "mode": "w8a8", "M": 1, "D": 4096, "blocks": 8},
        # batched decode with weight-only layers
        {"name": "decode_w8a32_m16", "kind": "chain", "mode": "w8a32", "M": 16, "D": 4096, "blocks": 8},
        # ViT-B/16's attention and its whole encoder layer, 32 images
        {"name": "attention_b32", "kind": "attention", "B": 32, "T": 197, "heads": 12},
        {"name": "vit_layer_b32", "kind": "encoder", "B": 32, "T": 197, "heads": 12},
        # whole forwards: CIFAR ResNet-18 with dynamic scales, EfficientNet-B0 with calibrated ones
        {"name": "resnet18_b16", "kind": "resnet18", "B": 16, "S": 32, "calibrated": False},
        {"name": "efficientnet_b0_b64", "kind": "efficientnet_b0", "B": 64, "S": 224, "calibrated": True},
        # a stack of 16 MiB int8 layers through a window that holds three of them
        {"name": "stream_int8_m16", "kind": "stream", "M": 16, "D": 4096, "blocks": 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "chain", "chain", "attention", "encoder", "conv", "conv",
                       "resnet18", "efficientnet_b0", "stream"])
    if kind == "linear":
        mode = rng.choice(["w8a8", "w8a32"])
        hi = 4096 if mode == "w8a8" else 3072
        K, N = _log(rng, 200, hi), _log(rng, 100, hi)
        if rng.random() < 0.6:  # most layers are multiples of 64 wide; the rest are anything
            K, N = max(64, K // 64 * 64), max(64, N // 64 * 64)
        return {"kind": kind, "mode": mode, "M": _log(rng, 1, 4096), "K": K, "N": N}
    if kind == "chain":
        D = rng.randint(1000, 4096)
        if rng.random() < 0.7:
            D = D // 128 * 128
        return {"kind": kind, "mode": rng.choice(["w8a8", "w8a32"]), "M": _log(rng, 1, 64), "D": D,
                "blocks": rng.randint(3, 8)}
    if kind == "attention":
        return {"kind": kind, "B": _log(rng, 1, 32), "T": rng.randint(16, 256), "heads": rng.randint(3, 12)}
    if kind == "encoder":
        return {"kind": kind, "B": _log(rng, 1, 32), "T": rng.randint(16, 256), "heads": rng.randint(6, 12)}
    if kind == "conv":
        k = rng.choice([1, 3, 3, 5])
        C, O = _log(rng, 16, 256), _log(rng, 16, 256)
        if rng.random() < 0.6:
            C, O = max(16, C // 16 * 16), max(16, O // 16 * 16)
        return {"kind": kind, "B": _log(rng, 1, 32), "C": C, "O": O, "H": rng.randint(7, 56), "W": rng.randint(7, 56),
                "k": k, "stride": rng.choice([1, 1, 2]), "residual": rng.random() < 0.5}
    if kind == "resnet18":
        return {"kind": kind, "B": _log(rng, 1, 64), "S": rng.randint(24, 40), "calibrated": rng.random() < 0.5}
    if kind == "efficientnet_b0":
        return {"kind": kind, "B": _log(rng, 2, 64), "S": rng.randint(96, 224), "calibrated": rng.random() < 0.5}
    return {"kind": "stream", "M": _log(rng, 1, 64), "D": rng.randint(1024 // 64, 4096 // 64) * 64,
            "blocks": rng.randint(3, 6)}


# ------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda") * std + mean


def _rand(g, *shape, lo=0.0, hi=1.0):
    return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo


def _linear_data(c, seed):
    """Activations N(0, 1), a Kaiming-normal weight, a small bias."""
    g = _gen(seed)
    return (_randn(g, c["M"], c["K"]), _randn(g, c["N"], c["K"], std=c["K"] ** -0.5), _randn(g, c["N"], std=0.1))


def _chain_data(c, seed):
    """Layers whose ReLU keeps the activations' scale (variance 2 / D)."""
    g, D = _gen(seed), c["D"]
    x = _randn(g, c["M"], D)
    return x, [(_randn(g, D, D, std=(2.0 / D) ** 0.5), _randn(g, D, std=0.1)) for _ in range(c["blocks"])]


def _attention_data(c, seed):
    return _randn(_gen(seed), c["B"], c["T"], 3 * 64 * c["heads"])


def _encoder_data(c, seed):
    g, D = _gen(seed), 64 * c["heads"]
    x = _randn(g, c["B"], c["T"], D)
    p = {}
    for name, o, i in (("qkv", 3 * D, D), ("proj", D, D), ("fc1", 4 * D, D), ("fc2", D, 4 * D)):
        p[name + ".weight"] = _rand(g, o, i, lo=-i ** -0.5, hi=i ** -0.5)
        p[name + ".bias"] = _rand(g, o, lo=-i ** -0.5, hi=i ** -0.5)
    for name in ("ln1", "ln2"):
        p[name + ".weight"] = _randn(g, D, std=0.1, mean=1.0)
        p[name + ".bias"] = _randn(g, D, std=0.1)
    return x, p


def _conv_out(c):
    pad = c["k"] // 2
    return [(n + 2 * pad - c["k"]) // c["stride"] + 1 for n in (c["H"], c["W"])]


def _conv_data(c, seed):
    g = _gen(seed)
    OH, OW = _conv_out(c)
    x = _randn(g, c["B"], c["C"], c["H"], c["W"]).contiguous(memory_format=torch.channels_last)
    w = _randn(g, c["O"], c["C"], c["k"], c["k"], std=(2.0 / (c["C"] * c["k"] ** 2)) ** 0.5)
    b = _randn(g, c["O"], std=0.1)
    r = (_randn(g, c["B"], c["O"], OH, OW).contiguous(memory_format=torch.channels_last) if c["residual"] else None)
    return x, w, b, r


def _put_conv(p, g, name, o, i, k):
    p[name + ".weight"] = _randn(g, o, i, k, k, std=math.sqrt(2.0 / (o * k * k) if i > 1 else 2.0 / (k * k)))


def _put_bn(p, g, name, n):
    p[name + ".running_mean"] = _randn(g, n, std=0.1)
    p[name + ".running_var"] = _rand(g, n, lo=0.5, hi=1.5)
    p[name + ".weight"] = _randn(g, n, std=0.1, mean=1.0)
    p[name + ".bias"] = _randn(g, n, std=0.1)


def _resnet_data(c, seed):
    """Normalised images and the network's parameters by their state-dict names."""
    g, p = _gen(seed), {}
    x, cal = _randn(g, c["B"], 3, c["S"], c["S"]), _randn(g, c["B"], 3, c["S"], c["S"])
    _put_conv(p, g, "stem", 64, 3, 3)
    _put_bn(p, g, "bn", 64)
    for i, (cin, cout, stride) in enumerate(_R18):
        b = f"body.{i}."
        _put_conv(p, g, b + "conv1", cout, cin, 3)
        _put_bn(p, g, b + "bn1", cout)
        _put_conv(p, g, b + "conv2", cout, cout, 3)
        _put_bn(p, g, b + "bn2", cout)
        if stride != 1 or cin != cout:
            _put_conv(p, g, b + "downConv", cout, cin, 1)
            _put_bn(p, g, b + "downBn", cout)
    p["fc.weight"] = _rand(g, 10, 512, lo=-512 ** -0.5, hi=512 ** -0.5)
    p["fc.bias"] = _rand(g, 10, lo=-512 ** -0.5, hi=512 ** -0.5)
    return x, cal, p


def _b0_blocks():
    """(state-dict prefix, in, out, kernel, stride, expand ratio) of every MBConv block."""
    n = 0
    for e, k, s, cin, cout, reps in _B0:
        for r in range(reps):
            yield f"blocks.{n}.", cin if r == 0 else cout, cout, k, s if r == 0 else 1, e
            n += 1


def _b0_data(c, seed):
    g, p = _gen(seed), {}
    x, cal = _rand(g, c["B"], 3, c["S"], c["S"]), _rand(g, c["B"], 3, c["S"], c["S"])
    _put_conv(p, g, "stem", 32, 3, 3)
    _put_bn(p, g, "bn", 32)
    for b, cin, cout, k, stride, e in _b0_blocks():
        mid, sq = cin * e, max(1, cin // 4)
        if e != 1:
            _put_conv(p, g, b + "expand", mid, cin, 1)
            _put_bn(p, g, b + "bn0", mid)
        _put_conv(p, g, b + "dw", mid, 1, k)
        _put_bn(p, g, b + "bn1", mid)
        for name, o, i in (("se_reduce", sq, mid), ("se_expand", mid, sq)):
            p[b + name + ".weight"] = _rand(g, o, i, 1, 1, lo=-i ** -0.5, hi=i ** -0.5)
            p[b + name + ".bias"] = _rand(g, o, lo=-i ** -0.5, hi=i ** -0.5)
        _put_conv(p, g, b + "project", cout, mid, 1)
        _put_bn(p, g, b + "bn2", cout)
    _put_conv(p, g, "head", 1280, 320, 1)
    _put_bn(p, g, "bn_head", 1280)
    p["fc.weight"] = _rand(g, 1000, 1280, lo=-1280 ** -0.5, hi=1280 ** -0.5)
    p["fc.bias"] = _rand(g, 1000, lo=-1280 ** -0.5, hi=1280 ** -0.5)
    return x, cal, p


# ---------------------------------------------------------------------- prepare and run

def _set(param, value):
    with torch.no_grad():
        param.copy_(value)


def _made_linear(w, b, mode):
    m = nn.Linear(w.shape[1], w.shape[0], device="cuda")
    _set(m.weight, w)
    _set(m.bias, b)
    return m.eval()


def _network(c, seed):
    """The network on its parameters, quantized (and calibrated on another batch), in a graph
    captured by one warm-up call, as a server does before its first request."""
    if c["kind"] == "resnet18":
        x, cal, p = _resnet_data(c, seed)
        model, split = nets.ResNet18(), 1
    else:
        x, cal, p = _b0_data(c, seed)
        # calibrated scales let the batch run as two chunks on parallel streams
        model, split = nets.EfficientNetB0(), 2 if c["calibrated"] else 1
    model = model.cuda().eval()
    model.load_state_dict(p, strict=False)
    net = borch_amd.compiled(model, int8=True, graph=True, tune=False, split=split, plan_cache=False)
    if c["calibrated"]:
        nn.calibrate_int8(model, [cal])
    net(cal)
    return {"net": net, "x": x}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b = _linear_data(case, seed)
        m = _made_linear(w, b, case["mode"])
        m.quantize_int8(weight_only=case["mode"] == "w8a32")
        return {"net": m, "x": x}
    if kind == "chain":
        x, layers = _chain_data(case, seed)
        m = torch.nn.Sequential(*[intrinsic.LinearReLU(_made_linear(w, b, case["mode"])) for w, b in layers]).eval()
        nn.quantize_for_int8(m, weight_only=case["mode"] == "w8a32")
        net = borch_amd.compiled(m, graph=True, tune=False, plan_cache=False)
        net(torch.zeros_like(x))  # the warm-up call captures the graph
        return {"net": net, "x": x}
    if kind == "attention":
        return {"x": _attention_data(case, seed)}
    if kind == "encoder":
        x, p = _encoder_data(case, seed)
        m = nets.EncoderLayer(64 * case["heads"], case["heads"], 256 * case["heads"]).cuda().eval()
        m.load_state_dict(p)
        m.fuse()
        nn.quantize_for_int8(m)
        return {"net": m, "x": x}
    if kind == "conv":
        x, w, b, r = _conv_data(case, seed)
        conv = nn.Conv2d(case["C"], case["O"], case["k"], case["stride"], case["k"] // 2, device="cuda")
        _set(conv.weight, w)
        _set(conv.bias, b)
        m = (intrinsic.ConvReLU2d if r is None else intrinsic.ConvAddReLU2d)(conv.eval())
        nn.quantize_for_int8(m)
        return {"net": m, "x": x, "residual": r}
    if kind == "stream":
        x, layers = _chain_data(case, seed)
        D = case["D"]

        def block(w, b):
            hw = streaming.pack_int8_host(w.cpu().numpy(), threads=8)
            return streaming.StreamBlock([hw], [(D, D)], lambda h, ws: torch.relu(F.linear(h, ws[0], b)))
        return {"blocks": [block(w, b) for w, b in layers], "x": x, "window": streaming.window(3 * D * D, "cuda")}
    return _network(case, seed)


def run(state):
    with torch.no_grad():
        if "blocks" in state:
            return streaming.stream_sequential(state["window"], state["x"], state["blocks"], int8=True)
        if "net" not in state:
            return int8.attention_f32(state["x"], state["x"].shape[2] // 192)
        if state.get("residual") is not None:
            return state["net"](state["x"], state["residual"])
        return state["net"](state["x"])


# ------------------------------------------------------------------- work and tolerance

def _conv_shapes(c):
    """(positions, outputs, products a position and output) of every convolution of a network,
    and the parameters' bytes (int8 weights, f32 head)."""
    shapes, S = [], c["S"]
    if c["kind"] == "resnet18":
        shapes.append((S * S, 64, 27))
        for cin, cout, stride in _R18:
            S = -(-S // stride)
            shapes += [(S * S, cout, 9 * cin), (S * S, cout, 9 * cout)]
            if stride != 1 or cin != cout:
                shapes.append((S * S, cout, cin))
        return shapes, 4 * 512 * 10
    S = -(-S // 2)
    shapes.append((S * S, 32, 27))
    extra = 4 * 1280 * 1000
    for _, cin, cout, k, stride, e in _b0_blocks():
        mid = cin * e
        if e != 1:
            shapes.append((S * S, mid, cin))
        S = -(-S // stride)
        shapes += [(S * S, mid, k * k), (S * S, cout, mid)]
        extra += 8 * mid * max(1, cin // 4)
    shapes.append((S * S, 1280, 320))
    return shapes, extra


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * M * K + N * K + 8 * N + 4 * M * N, "flops": 2 * M * N * K}
    if kind in ("chain", "stream"):
        M, D, n = c["M"], c["D"], c["blocks"]
        return {"bytes": n * (D * D + 8 * D) + 8 * M * D, "flops": 2 * n * M * D * D}
    if kind == "attention":
        B, T, H = c["B"], c["T"], c["heads"]
        return {"bytes": 4 * B * T * 64 * H * 4, "flops": 4 * B * H * T * T * 64}
    if kind == "encoder":
        B, T, D = c["B"], c["T"], 64 * c["heads"]
        return {"bytes": 8 * B * T * D + 12 * D * D, "flops": 24 * B * T * D * D + 4 * B * T * T * D}
    if kind == "conv":
        OH, OW = _conv_out(c)
        m = c["B"] * OH * OW
        return {"bytes": 4 * c["B"] * c["C"] * c["H"] * c["W"] + 4 * m * c["O"] * (2 if c["residual"] else 1)
                + c["O"] * c["C"] * c["k"] ** 2, "flops": 2 * m * c["O"] * c["C"] * c["k"] ** 2}
    shapes, extra = _conv_shapes(c)
    classes = 10 if kind == "resnet18" else 1000
    return {"bytes": 4 * c["B"] * (3 * c["S"] ** 2 + classes) + sum(o * k for _, o, k in shapes) + extra,
            "flops": 2 * c["B"] * sum(p * o * k for p, o, k in shapes)}


def tolerance(case):
    """About four times the largest relative error against ``exact`` that each kind showed."""
    kind = case["kind"]
    if kind == "linear" and case["mode"] == "w8a8" or kind == "conv":
        # exact integer sums, then one f32 rounding for each scale, the bias and the residual
        return {"rel": 5e-7}
    if kind in ("linear", "stream") or kind == "chain" and case["mode"] == "w8a32":
        return {"rel": 4e-6}  # sums of up to 4096 products in 32 bits
    if kind == "attention":
        return {"rel": 2e-6}
    # a last bit of an f32 input to a quantizer moves a value across a rounding boundary now and
    # then, and what follows by one of 127 steps of that value
    if kind == "chain":
        return {"rel": 5e-4}
    if kind == "encoder":
        return {"rel": 2e-3, "max": 0.1}
    return {"rel": 3e-2 if kind == "resnet18" else 2e-2}


# ------------------------------------------------------------------------ in 64 bits

def _scale(peak):
    return (peak.double() / 127.0).float().double()


def _q(v, s):
    """Whole values of v / s, half to even, within ±127 (0 where s is 0)."""
    return torch.where(s > 0, torch.round(v / s.clamp_min(1e-300)), torch.zeros_like(v)).clamp(-127, 127)


def _qrows(v):
    s = _scale(v.abs().amax(-1, keepdim=True))
    return _q(v, s), s


def _linear64(x, w, b, mode):
    qw, sw = _qrows(w.double())
    if mode == "w8a32":
        return x.double() @ (qw * sw).t() + b.double()
    qx, sx = _qrows(x.double())
    return (qx @ qw.t()) * sx * sw.t() + b.double()


def _conv64(x, w, stride, pad):
    """x [N, H, W, C] with w [O, C, k, k], or depthwise with w [C, 1, k, k]: a sum over taps."""
    k, out = w.shape[2], 0
    x = F.pad(x, (0, 0, pad, pad, pad, pad))
    OH, OW = ((n - k) // stride + 1 for n in x.shape[1:3])
    for i in range(k):
        for j in range(k):
            t = x[:, i:i + (OH - 1) * stride + 1:stride, j:j + (OW - 1) * stride + 1:stride]
            out = out + (t * w[:, 0, i, j] if w.shape[1] == 1 and x.shape[3] > 1 else t @ w[:, :, i, j].t())
    return out


class _Net64:
    """The convolutions of a network in 64 bits: as they are (recording the input maxima that
    calibration keeps) or with quantized inputs and weights."""

    def __init__(self, p):
        self.p, self.scales, self.mode = p, {}, "dynamic"

    def conv(self, x, name, bn, stride, pad):
        p = self.p
        g = p[bn + ".weight"] / torch.sqrt(p[bn + ".running_var"] + 1e-5)  # the fold, in the weights' own type
        w = (p[name + ".weight"] * g.reshape(-1, 1, 1, 1)).double()
        b = ((0 - p[bn + ".running_mean"]) * g + p[bn + ".bias"]).double()
        if self.mode == "float":
            self.scales[name] = _scale(x.abs().amax().float())
            return _conv64(x, w, stride, pad) + b
        s = self.scales[name] if self.mode == "calibrated" else _scale(x.abs().amax().float())
        qw, sw = _qrows(w.flatten(1))
        return _conv64(_q(x, s), qw.reshape(w.shape), stride, pad) * s * sw.flatten() + b

    def resnet18(self, x):
        h = torch.relu(self.conv(x, "stem", "bn", 1, 1))
        for i, (cin, cout, stride) in enumerate(_R18):
            b = f"body.{i}."
            side = self.conv(h, b + "downConv", b + "downBn", stride, 0) if b + "downBn.weight" in self.p else h
            h = torch.relu(self.conv(h, b + "conv1", b + "bn1", stride, 1))
            h = torch.relu(self.conv(h, b + "conv2", b + "bn2", 1, 1) + side)
        return self.head(h)

    def efficientnet_b0(self, x):
        p = self.p
        x = F.silu(self.conv(x, "stem", "bn", 2, 1))
        for b, cin, cout, k, stride, e in _b0_blocks():
            h = F.silu(self.conv(x, b + "expand", b + "bn0", 1, 0)) if e != 1 else x
            h = F.silu(self.conv(h, b + "dw", b + "bn1", stride, k // 2))
            w1, b1, w2, b2 = (p[b + n].double() for n in ("se_reduce.weight", "se_reduce.bias", "se_expand.weight",
                                                          "se_expand.bias"))
            z = F.silu(F.linear(h.mean(dim=(1, 2)), w1.flatten(1), b1))
            h = h * torch.sigmoid(F.linear(z, w2.flatten(1), b2))[:, None, None, :]
            y = self.conv(h, b + "project", b + "bn2", 1, 0)
            x = y + x if stride == 1 and cin == cout else y
        return self.head(F.silu(self.conv(x, "head", "bn_head", 1, 0)))

    def head(self, h):
        return F.linear(h.mean(dim=(1, 2)), self.p["fc.weight"].double(), self.p["fc.bias"].double())


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "linear":
            return _linear64(*_linear_data(case, seed), case["mode"])
        if kind in ("chain", "stream"):
            h, layers = _chain_data(case, seed)
            for w, b in layers:
                h = torch.relu(_linear64(h, w, b, case.get("mode", "w8a32")))
            return h
        if kind == "attention":
            return _attention64(_attention_data(case, seed).double(), case["heads"])
        if kind == "encoder":
            x, p = _encoder_data(case, seed)
            x, D = x.double(), x.shape[-1]

            def norm(v, n):
                return F.layer_norm(v, (D,), p[n + ".weight"].double(), p[n + ".bias"].double(), 1e-6)

            def lin(v, n):
                return _linear64(v, p[n + ".weight"], p[n + ".bias"], "w8a8")
            x = x + lin(_attention64(lin(norm(x, "ln1"), "qkv"), case["heads"]), "proj")
            return x + lin(F.gelu(lin(norm(x, "ln2"), "fc1")), "fc2")
        if kind == "conv":
            x, w, b, r = _conv_data(case, seed)
            x = x.double().permute(0, 2, 3, 1)
            s = _scale(x.abs().amax())
            qw, sw = _qrows(w.double().flatten(1))
            y = _conv64(_q(x, s), qw.reshape(w.shape), case["stride"], case["k"] // 2) * s * sw.flatten() + b.double()
            y = y.permute(0, 3, 1, 2)
            return torch.relu(y if r is None else y + r.double())
        x, cal, p = (_resnet_data if kind == "resnet18" else _b0_data)(case, seed)
        net = _Net64(p)
        if case["calibrated"]:
            net.mode = "float"
            getattr(net, kind)(cal.double().permute(0, 2, 3, 1))
            net.mode = "calibrated"
        return getattr(net, kind)(x.double().permute(0, 2, 3, 1))


def _attention64(qkv, heads):
    B, T, D3 = qkv.shape
    q, k, v = qkv.reshape(B, T, 3, heads, 64).permute(2, 0, 3, 1, 4).contiguous()
    a = torch.softmax((q @ k.transpose(-1, -2).contiguous()) / 8.0, -1)
    return (a @ v).transpose(1, 2).reshape(B, T, D3 // 3)
