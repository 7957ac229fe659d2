"""The workloads by which this framework's speed is followed, each one pass through its public entry points.

`listed()` names the workloads, `draw()` gives more of the same ranges; `prepare()` makes what a user's program holds
before the call, `run()` is one pass, `work()` what that pass cannot do without and `tolerance()` how far another
correct implementation of the same precision may be off.

A case is a dict of plain values.  `kind` says what is called:

  conv2d   a WTConv2d layer (`wtconv.WTConv2d`, or its fast twin's class)            B, C, H, W, K, L
  conv1d   a WTConv1d layer                                                         B, C, N, K, L
  haar2d   one level of the Haar transform and back (`wtconv.util.wavelet`)         B, C, H, W
  block    a WTConvNeXt block, the layer with LayerNorm, MLP and shortcut around it B, C, H, W, K, L
  model    WTConvNeXt-T, images to logits                                           B, H, W

`mode` is "infer" (forward, nothing recorded) or "train" (forward, then backward from a given upstream gradient, with
the gradients of the input and of every parameter).  `dtype` is that of the activations, `params` that of the
parameters (float32 parameters under 16-bit activations are what torch.autocast leaves a layer with).
"""
import math

import torch

from fast_wtconv.wtconv_cuda import WTConv2d as FastWTConv2d
from wtconv import WTConv2d
from wtconv.util import wavelet
from wtconv.wtconv1d import WTConv1d
from wtconvnext import wtconvnext

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
SIZE = {"float32": 4, "bfloat16": 2, "float16": 2}


def listed():
    return [
        # one small feature map through one layer, as in a forward pass over a handful of images: a call is over in
        # microseconds, so launches and host time count
        {"name": "conv2d infer small f32", "kind": "conv2d", "mode": "infer", "B": 8, "C": 32, "H": 64, "W": 64,
         "K": 5, "L": 3, "dtype": "float32", "params": "float32", "fast": False},
        # the first-stage layer of WTConvNeXt-T on 224 x 224 images in a training step, full precision
        {"name": "conv2d train 56x56 f32", "kind": "conv2d", "mode": "train", "B": 128, "C": 96, "H": 56, "W": 56,
         "K": 5, "L": 3, "dtype": "float32", "params": "float32", "fast": False},
        # the same layer with model and activations in bfloat16
        {"name": "conv2d train 56x56 bf16", "kind": "conv2d", "mode": "train", "B": 128, "C": 96, "H": 56, "W": 56,
         "K": 5, "L": 3, "dtype": "bfloat16", "params": "bfloat16", "fast": False},
        # the last stage: many channels of tiny planes with odd extents
        {"name": "conv2d train 7x7 bf16", "kind": "conv2d", "mode": "train", "B": 128, "C": 768, "H": 7, "W": 7,
         "K": 5, "L": 2, "dtype": "bfloat16", "params": "bfloat16", "fast": False},
        # the first stage of a segmentation network on 640 x 640 crops: planes too large for on-chip memory
        {"name": "conv2d train 160x160 f32", "kind": "conv2d", "mode": "train", "B": 8, "C": 96, "H": 160, "W": 160,
         "K": 5, "L": 3, "dtype": "float32", "params": "float32", "fast": False},
        # ragged maps under float16 autocast with a 7 x 7 kernel, through the fast twin's class
        {"name": "conv2d train 45x37 f16 k7", "kind": "conv2d", "mode": "train", "B": 16, "C": 72, "H": 45, "W": 37,
         "K": 7, "L": 2, "dtype": "float16", "params": "float32", "fast": True},
        # a sequence model's layer: long power-of-two rows, full precision
        {"name": "conv1d train 4096 f32", "kind": "conv1d", "mode": "train", "B": 64, "C": 64, "N": 4096, "K": 5,
         "L": 4, "dtype": "float32", "params": "float32"},
        # a recording of odd length under bfloat16 autocast, five levels
        {"name": "conv1d train 20011 bf16", "kind": "conv1d", "mode": "train", "B": 8, "C": 48, "N": 20011, "K": 7,
         "L": 5, "dtype": "bfloat16", "params": "float32"},
        # the transform by itself, forth and back, as used to build other layers from it
        {"name": "haar2d infer 128x128 f32", "kind": "haar2d", "mode": "infer", "B": 16, "C": 64, "H": 128, "W": 128,
         "dtype": "float32", "params": "float32"},
        # the commonest block of WTConvNeXt-T (half of its blocks are of the third stage) in a training step
        {"name": "block train 14x14 bf16", "kind": "block", "mode": "train", "B": 64, "C": 384, "H": 14, "W": 14,
         "K": 5, "L": 3, "dtype": "bfloat16", "params": "bfloat16"},
        # a single image through the whole model: latency
        {"name": "model infer 1 bf16", "kind": "model", "mode": "infer", "B": 1, "H": 224, "W": 224,
         "dtype": "bfloat16", "params": "bfloat16"},
        # a validation batch through the whole model: throughput
        {"name": "model infer 256 bf16", "kind": "model", "mode": "infer", "B": 256, "H": 224, "W": 224,
         "dtype": "bfloat16", "params": "bfloat16"},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batch(rng, per_item, least, most, cap=256):
    """A batch whose elements, per_item each, come to between `least` and `most` in all (at least one item)."""
    return max(1, min(cap, _log(rng, least, most) // per_item))


def draw(rng):
    kind = rng.choice(["conv2d"] * 6 + ["conv1d"] * 3 + ["haar2d", "block", "model"])
    mode = "train" if rng.random() < 0.7 else "infer"
    dtype, params = rng.choice([("float32", "float32")] * 3 + [("bfloat16", "bfloat16")] * 2
                               + [("bfloat16", "float32"), ("float16", "float32")])
    if kind == "model":
        return {"kind": kind, "mode": "infer", "B": _log(rng, 1, 200), "H": rng.choice([160, 192, 224]),
                "W": rng.choice([160, 192, 224]), "dtype": "bfloat16", "params": "bfloat16"}
    if kind == "block":
        side, c, lv = rng.choice([(56, 96, 5), (28, 192, 4), (14, 384, 3), (7, 768, 2)])
        h, w = max(4, side + rng.randint(-3, 3)), max(4, side + rng.randint(-3, 3))
        return {"kind": kind, "mode": mode, "B": _batch(rng, c * h * w, 2 ** 18, 2 ** 23), "C": c, "H": h, "W": w,
                "K": 5, "L": lv, "dtype": "bfloat16", "params": "bfloat16"}
    if kind == "conv1d":
        n, c, k = _log(rng, 64, 40000), _log(rng, 8, 256), rng.choice([3, 5, 5, 7])
        return {"kind": kind, "mode": mode, "B": _batch(rng, c * n, 2 ** 17, 2 ** 24), "C": c, "N": n, "K": k,
                "L": rng.randint(1, min(5, int(math.log2(n)) - 2)), "dtype": dtype, "params": params}
    side, c = _log(rng, 6, 200), _log(rng, 16, 768)
    h, w = side, max(5, int(side * rng.uniform(0.75, 1.3)))
    if kind == "haar2d":
        h, w = h + h % 2, w + w % 2
        return {"kind": kind, "mode": mode, "B": _batch(rng, c * h * w, 2 ** 17, 2 ** 24), "C": c, "H": h, "W": w,
                "dtype": dtype, "params": "float32"}
    return {"kind": kind, "mode": mode, "B": _batch(rng, c * h * w, 2 ** 17, 2 ** 25), "C": c, "H": h, "W": w,
            "K": rng.choice([3, 5, 5, 5, 7]), "L": rng.randint(1, min(5, int(math.log2(min(h, w))))),
            "dtype": dtype, "params": params, "fast": rng.random() < 0.25}


def _build(case):
    """The module, with the framework's own initialisation."""
    kind = case["kind"]
    if kind == "model":
        return wtconvnext.wtconvnext_tiny()
    if kind == "block":
        return wtconvnext.WTConvNeXtBlock(case["C"], kernel_size=case["K"], wt_levels=case["L"])
    if kind == "conv1d":
        return WTConv1d(case["C"], case["C"], case["K"], wt_levels=case["L"])
    cls = FastWTConv2d if case["fast"] else WTConv2d
    return cls(case["C"], case["C"], kernel_size=case["K"], wt_levels=case["L"])


def _as_trained(module, gen):
    """Scales move away from their initial constants in training (a layer scale that starts at 1e-6 most of all)."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("gamma"):
                p.uniform_(0.05, 0.5, generator=gen)
            elif "scale" in name:
                p.mul_(torch.empty_like(p).uniform_(0.5, 1.5, generator=gen))
    return module


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    kind, train = case["kind"], case["mode"] == "train"
    shape = ((case["B"], case["C"], case["N"]) if kind == "conv1d" else
             (case["B"], 3 if kind == "model" else case["C"], case["H"], case["W"]))
    state = {"case": case, "x": torch.randn(shape, generator=gen, device=dev).to(dtype).requires_grad_(train),
             "grad": torch.randn(shape, generator=gen, device=dev).to(dtype) if train else None}
    if kind == "haar2d":
        dec, rec = wavelet.create_2d_wavelet_filter("db1", case["C"], case["C"])
        state["dec"], state["rec"] = dec.to(dev), rec.to(dev)
        return state
    torch.manual_seed(seed)
    with dev:
        module = _build(case)
    state["module"] = _as_trained(module, gen).to(DTYPES[case["params"]]).train(train)
    state["params"] = [p for p in module.parameters() if p.requires_grad]
    return state


def run(state):
    case, x = state["case"], state["x"]
    train = case["mode"] == "train"
    with torch.set_grad_enabled(train):
        if case["kind"] == "haar2d":
            x.grad = None
            bands = wavelet.wavelet_2d_transform(x, state["dec"])
            out = wavelet.inverse_2d_wavelet_transform(bands, state["rec"])
            if not train:
                return {"bands": bands, "out": out}
            out.backward(state["grad"])
            return {"bands": bands, "out": out, "grad": x.grad}
        if not train:
            return state["module"](x)
        x.grad = None
        for p in state["params"]:
            p.grad = None
        out = state["module"](x)
        out.backward(state["grad"])
        return {"out": out, "grad": x.grad, "param_grads": [p.grad for p in state["params"]]}


def _layer_work(case):
    """Elements, multiply-adds an element and parameters of one layer."""
    two_d = case["kind"] != "conv1d"
    taps = case["K"] ** 2 if two_d else case["K"]
    bands, levels = (4, case["L"]) if two_d else (2, case["L"])
    p = case["B"] * case["C"] * (case["H"] * case["W"] if two_d else case["N"])
    macs = taps * (1 + sum(bands * (1 / bands) ** lv for lv in range(1, levels + 1)))
    return p, macs, case["C"] * (taps + 2 + levels * bands * (taps + 1))


def work(case):
    """Activations and parameters read once and results written once; multiply-adds as two operations.  A training pass
    reads the input forward and again, with the upstream gradient, backward, and writes output, input gradient and
    parameter gradients; it multiplies three times as often as the forward pass."""
    train, s, sp = case["mode"] == "train", SIZE[case["dtype"]], SIZE[case["params"]]
    if case["kind"] == "model":
        # per stage: blocks, channels, wavelet levels, reduction of the extents
        flops, params = 0.0, 0
        pixels = case["B"] * case["H"] * case["W"]
        prev, prev_side = 3, 1
        for depth, c, levels, side in ((3, 96, 5, 4), (3, 192, 4, 8), (9, 384, 3, 16), (3, 768, 2, 32)):
            px = pixels / side ** 2
            patch = prev * c * (side // prev_side) ** 2
            taps = 25 * (1 + sum(4.0 ** (1 - lv) for lv in range(1, levels + 1)))
            flops += 2 * px * (patch + depth * (8 * c * c + taps * c))
            params += patch + depth * (8 * c * c + c * (36 + 104 * levels))
            prev, prev_side = c, side
        flops += 2 * case["B"] * 768 * 1000
        params += 768 * 1000
        return {"bytes": 3 * pixels * s + params * sp + case["B"] * 1000 * s, "flops": flops}
    if case["kind"] == "haar2d":
        p = case["B"] * case["C"] * case["H"] * case["W"]
        # forth and back: x read, coefficients written and read, result written; the same of the gradient in training
        # but for its coefficients, which nobody is given
        return {"bytes": (5 if train else 3) * p * s, "flops": (16 if train else 8) * p / 2}
    p, macs, count = _layer_work(case)
    if case["kind"] == "block":
        macs += 8 * case["C"]
        count += 8 * case["C"] ** 2 + 8 * case["C"]
    return {"bytes": (5 if train else 2) * p * s + (3 if train else 1) * count * sp,
            "flops": (6 if train else 2) * macs * p}


def tolerance(case):
    """float32: sums of up to hundreds of thousands of products.  float16: one rounding of each result to 11 bits
    (float32 within).  bfloat16: results, coefficients and folded weights of 8 bits.  The block and the model pass
    many such results on from one operation to the next."""
    if case["kind"] in ("block", "model"):
        return {"rel": 2e-2}
    if case["kind"] == "haar2d":
        return {"rel": {"float32": 1e-6, "float16": 1e-3, "bfloat16": 5e-3}[case["dtype"]]}
    return {"rel": {"float32": 1e-5, "float16": 1e-3, "bfloat16": 1e-2}[case["dtype"]]}
