"""The measured workloads of the framework: quantized linear layers in inference and training, and the
quantizer on its own, through the public entry points (``quantize_model`` / ``FourOverSixLinear``,
``quantize``, ``dequantize``).

A case is a dict of plain values with a ``kind``:

* ``linear``: forward pass of an ``nn.Linear`` that ``quantize_model`` converted and whose weight was quantized
  when the model was loaded; activations are quantized on the fly.  Fields: tokens, inf, outf, format, bias.
* ``train``: forward and backward pass of a converted layer that keeps its high-precision weight
  (quantized on each pass): output, gradients of input, weight and bias.  Fields: tokens, inf, outf, master
  (type of the weight).
* ``quantize``: one tensor to packed codes, block scales and tensor maximum, and with ``back`` also
  dequantized to its own type.  Fields: rows, cols, type, format, rule, style, block2d, back.
"""

import math

import torch
from torch import nn

import fouroversix_amd as fos

TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _linear(name, tokens, inf, outf, fmt="nvfp4", bias=False):
    return {"name": name, "kind": "linear", "tokens": tokens, "inf": inf, "outf": outf, "format": fmt, "bias": bias}


def _train(name, tokens, inf, outf, master="bf16"):
    return {"name": name, "kind": "train", "tokens": tokens, "inf": inf, "outf": outf, "master": master}


def _quantize(name, rows, cols, type_="bf16", fmt="nvfp4", rule="mse", style="nearest", block2d=False, back=False):
    return {"name": name, "kind": "quantize", "rows": rows, "cols": cols, "type": type_, "format": fmt, "rule": rule,
            "style": style, "block2d": block2d, "back": back}


def listed():
    return [
        # one sequence being decoded: the gate projection of a 4096 / 14336 MLP for a single token
        _linear("decode_1x4096x14336", 1, 4096, 14336),
        # a decode batch through an attention projection
        _linear("decode_16x4096x4096", 16, 4096, 4096),
        # a large decode batch (or a short prompt) through the MLP's down projection
        _linear("batch_128x14336x4096", 128, 14336, 4096),
        # a prompt of ragged length through a layer with a bias
        _linear("ragged_1000x4096x14336", 1000, 4096, 14336, bias=True),
        # one prompt of ordinary length, attention projection
        _linear("prefill_2048x4096x4096", 2048, 4096, 4096),
        # eight prompts of 2048 tokens at once through the MLP's gate projection
        _linear("prefill_16384x4096x14336", 16384, 4096, 14336),
        # the same layer kinds in the two other formats that have kernels
        _linear("mxfp4_2048x14336x4096", 2048, 14336, 4096, fmt="mxfp4"),
        _linear("if4_2048x4096x4096", 2048, 4096, 4096, fmt="if4"),
        # a training step of a key / value projection (one sequence) and of an attention projection (four sequences)
        # with fp32 master weights
        _train("train_2048x4096x1024", 2048, 4096, 1024),
        _train("train_8192x4096x4096", 8192, 4096, 4096, master="fp32"),
        # the quantizer alone on a large activation
        _quantize("quantize_8192x8192", 8192, 8192),
        # weights of an fp16 checkpoint whose sizes fit no tile: quantized in 16 x 16 blocks and read back
        _quantize("roundtrip_fp16_5000x3000", 5000, 3000, type_="fp16", block2d=True, back=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng):
    # layer widths are multiples of 128, now and then only of 16
    return 128 * _log_int(rng, 8, 112) if rng.random() < 0.8 else 16 * _log_int(rng, 64, 896)


def draw(rng):
    pick = rng.random()
    if pick < 0.55:
        fmt = rng.choice(["nvfp4", "nvfp4", "nvfp4", "nvfp4", "mxfp4", "if4"])
        inf, outf = _features(rng), _features(rng)
        # (IF4 is the format with the slowest product: shorter batches)
        most = min(16384, (16384 * 4096 * 14336 // (16 if fmt == "if4" else 1)) // (inf * outf))
        case = _linear("", _log_int(rng, 1, most), inf, outf, fmt, rng.random() < 0.3)
    elif pick < 0.75:
        inf, outf = _features(rng), _features(rng)
        most = min(16384, (8192 * 4096 * 4096) // (inf * outf))
        case = _train("", _log_int(rng, 128, most), inf, outf, rng.choice(["bf16", "fp32"]))
    else:
        rows = _log_int(rng, 16, 16384)
        cols = _log_int(rng, 256, 14336) if rng.random() < 0.3 else 16 * _log_int(rng, 16, 896)
        fmt = rng.choice(["nvfp4", "nvfp4", "nvfp4", "mxfp4", "if4"])
        case = _quantize(
            "", rows, cols, rng.choice(["bf16", "bf16", "fp16", "fp32"]), fmt,
            {"nvfp4": rng.choice(["mse", "mse", "static_6", "mae", "abs_max"]), "mxfp4": "static_6", "if4": "mse"}[fmt],
            rng.choice(["nearest", "nearest", "stochastic"]) if fmt == "nvfp4" else "nearest",
            fmt != "mxfp4" and rng.random() < 0.4, rng.random() < 0.4)
    del case["name"]
    return case


def _activation(g, rows, cols, dtype):
    # N(0, 1) with 1 % of the channels scaled by 50, as activations have them
    x = torch.randn(rows, cols, generator=g, device="cuda")
    x[:, torch.randperm(cols, generator=g, device="cuda")[: max(1, cols // 100)]] *= 50
    return x.to(dtype)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "quantize":
        config = fos.QuantizationConfig(dtype=case["format"], scale_rule=case["rule"], round_style=case["style"],
                                        block_scale_2d=case["block2d"], kwargs={"seed": seed})
        dtype = TYPES[case["type"]]
        if case["block2d"]:  # (weights)
            x = (0.02 * torch.randn(case["rows"], case["cols"], generator=g, device="cuda")).to(dtype)
        else:
            x = _activation(g, case["rows"], case["cols"], dtype)
        return {"case": case, "x": x, "config": config}

    train = case["kind"] == "train"
    layer = nn.Linear(case["inf"], case["outf"], bias=train or case["bias"], device="cuda",
                      dtype=TYPES[case["master"]] if train else torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(0.02 * torch.randn(case["outf"], case["inf"], generator=g, device="cuda"))
        if layer.bias is not None:
            layer.bias.copy_(torch.randn(case["outf"], generator=g, device="cuda"))
            if train:
                layer.bias = nn.Parameter(layer.bias.to(torch.bfloat16))
    model = nn.Sequential(layer)
    x = _activation(g, case["tokens"], case["inf"], torch.bfloat16)
    if train:
        fos.quantize_model(model, fos.ModelQuantizationConfig(keep_master_weights=True, weight_scale_2d=True))
        grad = (0.001 * torch.randn(case["tokens"], case["outf"], generator=g, device="cuda")).bfloat16()
        return {"case": case, "model": model, "x": x.requires_grad_(), "grad": grad, "seed": seed}
    if case["format"] == "mxfp4":  # (one rule, 1 x 32 blocks)
        config = fos.ModelQuantizationConfig(dtype="mxfp4", scale_rule="static_6")
    else:
        config = fos.ModelQuantizationConfig(dtype=case["format"], weight_scale_2d=True)
    fos.quantize_model(model, config)
    model[0].quantize_weight_()
    return {"case": case, "model": model, "x": x}


def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        with torch.no_grad():
            return state["model"](state["x"])
    if kind == "train":
        # the gradients' stochastic rounding draws its key from torch's CPU generator: set, so that the step can be repeated
        torch.default_generator.manual_seed(state["seed"])
        layer = state["model"][0]
        out = state["model"](state["x"])
        return (out, *torch.autograd.grad(out, (state["x"], layer.weight, layer.bias), state["grad"]))
    q = fos.quantize(state["x"], state["config"])
    coded = (q.values, q.scale_factors.view(torch.uint8), q.amax)
    return (*coded, fos.dequantize(q, dtype=state["x"].dtype)) if state["case"]["back"] else coded


def work(case):
    if case["kind"] == "quantize":
        n, size = case["rows"] * case["cols"], TYPES[case["type"]].itemsize
        coded = 0.5 + (1 / 32 if case["format"] == "mxfp4" else 1 / 16)
        return {"bytes": n * (size + coded + (size if case["back"] else 0)), "flops": 0}
    m, k, n = case["tokens"], case["inf"], case["outf"]
    if case["kind"] == "train":
        # x, grad and the weight in; output and the three gradients out
        weight = TYPES[case["master"]].itemsize
        return {"bytes": 2 * (2 * m * k + 2 * m * n) + 2 * weight * k * n + 2 * 2 * n, "flops": 3 * 2 * m * n * k}
    coded = 0.5 + (1 / 32 if case["format"] == "mxfp4" else 1 / 16)
    return {"bytes": 2 * m * k + coded * k * n + 2 * m * n + (2 * n if case["bias"] else 0), "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # fp32 sums in another order, rounded to bf16: now and then a value falls on the other side of a rounding boundary
    # (one step of bf16 is up to 2^-7 of the value).  Against the fp64 product of the same operands rounded to bf16:
    # up to 1.2e-5 for NVFP4 and MXFP4 and 6.3e-5 for IF4, 7.8e-3 at most for one value
    return {"rel": 2.5e-4, "max": 0.032}
