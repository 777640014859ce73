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


def _tensors(case, seed):
    """Weight, bias, input and output gradient of a layer."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    train = case["kind"] == "train"
    weight = (0.02 * torch.randn(case["outf"], case["inf"], generator=g, device="cuda")).to(
        TYPES[case["master"]] if train else torch.bfloat16)
    bias = torch.randn(case["outf"], generator=g, device="cuda").bfloat16() if train or case["bias"] else None
    x = _activation(g, case["tokens"], case["inf"], torch.bfloat16)
    grad = (0.001 * torch.randn(case["tokens"], case["outf"], generator=g, device="cuda")).bfloat16() if train else None
    return weight, bias, x, grad


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
    weight, bias, x, grad = _tensors(case, seed)
    with torch.no_grad():
        layer.weight.copy_(weight)
        if layer.bias is not None:
            layer.bias = nn.Parameter(bias, requires_grad=train)
    model = nn.Sequential(layer)
    if train:
        fos.quantize_model(model, fos.ModelQuantizationConfig(keep_master_weights=True, weight_scale_2d=True))
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


def _e2m1(v):
    # round to nearest, ties to even, on 0, 0.5, 1, 1.5, 2, 3, 4, 6
    a = v.abs()
    r = torch.where(a < 2, (a + a).round() / 2, torch.where(a < 4, a.round(), 2 * (a / 2).round()))
    return r * v.sign()


def _decoded(x, fmt, block2d):
    """x quantized (the adaptive rule by squared error where the format has one) and read back, in plain torch.

    Scales, codes and decisions follow the formats' fp32 arithmetic; what the codes stand for comes back in 64 bits.
    """
    rows, cols = x.shape
    step = 32 if fmt == "mxfp4" else 16
    tall = 16 if block2d else 1
    x = nn.functional.pad(x.float(), (0, -cols % step, 0, -rows % tall))
    amax = x.abs().max()
    # (tensors: torch divides by a plain number on the GPU as a product with its reciprocal)
    six, seven_sixths = (torch.tensor(v, device=x.device) for v in (6.0, 7 / 6))
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for top in range(0, x.shape[0], 2048):
        part = x[top : top + 2048]
        blocks = part.reshape(-1, tall, part.shape[1] // step, step)
        bmax = blocks.abs().amax((1, 3), keepdim=True)
        if fmt == "mxfp4":  # smallest power of two that takes the block's maximum to at most 6
            mantissa, exponent = torch.frexp(bmax / six)
            exponent = torch.where(mantissa == 0.5, exponent - 1, exponent)
            scale = torch.where(bmax > 0, torch.ldexp(torch.ones_like(bmax), exponent), 0)
            read = _e2m1(torch.where(scale > 0, blocks / scale, 0)).double() * scale.double()
        else:
            whole = six * (448.0 if fmt == "if4" else 256.0)
            enc, dec = whole / amax, amax / whole

            def scaled(expand):
                s = ((bmax / six) * enc * expand).to(torch.float8_e4m3fn).float()
                return s, torch.where(s > 0, blocks * (1 / (dec * s)), 0)

            def error(q, s, factor):
                e = ((q * s * amax) * factor / whole - blocks) ** 2
                # (added as the sum of a contiguous run is on the CPU: even and odd rows, halves, eight columns)
                even, odd = e[:, 0], e[:, 1] if tall > 1 else None
                for row in range(2, tall, 2):
                    even, odd = even + e[:, row], odd + e[:, row + 1]
                lanes = even[..., :8] + even[..., 8:]
                if tall > 1:
                    lanes = lanes + odd[..., :8] + odd[..., 8:]
                total = lanes[..., 0]
                for lane in range(1, 8):
                    total = total + lanes[..., lane]
                return total[:, None, :, None]

            s6, v6 = scaled(1.0)
            q6 = _e2m1(v6)
            if fmt == "if4":  # the other candidate: whole numbers to 7 on the same scale, in sevenths of 6
                qi = (v6 * seven_sixths).clamp(-7, 7).round()
                integer = error(qi, s6, 6 / 7) < error(q6, s6, 1.0)
                # (an integer block's values are defined as products in fp16)
                read = torch.where(integer, (qi * (6 / 7)).half() * s6.half(), q6.half() * s6.half())
            else:  # the other candidate: maximum at 4
                s4, v4 = scaled(1.5)
                q4 = _e2m1(v4)
                read = torch.where(error(q4, s4, 1.0) < error(q6, s6, 1.0), q4 * s4, q6 * s6)
            read = read.double() * amax.double() / whole.double()
        out[top : top + 2048] = read.reshape(part.shape)
    return out[:rows, :cols]


def exact(case, seed):
    if case["kind"] == "quantize":
        return None  # (whole numbers and bytes)
    weight, bias, x, grad = _tensors(case, seed)
    fmt = case.get("format", "nvfp4")
    out = _decoded(x, fmt, False) @ _decoded(weight, fmt, fmt != "mxfp4").T
    if bias is not None:
        out += bias.double()
    # (the gradients of input and weight are products of randomly rounded operands)
    return (out, None, None, grad.double().sum(0)) if case["kind"] == "train" else out
