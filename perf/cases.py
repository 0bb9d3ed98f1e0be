"""The work this framework is used for, as timed cases.

Every case goes through the operators a quantized model calls (`torch.quantize_per_tensor`,
`torch.ops.quantized.*`, `Tensor.dequantize`, ...) on the GPU, with weights packed beforehand, as a
program that serves such a model does.  A case is one of these kinds:

  mlp          float activations -> quantize -> linear_relu -> linear -> dequantize: the two linear
               layers of a feed-forward block, from one row (decode) to thousands (prefill)
  dynamic      quantized::linear_dynamic: float activations in and out, range found on the way
  plain        quantized::linear_per_tensor: the exported-graph form, plain int8 tensors
  codec        quantize and dequantize with given parameters, per tensor
  range_codec  the same with the parameters from the tensor's own range
  channels     quantize and dequantize per channel, what a weight goes through when a model is made
  residual     1x1 -> 3x3 -> 1x1 + residual convolutions on a feature map (ReLU or SiLU)
  inverted     1x1 -> depthwise 3x3 -> 1x1, with a residual where the shapes allow one
  stem         image -> quantize -> first convolution -> max pooling -> dequantize

A chain that ends in a quantized tensor is dequantized, as at the end of a quantized model.
"""
import math

import torch

import torch_musa_amd  # noqa: F401  (registers the operators)

_OPS = torch.ops.quantized
_DTYPES = {"quint8": torch.quint8, "qint8": torch.qint8}


def listed():
    return [
        # one row through a small layer pair: launches and host time are all there is
        {"name": "mlp_one_row", "kind": "mlp", "rows": 1, "k": 1024, "hidden": 1024, "n": 1024,
         "dtype": "quint8", "per_channel": True, "bias": True},
        # a decode step of a feed-forward block: four sequences, the weights are the traffic
        {"name": "mlp_decode", "kind": "mlp", "rows": 4, "k": 4096, "hidden": 11008, "n": 4096,
         "dtype": "quint8", "per_channel": True, "bias": True},
        # the same block on a prompt (prefill): bound by the matrix cores
        {"name": "mlp_prefill", "kind": "mlp", "rows": 4096, "k": 4096, "hidden": 11008, "n": 4096,
         "dtype": "quint8", "per_channel": True, "bias": True},
        # feature counts that follow no tile: 1000 classes or measurements, an odd hidden size
        {"name": "mlp_ragged", "kind": "mlp", "rows": 517, "k": 1000, "hidden": 2051, "n": 1000,
         "dtype": "qint8", "per_channel": False, "bias": True},
        # dynamically quantized decode of a small batch: range, codes and product per call
        {"name": "dynamic_decode", "kind": "dynamic", "rows": 16, "k": 4096, "n": 11008, "per_channel": True,
         "bias": True, "relu": False},
        # an encoder's layer in a graph exported with plain int8 tensors
        {"name": "plain_encoder", "kind": "plain", "rows": 384, "k": 768, "n": 3072, "dtype": "uint8", "out": "uint8",
         "post": "relu"},
        # a tensor of a gigabyte, quantized and restored
        {"name": "codec_large", "kind": "codec", "rows": 1 << 14, "cols": 1 << 14, "dtype": "quint8"},
        # activations of one layer quantized by their own range
        {"name": "range_codec_small", "kind": "range_codec", "rows": 128, "cols": 1024, "dtype": "quint8"},
        # a linear layer's weight, per output channel
        {"name": "channels_weight", "kind": "channels", "shape0": 11008, "shape1": 4096, "axis": 0, "dtype": "qint8"},
        # a residual block of an image network at batch 32
        {"name": "residual_batch32", "kind": "residual", "batch": 32, "height": 56, "width": 56, "channels": 256,
         "mid": 64, "act": "relu"},
        # a depthwise block on a single image with sides that no tile divides
        {"name": "inverted_one_image", "kind": "inverted", "batch": 1, "height": 57, "width": 43, "channels": 24,
         "expand": 144, "n": 24, "stride": 1},
        # an image network's entry at batch 32
        {"name": "stem_batch32", "kind": "stem", "batch": 32, "height": 224, "width": 224, "kernel": 7, "n": 64,
         "channels_last": True},
    ]


# ---------------------------------------------------------------------------------------------
# the ranges the listed cases stand for
# ---------------------------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """A feature or channel count: half of them multiples of 64, a quarter of 8, the rest anything."""
    n, r = _log_int(rng, lo, hi), rng.random()
    step = 64 if r < 0.5 and n >= 64 else 8 if r < 0.75 and n >= 8 else 1
    return max(step, (n + step // 2) // step * step)


def draw(rng):
    while True:
        kind = rng.choice(["mlp", "mlp", "mlp", "dynamic", "dynamic", "plain", "codec", "range_codec", "channels",
                           "residual", "residual", "inverted", "inverted", "stem"])
        flip = lambda: rng.random() < 0.5  # noqa: E731
        if kind == "mlp":
            case = {"kind": kind, "rows": _log_int(rng, 1, 4096), "k": _features(rng, 64, 8192),
                    "hidden": _features(rng, 64, 12288), "n": _features(rng, 64, 8192),
                    "dtype": rng.choice(["quint8", "qint8"]), "per_channel": flip(), "bias": flip()}
        elif kind == "dynamic":
            case = {"kind": kind, "rows": _log_int(rng, 1, 4096), "k": _features(rng, 64, 8192),
                    "n": _features(rng, 64, 12288), "per_channel": flip(), "bias": flip(), "relu": flip()}
        elif kind == "plain":
            case = {"kind": kind, "rows": _log_int(rng, 1, 4096), "k": _features(rng, 64, 4096),
                    "n": _features(rng, 64, 4096), "dtype": rng.choice(["uint8", "int8"]),
                    "out": rng.choice(["uint8", "int8", "bfloat16"]), "post": rng.choice(["none", "relu"])}
        elif kind in ("codec", "range_codec"):
            case = {"kind": kind, "rows": _log_int(rng, 1, 16384), "cols": _features(rng, 64, 16384),
                    "dtype": rng.choice(["quint8", "qint8"])}
        elif kind == "channels":
            case = {"kind": kind, "shape0": _features(rng, 16, 12288), "shape1": _features(rng, 16, 12288),
                    "axis": rng.choice([0, 0, 0, 1]), "dtype": "qint8"}
        elif kind == "residual":
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "height": _log_int(rng, 7, 80),
                    "width": _log_int(rng, 7, 80), "channels": _features(rng, 32, 1024), "mid": _features(rng, 16, 512),
                    "act": rng.choice(["relu", "silu"])}
        elif kind == "inverted":
            channels = _features(rng, 16, 160)
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "height": _log_int(rng, 7, 112),
                    "width": _log_int(rng, 7, 112), "channels": channels, "expand": 6 * channels,
                    "n": channels if flip() else _features(rng, 16, 320), "stride": rng.choice([1, 1, 2])}
        else:
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "height": _log_int(rng, 96, 640),
                    "width": _log_int(rng, 96, 640), "kernel": rng.choice([3, 7]), "n": rng.choice([16, 24, 32, 48, 64]),
                    "channels_last": rng.random() < 0.75}
        # no more than the largest listed case: an odd feature count only up to a few dozen giga-operations
        w = work(case)
        most = 3e11 if not _odd(case) else 3e10
        if w["flops"] <= most and w["bytes"] <= 2.6e9:
            return case


def _odd(case):
    sizes = [case[x] for x in ("k", "hidden", "n", "channels", "mid", "expand") if x in case]
    return any(s % 16 for s in sizes)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * std


def _weight(gen, *shape, std, per_channel=True):
    """A float weight, quantized symmetrically to qint8 (per output channel or per tensor)."""
    w = _normal(gen, *shape, std=std)
    if per_channel:
        scales = w.abs().flatten(1).amax(1).clamp_min(1e-6) / 127
        return torch.quantize_per_channel(w, scales.double(), torch.zeros(shape[0], dtype=torch.long, device="cuda"), 0,
                                          torch.qint8)
    return torch.quantize_per_tensor(w, float(w.abs().max()) / 127, 0, torch.qint8)


def _linear(gen, n, k, per_channel, bias):
    b = _normal(gen, n, std=0.1) if bias else None
    return _OPS.linear_prepack(_weight(gen, n, k, std=0.02, per_channel=per_channel), b)


def _conv(gen, oc, ic_per_group, k, stride, pad, groups):
    w = _weight(gen, oc, ic_per_group, k, k, std=1.0 / math.sqrt(ic_per_group * k * k))
    return _OPS.conv2d_prepack(w, _normal(gen, oc, std=0.1), [stride, stride], [pad, pad], [1, 1], groups)


def _symmetric(dtype):
    return 0 if dtype == "qint8" else 128


def _feature_map(gen, case):
    """A quantized activation as it stands behind a ReLU: channels-last, quint8, zero point 0."""
    x = torch.relu(_normal(gen, case["batch"], case["height"], case["width"], case["channels"])).permute(0, 3, 1, 2)
    return torch.quantize_per_tensor(x, 4.0 / 255, 0, torch.quint8)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "mlp":
        k, h, n = case["k"], case["hidden"], case["n"]
        s["x"] = _normal(gen, case["rows"], k)
        s["dtype"] = _DTYPES[case["dtype"]]
        s["up"] = _linear(gen, h, k, case["per_channel"], case["bias"])
        s["down"] = _linear(gen, n, h, case["per_channel"], case["bias"])
        # four standard deviations to either side span the codes; behind the ReLU one side does
        mid = 0.02 * math.sqrt(k)
        s["q_in"] = (8.0 / 255, _symmetric(case["dtype"]))
        s["q_mid"] = (4 * mid / 255, 0) if case["dtype"] == "quint8" else (4 * mid / 127, 0)
        s["q_out"] = (8 * 0.02 * mid * math.sqrt(h / 2) / 255, _symmetric(case["dtype"]))
    elif kind == "dynamic":
        s["x"] = _normal(gen, case["rows"], case["k"])
        s["w"] = _linear(gen, case["n"], case["k"], case["per_channel"], case["bias"])
        s["op"] = _OPS.linear_relu_dynamic if case["relu"] else _OPS.linear_dynamic
    elif kind == "plain":
        m, k, n = case["rows"], case["k"], case["n"]
        signed = case["dtype"] == "int8"
        codes = (_normal(gen, m, k) * 32 + (0 if signed else 128)).round()
        s["x"] = codes.clamp(-128 if signed else 0, 127 if signed else 255).to(torch.int8 if signed else torch.uint8)
        s["x_q"] = (1.0 / 32, 0 if signed else 128)
        s["w"] = (_normal(gen, k, n) * 32).round().clamp(-127, 127).to(torch.int8)
        s["w_scales"] = torch.rand(n, generator=gen, device="cuda") * 2e-4 + 5e-4
        s["w_zps"] = torch.zeros(n, dtype=torch.long, device="cuda")
        s["bias"] = _normal(gen, n, std=0.1)
        s["out"] = getattr(torch, case["out"])
        s["y_q"] = (8 * 0.02 * math.sqrt(k) / 255, 128 if case["out"] == "uint8" else 0)
        if case["out"] == "bfloat16":
            s["y_q"] = (1.0, 0)
        s["post"] = case["post"]
    elif kind in ("codec", "range_codec"):
        x = _normal(gen, case["rows"], case["cols"], std=3.0)
        # one value in a hundred is an outlier
        s["x"] = x.masked_fill_(torch.rand(x.shape, generator=gen, device="cuda") < 0.01, 50.0)
        s["dtype"] = _DTYPES[case["dtype"]]
        s["q"] = (100.0 / 255, _symmetric(case["dtype"]))
    elif kind == "channels":
        s["x"] = _normal(gen, case["shape0"], case["shape1"], std=0.02)
        s["axis"] = case["axis"]
        s["dtype"] = _DTYPES[case["dtype"]]
        s["scales"] = s["x"].abs().amax(1 - case["axis"]).double().clamp_min(1e-6) / 127
        s["zps"] = torch.zeros(s["scales"].numel(), dtype=torch.long, device="cuda")
    elif kind == "residual":
        c, mid = case["channels"], case["mid"]
        s["x"] = _feature_map(gen, case)
        s["reduce"] = _conv(gen, mid, c, 1, 1, 0, 1)
        s["spatial"] = _conv(gen, mid, mid, 3, 1, 1, 1)
        s["expand"] = _conv(gen, c, mid, 1, 1, 0, 1)
        silu = case["act"] == "silu"
        s["op"] = _OPS.conv2d_silu if silu else _OPS.conv2d_relu
        s["add_op"] = _OPS.conv2d_add_silu if silu else _OPS.conv2d_add_relu
        s["q"] = (4.0 / 250, 14) if silu else (4.0 / 255, 0)
    elif kind == "inverted":
        c, e, n, st = case["channels"], case["expand"], case["n"], case["stride"]
        s["x"] = _feature_map(gen, case)
        s["expand"] = _conv(gen, e, c, 1, 1, 0, 1)
        s["depthwise"] = _conv(gen, e, 1, 3, st, 1, e)
        s["project"] = _conv(gen, n, e, 1, 1, 0, 1)
        s["add"] = n == c and st == 1
    else:
        x = torch.rand(case["batch"], 3, case["height"], case["width"], generator=gen, device="cuda") * 4 - 2
        s["x"] = x.contiguous(memory_format=torch.channels_last) if case["channels_last"] else x
        s["conv"] = _conv(gen, case["n"], 3, case["kernel"], 2, case["kernel"] // 2, 1)
    return s


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "mlp":
        x = torch.quantize_per_tensor(s["x"], *s["q_in"], s["dtype"])
        h = _OPS.linear_relu(x, s["up"], *s["q_mid"])
        return _OPS.linear(h, s["down"], *s["q_out"]).dequantize()
    if kind == "dynamic":
        return s["op"](s["x"], s["w"])
    if kind == "plain":
        return _OPS.linear_per_tensor(s["x"], *s["x_q"], s["w"], s["w_scales"], s["w_zps"], s["bias"], *s["y_q"],
                                      s["out"], s["post"], [], "")
    if kind == "codec":
        return torch.quantize_per_tensor(s["x"], *s["q"], s["dtype"]).dequantize()
    if kind == "range_codec":
        return torch.quantize_per_tensor_dynamic(s["x"], s["dtype"], False).dequantize()
    if kind == "channels":
        return torch.quantize_per_channel(s["x"], s["scales"], s["zps"], s["axis"], s["dtype"]).dequantize()
    if kind == "residual":
        x = s["x"]
        y = s["op"](x, s["reduce"], *s["q"])
        y = s["op"](y, s["spatial"], *s["q"])
        return s["add_op"](y, x, s["expand"], *s["q"]).dequantize()
    if kind == "inverted":
        x = s["x"]
        y = _OPS.conv2d_relu(x, s["expand"], 4.0 / 255, 0)
        y = _OPS.conv2d_relu(y, s["depthwise"], 4.0 / 255, 0)
        y = _OPS.conv2d(y, s["project"], 8.0 / 255, 128)
        if s["add"]:
            y = _OPS.add(y, x, 8.0 / 255, 100)
        return y.dequantize()
    x = torch.quantize_per_tensor(s["x"], 4.0 / 255, 128, torch.quint8)
    y = _OPS.conv2d_relu(x, s["conv"], 4.0 / 255, 0)
    return torch.nn.functional.max_pool2d(y, 3, 2, 1).dequantize()


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far another correct one may be off
# ---------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        m, k, h, n = case["rows"], case["k"], case["hidden"], case["n"]
        return {"bytes": 4 * m * (k + n) + h * (k + n) + 8 * (h + n), "flops": 2 * m * h * (k + n)}
    if kind == "dynamic":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 4 * m * (k + n) + n * k + 8 * n, "flops": 2 * m * n * k}
    if kind == "plain":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": m * k + n * k + 8 * n + m * n * (2 if case["out"] == "bfloat16" else 1), "flops": 2 * m * n * k}
    if kind in ("codec", "range_codec"):
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 4 * case["rows"] * case["cols"]}
    if kind == "channels":
        return {"bytes": 8 * case["shape0"] * case["shape1"], "flops": 4 * case["shape0"] * case["shape1"]}
    b, h, w = case["batch"], case["height"], case["width"]
    if kind == "residual":
        c, mid = case["channels"], case["mid"]
        weights = 2 * c * mid + 9 * mid * mid
        return {"bytes": 5 * b * h * w * c + weights, "flops": 2 * b * h * w * weights}
    if kind == "inverted":
        c, e, n, st = case["channels"], case["expand"], case["n"], case["stride"]
        oh, ow = (h - 1) // st + 1, (w - 1) // st + 1
        return {"bytes": b * h * w * c + 4 * b * oh * ow * n + e * (c + 9 + n),
                "flops": 2 * b * (h * w * c * e + oh * ow * e * (9 + n))}
    n, k = case["n"], case["kernel"]
    oh, ow = (h - 1) // 2 + 1, (w - 1) // 2 + 1
    ph, pw = (oh - 1) // 2 + 1, (ow - 1) // 2 + 1
    return {"bytes": 12 * b * h * w + 4 * b * ph * pw * n + 3 * n * k * k, "flops": 6 * b * oh * ow * n * k * k}


def tolerance(case):
    kind = case["kind"]
    if kind in ("codec", "range_codec", "channels"):
        return "exact"  # codes and their fp32 values are defined to the last bit
    if kind == "dynamic":
        return {"rel": 1e-5}  # exact integer sums of exact codes, scaled in fp32
    if kind == "plain":
        # one code more or less where the requantisation ties; a rounding of bf16 in the float form
        return {"rel": 4e-3, "max": 0.02} if case["out"] == "bfloat16" else {"rel": 1e-3, "differ": 1e-3}
    # one code more or less, of about 32 to a standard deviation, on the few values that tie
    return {"rel": 2e-3, "max": 0.1}
