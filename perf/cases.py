"""Workloads of the kernel library, called as a model's code calls them.

Each case is one call through a torch-facing function of hip_oracles: a
normalisation, a softmax, an activation, a layout change, a pooling or a
BatchNorm of a training or inference step.  listed() holds sizes that the
models of the corpus run (ViT / DeiT at 197 tokens, Visformer, NFNet,
EfficientNet, ShuffleNet, Qwen3-style head norms, causal attention); draw()
gives others of the same ranges: from calls whose launch is their cost up to
a few hundred MB, rows and planes that are whole vectors and ones that are
not, fp32 and bf16, and every option of the calls.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "better-benchmark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hip_oracles as ho  # noqa: E402

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def listed():
    return [
        # Classifier-sized fp32 row mean: a call that its launch dominates.
        {"name": "row_mean_300x1000", "op": "row_mean", "rows": 300, "cols": 1000,
         "dtype": "f32", "relu": False},
        # Residual LayerNorm of a ViT-Base block, 128 images of 197 tokens.
        {"name": "layernorm_25216x768", "op": "layernorm", "rows": 25216, "cols": 768,
         "outputs": "hy"},
        # Per-head RMSNorm of the queries: 1000 tokens x 16 heads of 128.
        {"name": "rmsnorm_16000x128", "op": "rmsnorm", "rows": 16000, "cols": 128,
         "residual": False, "want_h": False, "mode": 0, "scale": 1.0},
        # Attention probabilities of a ViT-Base block: rows of 197.
        {"name": "softmax_1536x197x197", "op": "softmax", "batch": 1536, "q": 197, "k": 197,
         "heads": 12, "kind": "plain"},
        # Causal attention, 24 sequences x 16 heads of 1024 tokens (the largest).
        {"name": "softmax_384x1024x1024", "op": "softmax", "batch": 384, "q": 1024, "k": 1024,
         "heads": 16, "kind": "causal"},
        # Bias + GELU of a convolution output to channels-last, 14 x 14 planes.
        {"name": "bias_gelu_128x384x14x14", "op": "bias_gelu", "n": 128, "c": 384, "h": 14,
         "w": 14},
        # Backward of the ViT-Base MLP's GELU with its bias gradient.
        {"name": "gelu_bwd_25216x3072", "op": "gelu_bwd", "rows": 25216, "cols": 3072},
        # Tokens to channels of a ViT feature map (matrices of 197 x 768).
        {"name": "transpose_128x197x768", "op": "transpose", "batch": 128, "rows": 197,
         "cols": 768, "dtype": "bf16"},
        # NFNet squeeze-excite pooling, channels-last 12 x 12.
        {"name": "spatial_mean_128x1536x12x12", "op": "spatial_mean", "n": 128, "c": 1536,
         "h": 12, "w": 12},
        # BatchNorm training forward of a ResNet's last stage (odd 7 x 7 planes, fp32).
        {"name": "bn_train_128x2048x7x7", "op": "bn_train", "n": 128, "c": 2048, "h": 7, "w": 7,
         "relu": True},
        # EfficientNet's BatchNorm + SiLU + pad, channels-last.
        {"name": "bn_nhwc_128x240x28x28", "op": "bn_nhwc", "n": 128, "c": 240, "h": 28, "w": 28,
         "act": "silu", "pad": 1},
        # ShuffleNet's last BatchNorm + ReLU + global pooling.
        {"name": "bn_nchw_mean_128x1024x7x7", "op": "bn_nchw", "n": 128, "c": 1024, "h": 7,
         "w": 7, "act": "relu"},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi):
    """A row length or channel count: half of them multiples of 64, a quarter
    multiples of 8, the others any number."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(step, v // step * step)


def _plane(rng, hi):
    """Height and width: the usual halvings of 224, or any rectangle."""
    if rng.random() < 0.6:
        s = rng.choice([v for v in (7, 14, 28, 56, 112) if v <= hi])
        return s, s
    h = rng.randint(5, hi)
    return h, max(5, min(hi, h + rng.randint(-3, 3)))


def draw(rng):
    op = rng.choice(("row_mean", "layernorm", "rmsnorm", "softmax", "bias_gelu", "gelu_bwd",
                     "transpose", "spatial_mean", "bn_train", "bn_nhwc", "bn_nchw"))
    most = 1 << 25  # elements of the main input
    if op == "row_mean":
        cols = _width(rng, 16, 16384)
        return {"op": op, "rows": _log(rng, 4, min(65536, most // cols)), "cols": cols,
                "dtype": rng.choice(("f32", "bf16")), "relu": rng.random() < 0.5}
    if op == "layernorm":
        cols = _width(rng, 64, 8192)
        return {"op": op, "rows": _log(rng, 8, min(65536, most // cols)), "cols": cols,
                "outputs": rng.choice(("all", "hy", "y"))}
    if op == "rmsnorm":
        cols = _width(rng, 64, 8192)
        residual = rng.random() < 0.5
        return {"op": op, "rows": _log(rng, 8, min(65536, most // cols)), "cols": cols,
                "residual": residual, "want_h": residual and rng.random() < 0.5,
                "mode": rng.choice((0, 1)), "scale": rng.choice((1.0, 1.0, 0.125))}
    if op == "softmax":
        heads = rng.choice((4, 6, 8, 12, 16))
        k = _width(rng, 48, 2048)
        q = k if rng.random() < 0.75 else _log(rng, 1, k)
        seqs = max(1, min(64, _log(rng, 1, 64), most // (heads * q * k)))
        return {"op": op, "batch": seqs * heads, "q": q, "k": k, "heads": heads,
                "kind": rng.choice(("plain", "causal", "bias"))}
    if op == "bias_gelu":
        h, w = _plane(rng, 112)
        c = _width(rng, 16, 1024)
        return {"op": op, "n": max(1, min(128, _log(rng, 2, 128), most // (c * h * w))), "c": c,
                "h": h, "w": w}
    if op == "gelu_bwd":
        cols = max(64, _log(rng, 64, 8192) // 8 * 8)
        return {"op": op, "rows": _log(rng, 8, min(32768, most // cols)), "cols": cols}
    if op == "transpose":
        rows, cols = _width(rng, 32, 4096), _width(rng, 32, 2048)
        return {"op": op, "batch": max(1, min(768, _log(rng, 1, 768), most // (rows * cols))),
                "rows": rows, "cols": cols, "dtype": rng.choice(("bf16", "bf16", "f32"))}
    if op == "spatial_mean":
        h, w = _plane(rng, 64)
        c = _width(rng, 16, 2304)
        return {"op": op, "n": max(1, min(128, _log(rng, 4, 128), most // (c * h * w))), "c": c,
                "h": h, "w": w}
    if op == "bn_train":
        h, w = _plane(rng, 112)
        c = _width(rng, 16, 2048)
        return {"op": op, "n": max(2, min(128, _log(rng, 4, 128), most // (c * h * w))), "c": c,
                "h": h, "w": w, "relu": rng.random() < 0.5}
    if op == "bn_nhwc":
        h, w = _plane(rng, 112)
        c = _width(rng, 16, 1024)
        return {"op": op, "n": max(2, min(128, _log(rng, 4, 128), most // (c * h * w))), "c": c,
                "h": h, "w": w, "act": rng.choice(("silu", "relu", "none")),
                "pad": rng.choice((0, 1))}
    h, w = _plane(rng, 28)
    c = _width(rng, 32, 2048)
    return {"op": op, "n": max(2, min(256, _log(rng, 4, 256), most // (c * h * w))), "c": c,
            "h": h, "w": w, "act": rng.choice(("silu", "relu", "none"))}


def _bn_params(c, rand):
    return {"gamma": 1 + 0.1 * rand(c), "beta": 0.1 * rand(c),
            "rm": torch.zeros(c, dtype=F32, device="cuda"),
            "rv": torch.ones(c, dtype=F32, device="cuda")}


def _bessel(case):
    m = case["n"] * case["h"] * case["w"]
    return m / (m - 1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))

    def rand(*shape, dtype=F32):
        return torch.randn(*shape, generator=gen, dtype=dtype, device="cuda")

    op = case["op"]
    s = {"case": case}
    if op == "row_mean":
        s["x"] = rand(case["rows"], case["cols"], dtype=F32 if case["dtype"] == "f32" else BF16)
    elif op in ("layernorm", "rmsnorm"):
        rows, cols = case["rows"], case["cols"]
        s["x"] = rand(rows, cols, dtype=BF16)
        if op == "layernorm" or case["residual"]:
            s["res"] = rand(rows, cols, dtype=BF16)
        s["gamma"] = (1 + 0.1 * rand(cols)).to(BF16)
        if op == "layernorm":
            s["beta"] = (0.1 * rand(cols)).to(BF16)
    elif op == "softmax":
        b, q, k = case["batch"], case["q"], case["k"]
        s["x"] = rand(b, q, k, dtype=BF16)
        if case["kind"] == "causal":
            s["mask"] = torch.full((q, k), -math.inf, dtype=BF16, device="cuda").triu(k - q + 1)
        elif case["kind"] == "bias":
            s["bias"] = rand(b // case["heads"], q, k, dtype=BF16)
    elif op == "bias_gelu":
        s["x"] = rand(case["n"], case["c"], case["h"], case["w"], dtype=BF16)
        s["bias"] = (0.1 * rand(case["c"])).to(BF16)
    elif op == "gelu_bwd":
        s["grad"] = rand(case["rows"], case["cols"], dtype=BF16)
        s["x"] = rand(case["rows"], case["cols"], dtype=BF16)
    elif op == "transpose":
        s["x"] = rand(case["batch"], case["rows"], case["cols"],
                      dtype=F32 if case["dtype"] == "f32" else BF16)
    elif op == "spatial_mean":
        s["x"] = rand(case["n"], case["h"], case["w"], case["c"], dtype=BF16).permute(0, 3, 1, 2)
    elif op == "bn_train":
        s["x"] = rand(case["n"], case["c"], case["h"], case["w"]).mul_(2).add_(0.5)
        s.update(_bn_params(case["c"], rand))
    elif op == "bn_nhwc":
        x = rand(case["n"], case["h"], case["w"], case["c"], dtype=BF16).mul_(2).add_(0.5)
        s["x"] = x.permute(0, 3, 1, 2)
        s.update(_bn_params(case["c"], rand))
    else:
        s["x"] = rand(case["n"], case["c"], case["h"], case["w"], dtype=BF16).mul_(2).add_(0.5)
        s.update(_bn_params(case["c"], rand))
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "row_mean":
        if case["dtype"] == "f32":
            return ho.row_mean(s["x"])
        return ho.row_mean_bf16(s["x"], relu=case["relu"])
    if op == "layernorm":
        return ho.residual_layernorm(s["x"], s["res"], s["gamma"], s["beta"], 1e-5,
                                     outputs=case["outputs"])
    if op == "rmsnorm":
        return ho.rmsnorm_ex(s["x"], s["gamma"], 1e-6, residual=s.get("res"),
                             scale=case["scale"], mode=case["mode"], want_h=case["want_h"])
    if op == "softmax":
        if case["kind"] == "plain":
            return ho.softmax_lastdim(s["x"])
        if case["kind"] == "causal":
            return ho.scaled_masked_softmax(s["x"], s["mask"], 0.125)
        return ho.scaled_bias_softmax(s["x"], s["bias"], 0.125, case["heads"])
    if op == "bias_gelu":
        return ho.bias_gelu_nchw_to_nhwc(s["x"], s["bias"])
    if op == "gelu_bwd":
        return ho.gelu_erf_bwd_colsum(s["grad"], s["x"])
    if op == "transpose":
        return ho.transpose_last2(s["x"])
    if op == "spatial_mean":
        return ho.spatial_mean_nhwc(s["x"])
    if op == "bn_train":
        out = ho.batchnorm_train(s["x"], s["gamma"], s["beta"], s["rm"], s["rv"], momentum=0.1,
                                 eps=1e-5, relu=case["relu"])
    elif op == "bn_nhwc":
        out = ho.batchnorm_nhwc_act_pad(s["x"], s["gamma"], s["beta"], s["rm"], s["rv"],
                                        momentum=0.1, eps=1e-3, var_scale=_bessel(case),
                                        act=case["act"], pad_bottom=case["pad"],
                                        pad_right=case["pad"])
    else:
        out = ho.batchnorm_nchw_act_mean(s["x"], s["gamma"], s["beta"], s["rm"], s["rv"],
                                         momentum=0.1, eps=1e-5, var_scale=_bessel(case),
                                         act=case["act"])
    return (*out, s["rm"], s["rv"])


def work(case):
    op = case["op"]
    if op == "row_mean":
        e = 4 if case["dtype"] == "f32" else 2
        m = case["rows"] * case["cols"]
        return {"bytes": m * e + case["rows"] * e, "flops": m}
    if op in ("layernorm", "rmsnorm"):
        rows, cols = case["rows"], case["cols"]
        m = rows * cols
        if op == "layernorm":
            streams = 3 + (case["outputs"] != "y")
            side = 8 * rows if case["outputs"] == "all" else 0
            return {"bytes": 2 * streams * m + side + 4 * cols, "flops": 8 * m}
        streams = 2 + case["residual"] + case["want_h"]
        return {"bytes": 2 * streams * m + 2 * cols, "flops": 5 * m}
    if op == "softmax":
        m = case["batch"] * case["q"] * case["k"]
        extra = {"plain": 0, "causal": case["q"] * case["k"],
                 "bias": m // case["heads"]}[case["kind"]]
        return {"bytes": 4 * m + 2 * extra, "flops": 8 * m}
    if op == "gelu_bwd":
        m = case["rows"] * case["cols"]
        return {"bytes": 6 * m + 4 * case["cols"], "flops": 2 * m}
    if op == "transpose":
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": 2 * e * case["batch"] * case["rows"] * case["cols"], "flops": 0}
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    m = n * c * h * w
    if op == "bias_gelu":
        return {"bytes": 4 * m + 2 * c, "flops": 10 * m}
    if op == "spatial_mean":
        return {"bytes": 2 * m + 2 * n * c, "flops": m}
    if op == "bn_train":
        return {"bytes": 8 * m + 32 * c, "flops": 6 * m}
    if op == "bn_nhwc":
        out = n * c * (h + case["pad"]) * (w + case["pad"])
        return {"bytes": 2 * m + 2 * out + 32 * c, "flops": 10 * m}
    return {"bytes": 2 * m + 2 * n * c + 32 * c, "flops": 10 * m}


def tolerance(case):
    """About four times the distance from the 64-bit result: one rounding to
    bf16 is 1.7e-3 of the norm (and up to 2^-8 of a value), two or three in a
    row 3e-3."""
    op = case["op"]
    if op == "transpose":
        return "exact"
    if op == "bn_train" or (op == "row_mean" and case["dtype"] == "f32"):
        return {"rel": 2e-6, "max": 1e-4}
    if op == "rmsnorm" and case["mode"] == 1:
        return {"rel": 1.2e-2, "max": 4e-2}
    return {"rel": 7e-3, "max": 2e-2}


def _act(y, act):
    if act == "relu":
        return torch.relu(y)
    return y * torch.sigmoid(y) if act == "silu" else y


def _bn_exact(s, case, eps):
    x = s["x"].to(F64)
    mean = x.mean((0, 2, 3))
    var = ((x - mean[:, None, None]) ** 2).mean((0, 2, 3))
    rstd = 1 / torch.sqrt(var + eps)
    y = (x - mean[:, None, None]) * (rstd * s["gamma"].to(F64))[:, None, None]
    y += s["beta"].to(F64)[:, None, None]
    rm = 0.1 * mean + 0.9 * s["rm"].to(F64)
    rv = 0.1 * var * _bessel(case) + 0.9 * s["rv"].to(F64)
    return y, mean, rstd, rm, rv


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op == "row_mean":
        x = s["x"].to(F64)
        return (torch.relu(x) if case["relu"] and case["dtype"] == "bf16" else x).mean(1)
    if op == "layernorm":
        hb = (s["x"].to(F32) + s["res"].to(F32)).to(BF16)  # the sum is defined as bf16
        h = hb.to(F64)
        mean = h.mean(1)
        rstd = 1 / torch.sqrt(((h - mean[:, None]) ** 2).mean(1) + 1e-5)
        y = (h - mean[:, None]) * rstd[:, None] * s["gamma"].to(F64) + s["beta"].to(F64)
        return {"all": (h, y, mean, rstd), "hy": (h, y), "y": y}[case["outputs"]]
    if op == "rmsnorm":
        h = s["x"].to(F64)
        if case["residual"]:
            h = (s["x"].to(F32) + s["res"].to(F32)).to(BF16).to(F64)
        y = h / torch.sqrt((h * h).mean(1, keepdim=True) + 1e-6) * s["gamma"].to(F64)
        y = y * case["scale"]
        return (h, y) if case["want_h"] else y
    if op == "softmax":
        x = s["x"].to(F64)
        if case["kind"] == "causal":
            x = x.mul_(0.125).add_(s["mask"].to(F64))
        elif case["kind"] == "bias":
            x = x * 0.125 + s["bias"].to(F64).repeat_interleave(case["heads"], 0)
        return torch.softmax(x, -1)
    if op == "bias_gelu":
        t = (s["x"].to(F32) + s["bias"].to(F32)[:, None, None]).to(BF16).to(F64)
        u = math.sqrt(2 / math.pi) * (t + 0.044715 * t ** 3)
        return t * torch.sigmoid(2 * u)
    if op == "gelu_bwd":
        t = s["x"].to(F64)
        d = 0.5 * torch.erfc(-t / math.sqrt(2)) + t * torch.exp(-t * t / 2) / math.sqrt(2 * math.pi)
        y = s["grad"].to(F64) * d
        return y, y.to(BF16).to(F64).sum(0)  # the bias gradient sums the stored bf16 values
    if op == "transpose":
        return None
    if op == "spatial_mean":
        return s["x"].to(F64).mean((2, 3), keepdim=True)
    if op == "bn_train":
        y, mean, rstd, rm, rv = _bn_exact(s, case, 1e-5)
        return torch.relu(y) if case["relu"] else y, mean, rstd, rm, rv
    eps = 1e-3 if op == "bn_nhwc" else 1e-5
    y, mean, rstd, rm, rv = _bn_exact(s, case, eps)
    y = _act(y, case["act"])
    mean, rstd = mean[None, :, None, None], rstd[None, :, None, None]
    if op == "bn_nchw":
        return mean, rstd, y.mean((2, 3)), rm, rv
    pad = case["pad"]
    return mean, rstd, torch.nn.functional.pad(y, (0, pad, 0, pad)), rm, rv
