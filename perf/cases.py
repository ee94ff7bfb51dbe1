"""The workloads that the speed of this library is judged by, through ``torch.ops.mi355x``.

Twelve listed cases stand for what a program has this operator family do: the decode step and the
training steps of a language model (RMSNorm, LayerNorm, attention softmax, the cross-entropy's
log_softmax), attention rows of image models, GroupNorm over feature maps, normalization over
whole images, softmax over a leading dimension, and rows that fit no vector width.  Sizes are those
of ``bench.py`` and of the tests.  ``draw`` gives further cases of the same kinds over the ranges
that ``RANGES`` states.

A case is a dict of plain values; ``kind`` names the operator and the other entries its sizes and
types.  Every kind but the decode step runs forward and backward and returns all outputs of both.
"""
import importlib
import math

import torch

EPS = 1e-5
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def listed():
    return [
        # one token for each of 8 sequences: the residual add and RMSNorm between two layers of
        # a 4096-wide model while it decodes.  Latency, not bandwidth.
        {"name": "decode_add_rms_norm", "kind": "add_rms_norm", "dtype": "bfloat16", "rows": 8,
         "n": 4096},
        # LayerNorm in float32 over a batch that fits the caches
        {"name": "layer_norm_float32", "kind": "layer_norm", "dtype": "float32",
         "weight": "float32", "rows": 4096, "n": 1024, "offset": 0, "outliers": False},
        # a training micro-batch of 16384 tokens through RMSNorm at hidden 4096
        {"name": "rms_norm_training", "kind": "rms_norm", "dtype": "bfloat16", "rows": 16384,
         "n": 4096},
        # mixed precision: bfloat16 activations, float32 weights, hidden 8192
        {"name": "layer_norm_mixed", "kind": "layer_norm", "dtype": "bfloat16",
         "weight": "float32", "rows": 16384, "n": 8192, "offset": 0, "outliers": False},
        # rows off every vector width in tensors off a 16-byte boundary, with outliers
        {"name": "layer_norm_irregular", "kind": "layer_norm", "dtype": "float16",
         "weight": "float16", "rows": 8192, "n": 4097, "offset": 2, "outliers": True},
        # normalization over whole feature maps: few rows of 0.4 M elements
        {"name": "layer_norm_maps", "kind": "layer_norm", "dtype": "bfloat16",
         "weight": "bfloat16", "rows": 512, "n": 3136 * 128, "offset": 0, "outliers": False},
        # attention scores of a language model under a causal mask (-inf above the diagonal)
        {"name": "softmax_causal", "kind": "softmax", "dtype": "bfloat16", "heads": 4 * 32,
         "queries": 2048, "n": 2048, "causal": True, "log": False},
        # attention of a vision transformer: 14 x 14 patches and a class token
        {"name": "softmax_vision", "kind": "softmax", "dtype": "bfloat16", "heads": 64 * 12,
         "queries": 197, "n": 197, "causal": False, "log": False},
        # the cross-entropy of 4096 tokens over a vocabulary of 128256
        {"name": "log_softmax_vocabulary", "kind": "softmax", "dtype": "bfloat16", "heads": 1,
         "queries": 4096, "n": 128256, "causal": False, "log": True},
        # softmax over the leading dimension of a matrix
        {"name": "softmax_leading", "kind": "softmax_dim", "dtype": "bfloat16", "outer": 1,
         "d": 8192, "inner": 8192},
        # GroupNorm in a convolutional network: 14 x 14 maps, 32 groups
        {"name": "group_norm_conv", "kind": "group_norm", "dtype": "bfloat16", "batch": 256,
         "channels": 1024, "side": 14, "groups": 32},
        # GroupNorm in an image decoder: few, large maps
        {"name": "group_norm_decoder", "kind": "group_norm", "dtype": "bfloat16", "batch": 2,
         "channels": 256, "side": 256, "groups": 32},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high, step):
    """A row length in [low, high]: three of four are whole multiples of `step`, as the widths of
    models are, the others anything."""
    n = _log_uniform(rng, low, high)
    return max(step, n // step * step) if rng.random() < 0.75 else n


def draw(rng):
    kind = rng.choice(["decode", "rms_norm", "layer_norm", "mixed", "irregular", "maps", "causal",
                       "vision", "vocabulary", "softmax_dim", "conv", "decoder"])
    if kind == "decode":
        return {"kind": "add_rms_norm", "dtype": rng.choice(["bfloat16", "float16"]),
                "rows": _log_uniform(rng, 1, 256), "n": _width(rng, 1024, 8192, 64)}
    if kind == "rms_norm":
        return {"kind": "rms_norm", "dtype": rng.choice(["bfloat16", "float16"]),
                "rows": _log_uniform(rng, 256, 16384), "n": _width(rng, 1024, 8192, 128)}
    if kind == "layer_norm":
        return {"kind": "layer_norm", "dtype": "float32", "weight": "float32",
                "rows": _log_uniform(rng, 64, 16384), "n": _width(rng, 256, 4096, 64),
                "offset": 0, "outliers": False}
    if kind == "mixed":
        return {"kind": "layer_norm", "dtype": rng.choice(["bfloat16", "float16"]),
                "weight": rng.choice(["float32", "same"]), "rows": _log_uniform(rng, 256, 16384),
                "n": _width(rng, 1024, 12288, 128), "offset": 0, "outliers": False}
    if kind == "irregular":
        return {"kind": "layer_norm", "dtype": rng.choice(["float16", "float32"]),
                "weight": "same", "rows": _log_uniform(rng, 1024, 8192),
                "n": _log_uniform(rng, 64, 16384) | 1, "offset": 2, "outliers": True}
    if kind == "maps":
        n = 128 * _log_uniform(rng, 400, 16384)
        return {"kind": "layer_norm", "dtype": "bfloat16", "weight": "bfloat16",
                "rows": _log_uniform(rng, 2, max(4, min(512, (200 << 20) // n))), "n": n,
                "offset": 0, "outliers": False}
    if kind == "causal":
        t = _width(rng, 128, 2048, 64)
        return {"kind": "softmax", "dtype": rng.choice(["bfloat16", "float16"]),
                "heads": _log_uniform(rng, 8, 128), "queries": t, "n": t, "causal": True,
                "log": False}
    if kind == "vision":
        t = rng.randint(49, 729)
        return {"kind": "softmax", "dtype": rng.choice(["bfloat16", "float16"]),
                "heads": _log_uniform(rng, 16, 1024), "queries": t, "n": t, "causal": False,
                "log": False}
    if kind == "vocabulary":
        return {"kind": "softmax", "dtype": "bfloat16", "heads": 1,
                "queries": _log_uniform(rng, 64, 4096), "n": _width(rng, 30000, 152064, 64),
                "causal": False, "log": rng.random() < 0.75}
    if kind == "softmax_dim":
        d, inner = _log_uniform(rng, 16, 8192), _width(rng, 64, 16384, 64)
        return {"kind": "softmax_dim", "dtype": "bfloat16",
                "outer": _log_uniform(rng, 1, max(1, min(256, (1 << 26) // (d * inner)))), "d": d,
                "inner": inner}
    if kind == "conv":
        side = rng.choice([7, 8, 14, 16, 28, 32, 56, 64])
        channels = 32 * rng.randint(4, 64)
        most = max(1, min(256, (50 << 20) // (channels * side * side)))
        return {"kind": "group_norm", "dtype": "bfloat16", "batch": _log_uniform(rng, 1, most),
                "channels": channels, "side": side, "groups": 32}
    channels, side = rng.choice([128, 256, 512]), _log_uniform(rng, 96, 512) // 8 * 8
    most = max(1, (34 << 20) // (channels * side * side))
    return {"kind": "group_norm", "dtype": "bfloat16", "batch": rng.randint(1, min(8, most)),
            "channels": channels, "side": side, "groups": 32}


def _row_shape(case):
    kind = case["kind"]
    if kind == "softmax":
        return (case["heads"], case["queries"], case["n"])
    if kind == "softmax_dim":
        return (case["outer"], case["d"], case["inner"])
    if kind == "group_norm":
        return (case["batch"], case["channels"], case["side"], case["side"])
    return (case["rows"], case["n"])


def _weight_dtype(case):
    name = case.get("weight", "same")
    return DTYPES[case["dtype"] if name == "same" else name]


def _normal(g, shape, dtype, scale=1.0, offset=0, outliers=False):
    """N(0, scale), `offset` elements into its buffer; with `outliers` one entry in a thousand is
    +-1e4 and the first row is constant."""
    numel = math.prod(shape)
    flat = torch.empty(numel + offset, dtype=dtype, device="cuda")[offset:]
    flat.normal_(0.0, scale, generator=g)
    if outliers:
        at = torch.randint(0, numel, (max(1, numel // 1000),), device="cuda", generator=g)
        flat[at] = torch.where(at % 2 == 0, -1e4, 1e4).to(dtype)
        flat[:shape[-1]] = 0.5
    return flat.view(shape)


def prepare(case, seed):
    ops = importlib.import_module("torch-xpu-ops_amd").load_host_library()
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype, shape, kind = DTYPES[case["dtype"]], _row_shape(case), case["kind"]
    state = {"case": dict(case), "ops": ops}
    softmax = kind in ("softmax", "softmax_dim")
    state["x"] = _normal(g, shape, dtype, 3.0 if softmax else 1.0, case.get("offset", 0),
                         case.get("outliers", False))
    if case.get("causal"):
        above = torch.ones(shape[1:], dtype=torch.bool, device="cuda").triu_(1)
        state["x"].masked_fill_(above, float("-inf"))
    # the residual stream of the decode step, the gradient of the output everywhere else
    state["dy"] = _normal(g, shape, dtype, 1.0, case.get("offset", 0))
    if not softmax:
        width = case["channels"] if kind == "group_norm" else case["n"]
        wd = _weight_dtype(case)
        state["w"] = (1 + 0.1 * torch.randn(width, device="cuda", generator=g)).to(wd)
        state["b"] = (0.1 * torch.randn(width, device="cuda", generator=g)).to(wd)
    return state


def run(state):
    case, ops, x, dy = state["case"], state["ops"], state["x"], state["dy"]
    kind = case["kind"]
    if kind == "add_rms_norm":
        return ops.add_rms_norm(x, dy, [case["n"]], state["w"], EPS)
    if kind == "rms_norm":
        y, rstd = ops._fused_rms_norm(x, [case["n"]], state["w"], EPS)
        return [y, rstd, ops._fused_rms_norm_backward(dy, x, [case["n"]], rstd, state["w"],
                                                      [True, True])]
    if kind == "layer_norm":
        w, b = state["w"], state["b"]
        y, mean, rstd = ops.native_layer_norm(x, [case["n"]], w, b, EPS)
        return [y, mean, rstd, ops.native_layer_norm_backward(dy, x, [case["n"]], mean, rstd, w, b,
                                                              [True, True, True])]
    if kind == "group_norm":
        n, c, side, groups = case["batch"], case["channels"], case["side"], case["groups"]
        w, b = state["w"], state["b"]
        y, mean, rstd = ops.native_group_norm(x, w, b, n, c, side * side, groups, EPS)
        return [y, mean, rstd, ops.native_group_norm_backward(dy, x, mean, rstd, w, n, c,
                                                              side * side, groups,
                                                              [True, True, True])]
    dim = 1 if kind == "softmax_dim" else -1
    if case.get("log"):
        y = ops._log_softmax(x, dim, False)
        return [y, ops._log_softmax_backward_data(dy, y, dim, x.dtype)]
    y = ops._softmax(x, dim, False)
    return [y, ops._softmax_backward_data(dy, y, dim, x.dtype)]


def work(case):
    """Forward: x read, y written (and the residual read, h written in the decode step).  Backward:
    dy and x (softmax: y) read, dx written.  Weights, statistics and weight gradients once each."""
    kind, numel = case["kind"], math.prod(_row_shape(case))
    esize = DTYPES[case["dtype"]].itemsize
    if kind in ("softmax", "softmax_dim"):
        return {"bytes": 5 * numel * esize, "flops": 9 * numel}
    if kind == "add_rms_norm":
        return {"bytes": 4 * numel * esize + case["n"] * esize + 4 * case["rows"],
                "flops": 5 * numel}
    wsize = _weight_dtype(case).itemsize
    if kind == "group_norm":
        width, rows, stat = case["channels"], case["batch"] * case["groups"], wsize
    else:
        width, rows, stat = case["n"], case["rows"], 4
    if kind == "rms_norm":
        return {"bytes": 5 * numel * esize + 3 * width * wsize + 2 * rows * stat,
                "flops": 14 * numel}
    return {"bytes": 5 * numel * esize + 5 * width * wsize + 4 * rows * stat, "flops": 20 * numel}


def tolerance(case):
    """About four times the distance of the outputs from the same formulas in float64."""
    return {"float32": {"rel": 2e-6, "max": 1e-5}, "float16": {"rel": 9e-4, "max": 4e-2},
            "bfloat16": {"rel": 7e-3, "max": 8e-2}}[case["dtype"]]
