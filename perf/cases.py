"""The work a user has this library do, as measured cases: forwards of the quantised Linears (decode and prefill),
weight quantisation, the MX / HiFloat8 activation formats (both directions) and the calibration loops around them
(MinMax, SmoothQuant, AWQ, GPTQ), each through the entry points that a program calls.

`listed()` names the fixed cases, `draw(rng)` gives one more of the same ranges, `prepare` builds what a program holds
before the call, `run` is one pass, `work` the bytes and operations it cannot do without, `tolerance` how far another
correct implementation of the same precision may differ."""
import math
import types

import torch

from amct_amd import ops
from amct_amd.algorithm import awq
from amct_amd.deploy_op import HipQuantizationLinear, HipWeightQuantizedLinear
from amct_amd.quantize_op import gptq, smooth_quant_stats
from amct_amd.quantize_op.utils import calculate_scale_offset, get_weight_min_max_by_granularity
from amct_amd.utils.quant_util import quant_dequant_weight

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
# input widths of the repository's tests and benchmark (hidden and intermediate sizes of Linear layers)
_WIDTHS = (1024, 2048, 4096, 5120, 8192, 11008, 13824, 14336)


def listed():
    return [
        # one token of one request: int4 weight-only up projection with AWQ scaling (the smallest forward)
        dict(name="int4_token", path="weight_only", bits=4, rows=1, n=14336, k=4096, group=128, symmetric=False,
             scaled=True, bias=False, dtype="bf16"),
        # a whole prompt through the same layer (the largest int4 forward)
        dict(name="int4_prompt", path="weight_only", bits=4, rows=2048, n=14336, k=4096, group=128, symmetric=False,
             scaled=True, bias=False, dtype="bf16"),
        # a chunk of a prompt, or many requests at once, through an int8 weight-only down projection of an fp16 model
        dict(name="int8_weight_chunk", path="weight_only", bits=8, rows=200, n=4096, k=11008, group=0, symmetric=True,
             scaled=False, bias=True, dtype="fp16"),
        # a decode batch through an int8 x int8 Linear with live per-token activation scales
        dict(name="w8a8_batch", path="w8a8", rows=16, n=14336, k=4096, dynamic=True, scaled=False, bias=False, dtype="bf16"),
        # a prompt of ragged length through the calibrated (static, SmoothQuant) int8 x int8 Linear
        dict(name="w8a8_prompt", path="w8a8", rows=1500, n=14336, k=4096, dynamic=False, scaled=True, bias=True,
             dtype="bf16"),
        # weight preparation of an int4 deployment: codes, scales and zero-points of one layer
        dict(name="int4_pack", path="pack", n=14336, k=4096, group=128, symmetric=False, dtype="bf16"),
        # MinMax calibration of one layer: extrema -> factors -> fake-quantised weight
        dict(name="minmax_weight", path="minmax", n=4096, k=4096, bits=8, symmetric=True, group=0, dtype="fp32"),
        # activations into MXFP8 and back
        dict(name="mxfp8_round_trip", path="format", fmt="mxfp8", rows=8192, k=4096, dtype="bf16"),
        # AWQ: the scale search of one layer over 20 grid points, then the layer quantised with the winner
        dict(name="awq_search", path="awq", rows=1024, n=4096, k=4096, bits=4, group=128, grids=20, dtype="bf16"),
        # SmoothQuant: the running channel extrema over one calibration batch
        dict(name="smooth_stats", path="stats", rows=8192, k=4096, dtype="bf16"),
        # GPTQ: the Hessian over two calibration batches (the first one starts it, the second one accumulates)
        dict(name="gptq_hessian", path="hessian", rows=2048, k=4096, dtype="bf16"),
        # GPTQ: the optimised weight of one layer
        dict(name="gptq_layer", path="gptq", n=4096, k=4096, bits=4, symmetric=False, group=128, dtype="bf16"),
    ]


def _log(rng, lo, hi, step=1):
    """Log-uniform over [lo, hi], rounded to a multiple of step."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    path = rng.choice(["weight_only"] * 3 + ["w8a8"] * 2 + ["pack", "minmax", "format", "awq", "stats", "hessian", "gptq"])
    dt16 = rng.choice(["bf16", "bf16", "fp16"])
    if path == "weight_only":
        bits = rng.choice([4, 4, 8])
        return dict(path=path, bits=bits, rows=_log(rng, 1, 2048), n=_log(rng, 512, 14336, 8), k=rng.choice(_WIDTHS),
                    group=rng.choice([128, 128, 64] if bits == 4 else [0, 128]), symmetric=rng.random() < 0.5,
                    scaled=rng.random() < 0.5, bias=rng.random() < 0.3, dtype=dt16)
    if path == "w8a8":
        return dict(path=path, rows=_log(rng, 1, 2048), n=_log(rng, 512, 14336, 8), k=rng.choice(_WIDTHS),
                    dynamic=rng.random() < 0.5, scaled=rng.random() < 0.5, bias=rng.random() < 0.3, dtype=dt16)
    if path == "pack":
        return dict(path=path, n=_log(rng, 512, 14336), k=rng.choice(_WIDTHS), group=rng.choice([32, 64, 128]),
                    symmetric=rng.random() < 0.3, dtype=rng.choice(["bf16", "fp16", "fp32"]))
    if path == "minmax":
        return dict(path=path, n=_log(rng, 512, 14336), k=rng.choice(_WIDTHS), bits=rng.choice([4, 8]),
                    symmetric=rng.random() < 0.5, group=rng.choice([0, 0, 128]), dtype=rng.choice(["bf16", "fp16", "fp32"]))
    if path == "format":
        return dict(path=path, fmt=rng.choice(["mxfp8", "mxfp4", "hif8"]), rows=_log(rng, 1, 8192),
                    k=rng.choice([1024, 2048, 4096]), dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    if path == "awq":
        return dict(path=path, rows=_log(rng, 128, 1024), n=_log(rng, 512, 4096, 8), k=rng.choice([1024, 2048, 4096]),
                    bits=4, group=rng.choice([0, 64, 128]), grids=20, dtype=dt16)
    if path == "stats":
        return dict(path=path, rows=_log(rng, 128, 8192), k=rng.choice([1024, 2048, 4096, 5120, 14336]), dtype=dt16)
    if path == "hessian":
        return dict(path=path, rows=_log(rng, 128, 2048), k=rng.choice([512, 1024, 2048, 2816, 4096]), dtype=dt16)
    return dict(path=path, n=_log(rng, 512, 4096, 8), k=rng.choice([1024, 2048, 2816, 4096]), bits=rng.choice([4, 4, 8]),
                symmetric=rng.random() < 0.5, group=rng.choice([0, 64, 128]), dtype=dt16)


# ---- inputs -----------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(g, n, k, dtype, outliers=True):
    """N(0, 0.02), with one entry in a thousand at 20 standard deviations as trained Linear weights have them.  The
    calibration searches get none: there one code on the other side of a rounding boundary is an error of the whole
    step, which an outlier makes larger than the weights around it."""
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    if outliers:
        far = torch.rand(n, k, generator=g, device="cuda") < 0.001
        w = torch.where(far, torch.sign(w) * 0.4, w)
    return w.to(_DTYPES[dtype])


def _activations(g, rows, k, dtype, hot=50.0):
    """Student-t (3 degrees of freedom) values with one channel in 512 scaled up: the outlier channels that SmoothQuant
    and AWQ exist for."""
    x = torch.randn(rows, k, generator=g, device="cuda")
    c = torch.randn(rows, k, generator=g, device="cuda").square_()
    for _ in range(2):
        c += torch.randn(rows, k, generator=g, device="cuda").square_()
    x *= torch.rsqrt(c / 3.0)
    x[:, torch.randint(0, k, (max(1, k // 512),), generator=g, device="cuda")] *= hot
    return x.clamp_(-3e4, 3e4).to(_DTYPES[dtype])


def _wts_cfg(case):
    cfg = {"quant_type": "int%d" % case["bits"], "symmetric": case.get("symmetric", False),
           "strategy": "group" if case["group"] else "channel"}
    if case["group"]:
        cfg["group_size"] = case["group"]
    return {"weights_cfg": cfg}


def _channel_factors(g, k, dtype):
    return torch.exp(0.4 * torch.randn(1, k, generator=g, device="cuda")).to(_DTYPES[dtype])


def prepare(case, seed):
    g = _gen(seed)
    path, dtype = case["path"], case["dtype"]
    if path in ("weight_only", "w8a8"):
        n, k = case["n"], case["k"]
        w = _weight(g, n, k, dtype)
        scale = _channel_factors(g, k, dtype) if case["scaled"] else None
        bias = torch.randn(n, generator=g, device="cuda").to(_DTYPES[dtype]) if case["bias"] else None
        if path == "weight_only":
            quantised, cfg = (w / scale if scale is not None else w), _wts_cfg(case)
            wmin, wmax = get_weight_min_max_by_granularity(quantised, cfg)
            scale_w, offset_w = calculate_scale_offset(wmax, wmin, case["symmetric"], "int%d" % case["bits"])
            layer = HipWeightQuantizedLinear(types.SimpleNamespace(
                weight=torch.nn.Parameter(w, requires_grad=False), wts_type="int%d" % case["bits"],
                group_size=case["group"] or None, scale=scale, scale_w=scale_w, offset_w=offset_w, bias=bias))
            x = torch.randn(case["rows"], k, generator=g, device="cuda").to(_DTYPES[dtype])
        else:
            x = _activations(g, case["rows"], k, dtype, hot=10.0)
            smoothed = w * scale if scale is not None else w
            cfg = {"weights_cfg": {"quant_type": "int8", "symmetric": True, "strategy": "channel"}}
            wmin, wmax = get_weight_min_max_by_granularity(smoothed, cfg)
            scale_w, _ = calculate_scale_offset(wmax, wmin, True, "int8")
            calm = x / scale if scale is not None else x
            scale_d, offset_d = calculate_scale_offset(calm.max().reshape(1).float(), calm.min().reshape(1).float(), False,
                                                       "int8")
            layer = HipQuantizationLinear(types.SimpleNamespace(
                weight=torch.nn.Parameter(w, requires_grad=False), act_type="int8", wts_type="int8", scale_d=scale_d,
                offset_d=offset_d, scale=scale, scale_w=scale_w,
                bias=None if bias is None else torch.nn.Parameter(bias.float(), requires_grad=False)),
                dynamic_act=case["dynamic"])
        return dict(case=case, layer=layer, x=x)
    if path in ("pack", "minmax"):
        return dict(case=case, w=_weight(g, case["n"], case["k"], dtype))
    if path in ("format", "stats"):
        state = dict(case=case, x=_activations(g, case["rows"], case["k"], dtype))
        if path == "stats":      # extrema of the batches before this one
            earlier = _activations(g, 16, case["k"], dtype)
            state["max"], state["min"] = earlier.amax(0, keepdim=True), earlier.amin(0, keepdim=True)
        return state
    if path == "awq":
        layer = torch.nn.Linear(case["k"], case["n"], bias=False, device="cuda", dtype=_DTYPES[dtype])
        layer.weight.requires_grad_(False)
        layer.weight.data = _weight(g, case["n"], case["k"], dtype, outliers=False)
        cfg = _wts_cfg(case)
        cfg["algorithm"] = {"awq": {"grids_num": case["grids"]}}
        return dict(case=case, layer=layer, cfg=cfg, x=_activations(g, case["rows"], case["k"], dtype, hot=10.0).unsqueeze(0))
    if path == "hessian":
        return dict(case=case, batches=[_activations(g, case["rows"], case["k"], dtype, hot=4.0).unsqueeze(0) for _ in range(2)])
    hessian, _ = gptq.update_hessian(None, 0, _activations(g, 2 * case["k"], case["k"], "bf16", hot=4.0).unsqueeze(0), case["k"])
    return dict(case=case, w=_weight(g, case["n"], case["k"], dtype, outliers=False), hessian=hessian, cfg=_wts_cfg(case))


# ---- one pass ---------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    path = case["path"]
    if path in ("weight_only", "w8a8"):
        return state["layer"](state["x"])
    if path == "pack":
        packed, scales, zeros, _ = ops.quant_int4_group_pack(state["w"], case["group"], case["symmetric"])
        return packed, scales, zeros
    if path == "minmax":
        cfg = _wts_cfg(case)
        wmin, wmax = get_weight_min_max_by_granularity(state["w"], cfg)
        scale, offset = calculate_scale_offset(wmax, wmin, case["symmetric"], cfg["weights_cfg"]["quant_type"])
        fake = quant_dequant_weight(state["w"], cfg, scale, offset)
        return (fake, scale) if offset is None else (fake, scale, offset)
    if path == "format":
        x = state["x"]
        if case["fmt"] == "hif8":
            codes = ops.hif8_encode(x)
            return codes, ops.hif8_decode(codes, x.dtype)
        fmt = ops.MX_E4M3 if case["fmt"] == "mxfp8" else ops.MX_E2M1
        elements, exponents = ops.mx_quant(x, fmt)
        return elements, exponents, ops.mx_dequant(elements, exponents, fmt, x.dtype)
    if path == "awq":
        layer = state["layer"]
        scale = awq.search_scale(state["x"], [layer], layer, state["cfg"])
        original = layer.weight.data
        awq.process_weights_for_layers([layer], scale, state["cfg"])
        quantised, layer.weight.data = layer.weight.data, original
        return scale, quantised
    if path == "stats":
        return smooth_quant_stats.update_channel_min_max(state["x"], state["max"], state["min"])
    if path == "hessian":
        hessian, seen = None, 0
        for batch in state["batches"]:
            hessian, seen = gptq.update_hessian(hessian, seen, batch, case["k"])
        return hessian
    weight, scale, offset = gptq.get_opt_weight_and_quant_factor(state["w"], state["hessian"], state["cfg"])
    return (weight, scale) if offset is None else (weight, scale, offset)


# ---- what a pass cannot do without ------------------------------------------------------------------------------
def work(case):
    path, e = case["path"], _SIZE[case["dtype"]]
    n, k, rows = case.get("n", 0), case["k"], case.get("rows", 0)
    if path == "weight_only":
        factors = n * (k // (case["group"] or k)) * (2 if case["bits"] == 8 and case["symmetric"] else 3)
        return dict(bytes=rows * k * e + n * k * case["bits"] // 8 + factors + rows * n * e, flops=2 * rows * n * k)
    if path == "w8a8":
        return dict(bytes=rows * k * e + n * k + 4 * n + rows * n * e, flops=2 * rows * n * k)
    if path == "pack":
        return dict(bytes=n * k * e + n * k // 2 + 3 * n * (k // case["group"]), flops=0)
    if path == "minmax":
        return dict(bytes=2 * n * k * e + 4 * n * (k // (case["group"] or k)) * (1 if case["symmetric"] else 2), flops=0)
    if path == "format":
        values = rows * k
        coded = values // 2 if case["fmt"] == "mxfp4" else values
        coded += 0 if case["fmt"] == "hif8" else values // 32
        return dict(bytes=2 * values * e + 2 * coded, flops=0)
    if path == "awq":
        return dict(bytes=rows * k * e + 2 * n * k * e, flops=2 * rows * n * k * (case["grids"] + 1))
    if path == "stats":
        return dict(bytes=rows * k * e + 4 * k * e, flops=0)
    if path == "hessian":    # one triangle of the symmetric product
        return dict(bytes=2 * rows * k * e + 4 * k * k, flops=2 * rows * k * (k + 1))
    # one factorisation and one triangular inverse (k^3 / 3 each), the update of the columns behind each block
    return dict(bytes=2 * n * k * e + 4 * k * k, flops=2 * k ** 3 // 3 + n * k * k)


def tolerance(case):
    """Whole numbers, bytes and the values that follow from them by one stated rounding are exact.  The others, as
    measured against the same path in 64 bits (the largest of the listed sizes), times four:
      weight_only  2.1e-3 (bf16), 2.5e-4 (fp16): the rounding of the weight and of the output to the model's type
      awq          3e-3: a channel mean one bf16 unit off in a hundredth of the channels moves codes in those columns;
                   a moved code is off by its step, up to about the weights' standard deviation
      hessian      2.5e-7 as it is, 1.5e-6 for the fp32 product of a library
      gptq         3.7e-3: 1e-4 of the codes sit on the other side of a rounding boundary, by one step or two"""
    path = case["path"]
    if path == "weight_only":
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}
    if path == "awq":
        return {"rel": 0.012, "max": 0.99}
    if path == "hessian":
        return {"rel": 4e-6}
    if path == "gptq":
        return {"rel": 0.015, "max": 0.99}
    return "exact"
