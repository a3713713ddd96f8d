"""The workloads this framework is timed on: quantized linears, RoPE, quantize and dequantize
as a diffusion transformer's forward pass calls them, from one conditioning row to 8192 tokens.

A case is a dict of plain values with a "kind":
  linear   a bf16 / f16 activation is quantized by its layout (`QuantizedTensor.from_float`) and
           goes through `F.linear` with quantized weights and a bias, once for each of `layers`
           weights of the same size (the layers of several blocks that read one input)
  rope     `ck.apply_rope` on q, k (or `ck.apply_rope1` on x) of `layers` blocks
  decode   `ck.dequantize_*` of the weights of `layers` layers to 16 bits
  encode   `ck.quantize_per_tensor_fp8` and `ck.dequantize_per_tensor_fp8` of one tensor
With "graph" true the program has captured its calls in a HIP graph and a pass replays it, as a
sampler does with a launch-bound step; else a pass makes the calls.
"""
from __future__ import annotations

import sys
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "comfy-kitchen_amd"))

LAYOUTS = {"fp8": "TensorCoreFP8Layout", "mxfp8": "TensorCoreMXFP8Layout", "nvfp4": "TensorCoreNVFP4Layout"}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _linear(name, layout, m, n, k, layers, graph, dtype="bf16"):
    return {"name": name, "kind": "linear", "layout": layout, "m": m, "n": n, "k": k, "layers": layers,
            "graph": graph, "dtype": dtype}


def listed():
    return [
        # smallest call: a short text embedding stored as FP8 and read back
        {"name": "encode_small_fp8", "kind": "encode", "rows": 77, "cols": 4096, "dtype": "bf16"},
        # one modulation linear on one conditioning row, called from Python
        _linear("modulation_call_mxfp8", "mxfp8", 1, 18432, 3072, 1, False),
        # the modulation linears of several blocks on one conditioning row, in a captured step
        _linear("modulation_step_mxfp8", "mxfp8", 1, 18432, 3072, 6, True),
        # the same with four rows (a batch of conditionings) and FP4 weights
        _linear("modulation_step_nvfp4", "nvfp4", 4, 18432, 3072, 6, True),
        # text stream: the qkv linears of 256 text tokens
        _linear("text_qkv_fp8", "fp8", 256, 9216, 3072, 4, True),
        # cross-attention: key and value projections of a 512-token context in several blocks
        _linear("context_kv_mxfp8", "mxfp8", 512, 5120, 5120, 6, True),
        # a wide feed-forward on 256 tokens, FP4 weights
        _linear("text_ffn_nvfp4", "nvfp4", 256, 13824, 5120, 4, True),
        # a small image with an odd number of tokens, f16 activations
        _linear("image_mlp_mxfp8", "mxfp8", 1333, 12288, 3072, 2, True, "f16"),
        # a full-size image: the MLP's up-projection
        _linear("mlp_up_mxfp8", "mxfp8", 4608, 12288, 3072, 1, False),
        # a video's feed-forward: the largest call
        _linear("ffn_up_nvfp4", "nvfp4", 8192, 13824, 5120, 1, False),
        # q and k of several blocks of a full-size image
        {"name": "rope_image", "kind": "rope", "batch": 1, "heads": 24, "seq": 4608, "dim": 128, "pair": True,
         "layers": 4, "graph": True, "dtype": "bf16"},
        # FP4 weights decoded to 16 bits (merging, or a layer run unquantized)
        {"name": "decode_weight_nvfp4", "kind": "decode", "layout": "nvfp4", "rows": 13824, "cols": 5120,
         "layers": 4, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["rope", "decode", "encode"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "linear":
        layout = rng.choice(["fp8", "mxfp8", "nvfp4"])
        m = _log_int(rng, 1, 8192)
        n = 8 * _log_int(rng, 128, 2304)    # 1024 .. 18432
        k = 32 * _log_int(rng, 32, 432)     # 1024 .. 13824
        while m * n * k > 8192 * 13824 * 5120:
            m = max(1, m // 2)
        layers = max(1, min(6, 2 ** 36 // (max(m, 256) * n * k)))
        return {"kind": kind, "layout": layout, "m": m, "n": n, "k": k, "layers": layers,
                "graph": layers > 1, "dtype": dtype}
    if kind == "rope":
        heads, dim = rng.choice([8, 12, 24, 40]), rng.choice([64, 96, 128])
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "heads": heads, "seq": _log_int(rng, 64, 8192),
                "dim": dim, "pair": rng.random() < 0.7, "layers": 4, "graph": True, "dtype": dtype}
    if kind == "decode":
        return {"kind": kind, "layout": rng.choice(["fp8", "mxfp8", "nvfp4"]), "rows": 16 * _log_int(rng, 16, 1152),
                "cols": 64 * _log_int(rng, 8, 216), "layers": 4, "dtype": dtype}
    return {"kind": kind, "rows": _log_int(rng, 16, 8192), "cols": 8 * _log_int(rng, 64, 768), "dtype": dtype}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activation(g, rows, cols, dtype):
    """Normal values whose magnitude varies log-normally from row to row."""
    x = torch.randn(rows, cols, generator=g, device="cuda")
    return (x * torch.exp(0.5 * torch.randn(rows, 1, generator=g, device="cuda"))).to(DTYPES[dtype])


def _weight(g, n, k, dtype):
    return (0.02 * torch.randn(n, k, generator=g, device="cuda")).to(DTYPES[dtype])


def _inputs(case, seed):
    """The plain tensors of a case: what exact() works on and prepare() quantizes."""
    g = _gen(seed)
    kind, dt = case["kind"], case["dtype"]
    if kind == "linear":
        return {"x": _activation(g, case["m"], case["k"], dt),
                "w": [_weight(g, case["n"], case["k"], dt) for _ in range(case["layers"])],
                "bias": [torch.randn(case["n"], generator=g, device="cuda").to(DTYPES[dt])
                         for _ in range(case["layers"])]}
    if kind == "rope":
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        x = [torch.randn(shape, generator=g, device="cuda").to(DTYPES[dt])
             for _ in range(case["layers"] * (2 if case["pair"] else 1))]
        theta = 1.0 / 10000.0 ** (torch.arange(0, case["dim"], 2, device="cuda", dtype=torch.float64) / case["dim"])
        start = 64.0 * torch.rand((), generator=g, device="cuda", dtype=torch.float64)
        phi = (start + torch.arange(case["seq"], device="cuda", dtype=torch.float64))[:, None] * theta
        f = torch.stack([phi.cos(), -phi.sin(), phi.sin(), phi.cos()], -1)
        return {"x": x, "freqs": f.float().reshape(1, 1, case["seq"], case["dim"] // 2, 2, 2)}
    if kind == "decode":
        return {"w": [_weight(g, case["rows"], case["cols"], dt) for _ in range(case["layers"])]}
    return {"x": _activation(g, case["rows"], case["cols"], dt)}


def _capture(calls):
    """(graph, outputs) of calls() captured after a warm-up on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = calls()
    return graph, out


def prepare(case, seed):
    import comfy_kitchen as ck
    from comfy_kitchen.tensor import QuantizedTensor

    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        layout, x, bias = LAYOUTS[case["layout"]], t["x"], t["bias"]
        w = [QuantizedTensor.from_float(v, layout) for v in t["w"]]

        def calls():
            return [F.linear(QuantizedTensor.from_float(x, layout), wl, bl) for wl, bl in zip(w, bias)]
    elif kind == "rope":
        x, f = t["x"], t["freqs"]

        def calls():
            if case["pair"]:
                return [ck.apply_rope(x[i], x[i + 1], f) for i in range(0, len(x), 2)]
            return [ck.apply_rope1(v, f) for v in x]
    elif kind == "decode":
        out = DTYPES[case["dtype"]]
        w = [QuantizedTensor.from_float(v, LAYOUTS[case["layout"]]) for v in t["w"]]

        def calls():
            if case["layout"] == "fp8":
                return [ck.dequantize_per_tensor_fp8(v._qdata, v.params.scale, out) for v in w]
            if case["layout"] == "mxfp8":
                return [ck.dequantize_mxfp8(v._qdata, v.params.scale, out) for v in w]
            return [ck.dequantize_nvfp4(v._qdata, v.params.scale, v.params.block_scale, out) for v in w]
    else:
        x, out = t["x"], DTYPES[case["dtype"]]
        scale = (x.abs().amax().float() / 448.0).reshape(1)

        def calls():
            q = ck.quantize_per_tensor_fp8(x, scale)
            return [q, ck.dequantize_per_tensor_fp8(q, scale, out)]
    if not case.get("graph"):
        return {"calls": calls}
    graph, out = _capture(calls)
    return {"calls": calls, "graph": graph, "out": out}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["calls"]()


# ------------------------------------------------------------------ bounds
def _code_bytes(layout, rows, cols):
    """Bytes of a quantized [rows, cols] tensor: codes and block scales."""
    return rows * cols * {"fp8": 1.0, "mxfp8": 1.0 + 1 / 32, "nvfp4": 0.5 + 1 / 16}[layout]


def work(case):
    kind, layers = case["kind"], case.get("layers", 1)
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * m * k + layers * (_code_bytes(case["layout"], n, k) + 2 * n + 2 * m * n),
                "flops": 2 * layers * m * n * k}
    if kind == "rope":
        x = case["batch"] * case["heads"] * case["seq"] * case["dim"] * layers * (2 if case["pair"] else 1)
        return {"bytes": 4 * x + 8 * case["seq"] * case["dim"], "flops": 3 * x}
    n = case["rows"] * case["cols"]
    if kind == "decode":
        return {"bytes": layers * (_code_bytes(case["layout"], case["rows"], case["cols"]) + 2 * n), "flops": layers * n}
    return {"bytes": 6 * n, "flops": 2 * n}


def tolerance(case):
    # codes and decoded values are defined to the bit; linears and rotations end in one
    # rounding to 16 bits (relative 2-norm against 64 bits: 1.7e-3 in bf16, 2.1e-4 in f16)
    if case["kind"] in ("encode", "decode"):
        return "exact"
    return {"rel": 7e-3 if case["dtype"] == "bf16" else 9e-4}


# ------------------------------------------------- the same results in 64 bits
def _amax_scale(x, limit):
    """amax(|x|) / limit as torch divides a GPU tensor by a number: times the 32-bit reciprocal,
    rounded to x's type."""
    inv = torch.tensor(1.0) / torch.tensor(limit)
    return (x.abs().amax().float() * inv.to(x.device)).to(x.dtype).float()


def _rounded(x, layout):
    """x after quantization, as 64-bit values (the exact values its codes and scales stand for)."""
    if layout == "fp8":
        s = _amax_scale(x, 448.0)
        q = (x * (1.0 / s).to(x.dtype)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return q.double() * s.double()
    if layout == "mxfp8":
        b = x.float().reshape(x.shape[0], -1, 32)
        mant, e = torch.frexp((b.abs().amax(-1, keepdim=True) / 448.0).double())
        s = torch.ldexp(torch.ones_like(mant), e - (mant == 0.5).to(e.dtype))
        q = (b.double() / s).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn)
        return (q.double() * s).reshape(x.shape)
    g = _amax_scale(x, 448.0 * 6.0)
    b = x.float().reshape(x.shape[0], -1, 16)
    s = (b.abs().amax(-1, keepdim=True) / 6.0 / g).clamp(max=448.0).to(torch.float8_e4m3fn).float()
    total = g * s
    v = (b / torch.where(total == 0, torch.ones_like(total), total)).clamp(-6.0, 6.0)
    a = v.abs()
    mag = torch.zeros_like(a)
    for limit, even, value in ((0.25, False, 0.5), (0.75, True, 1.0), (1.25, False, 1.5), (1.75, True, 2.0),
                               (2.5, False, 3.0), (3.5, True, 4.0), (5.0, False, 6.0)):
        mag = torch.where((a >= limit) if even else (a > limit), torch.full_like(a, value), mag)
    return (torch.copysign(mag, v).double() * s.double() * g.double()).reshape(x.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return None
    t = _inputs(case, seed)
    if kind == "linear":
        x = _rounded(t["x"], case["layout"])
        return [x @ _rounded(w, case["layout"]).t() + b.double() for w, b in zip(t["w"], t["bias"])]
    if kind == "decode":
        return [_rounded(w, case["layout"]) for w in t["w"]]
    f = t["freqs"].double()
    out = []
    for x in t["x"]:
        v = x.double().reshape(*x.shape[:-1], -1, 1, 2)
        out.append((f[..., 0] * v[..., 0] + f[..., 1] * v[..., 1]).reshape(x.shape))
    return [(out[i], out[i + 1]) for i in range(0, len(out), 2)] if case["pair"] else out
