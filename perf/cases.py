"""The work a program that uses this framework has it do, as cases that can be timed.

A case is a dict of plain values; its ``kind`` names one of the framework's uses:

* ``linear``       ``TernaryLinearInference.forward``: a deployed layer on ``rows`` activation rows (decode, prompt
                   chunks, prefill), float arithmetic;
* ``tensor_core``  ``ops.ternary_linear_tensor_core_forward(version=2)``: per-row int8 activations times packed weights,
                   the functional entry point;
* ``mlp``          ``TernarySwiGLU``: RMSNorm, fused gate|up, SwiGLU, down, residual, in float or int8 arithmetic;
* ``grouped``      ``ops.ternary_linear_grouped`` / ``ops.ternary_linear_int8_grouped``: one decode step through ``units``
                   same-shaped layers;
* ``train``        ``TernaryLinear`` forward and backward: a training step's share of one layer;
* ``convert``      ``create_ternary_linear_inference``: quantize and pack full-precision weights for deployment.
"""

import math

import torch

from bittorch_amd import nn, ops

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}


def listed():
    return [
        # One decoded token through one layer: the smallest call, launch and host latency.
        dict(name="decode_row", kind="linear", rows=1, n=4096, k=4096, dtype="fp16", bias=True, residual=False),
        # One decoded token through the MLP of a block of the 2B-parameter stack.
        dict(name="decode_mlp", kind="mlp", rows=1, d=2560, ffn=6912, dtype="bf16", compute="float"),
        # A batched decode step (16 sequences) through an up projection, int8 activations.
        dict(name="decode_batch_int8", kind="tensor_core", rows=16, n=11008, k=4096, dtype="bf16", bias=False),
        # A short prompt through the fused q|k|v projection, with a row count that fills no tile.
        dict(name="prompt_chunk", kind="linear", rows=77, n=7680, k=2560, dtype="bf16", bias=False, residual=False),
        # Decode rows of many sequences through as many layers of one shape, one launch.
        dict(name="grouped_decode", kind="grouped", units=128, rows=1, n=4096, k=4096, dtype="fp16", int8=False),
        # A prefill of 2048 tokens through an up projection on the int8 matrix cores.
        dict(name="prefill_int8", kind="tensor_core", rows=2048, n=11008, k=4096, dtype="bf16", bias=False),
        # The MLP of a block of the 2B-parameter stack over 8 x 512 tokens, int8 arithmetic.
        dict(name="prefill_mlp_int8", kind="mlp", rows=4096, d=2560, ffn=6912, dtype="bf16", compute="int8"),
        # The same MLP in float arithmetic on a prompt of a thousand tokens.
        dict(name="prefill_mlp_float", kind="mlp", rows=1000, d=2560, ffn=6912, dtype="bf16", compute="float"),
        # A small network's layer in training: the plumbing configuration, all launches.
        dict(name="train_small", kind="train", rows=32, n=256, k=512, mode="fp32", bias=True),
        # Training in the layers' default dtype on many short rows.
        dict(name="train_fp32", kind="train", rows=16384, n=768, k=768, mode="fp32", bias=True),
        # Mixed-precision training of a large layer: fp32 masters under autocast.
        dict(name="train_amp", kind="train", rows=4096, n=11008, k=4096, mode="amp", bias=False),
        # A trained layer converted for deployment.
        dict(name="convert", kind="convert", n=11008, k=4096, dtype="fp32", bias=True),
    ]


# ---- draws -----------------------------------------------------------------------------------------------------------

_MAX_FLOPS = 1.1e12    # of a 16-bit or int8 case: train_amp's
_MAX_FLOPS_FP32 = 1.4e11
_MAX_BYTES = 5.4e8     # grouped_decode's


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi, odd=True):
    """A layer dimension: mostly a multiple of 256 or of 16 as layers have them, now and then any number."""
    v = _log_uniform(rng, lo, hi)
    step = rng.choice((256, 256, 64, 16, 1) if odd else (256, 256, 64, 16))
    return max(lo, v // step * step)


def _draw(rng):
    kind = rng.choice(("linear", "linear", "tensor_core", "tensor_core", "mlp", "mlp", "grouped", "train", "train", "convert"))
    if kind == "linear":
        return dict(kind=kind, rows=rng.choice((1, _log_uniform(rng, 1, 64), _log_uniform(rng, 1, 4096))),
                    n=_features(rng, 256, 16384), k=_features(rng, 256, 16384), dtype=rng.choice(("fp16", "bf16", "bf16", "fp32")),
                    bias=rng.random() < 0.5, residual=rng.random() < 0.25)
    if kind == "tensor_core":
        return dict(kind=kind, rows=rng.choice((_log_uniform(rng, 1, 64), _log_uniform(rng, 64, 4096))), n=_features(rng, 256, 16384),
                    k=_features(rng, 256, 16384), dtype=rng.choice(("fp16", "bf16", "bf16", "fp32")), bias=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind=kind, rows=rng.choice((1, _log_uniform(rng, 2, 64), _log_uniform(rng, 64, 4096))), d=_features(rng, 512, 5120, False),
                    ffn=_features(rng, 1024, 14336, False), dtype=rng.choice(("fp16", "bf16", "bf16")), compute=rng.choice(("float", "int8")))
    if kind == "grouped":
        int8 = rng.random() < 0.5
        return dict(kind=kind, units=_log_uniform(rng, 3, 128), rows=rng.randint(1, 16) if int8 else 1, n=_features(rng, 1024, 11008, False),
                    k=_features(rng, 1024, 11008, False), dtype=rng.choice(("fp16", "bf16")), int8=int8)
    if kind == "train":
        return dict(kind=kind, rows=_log_uniform(rng, 16, 16384), n=_features(rng, 128, 11008), k=_features(rng, 128, 11008),
                    mode=rng.choice(("fp32", "amp", "bf16")), bias=rng.random() < 0.5)
    return dict(kind=kind, n=_features(rng, 256, 16384), k=_features(rng, 256, 16384), dtype=rng.choice(("fp32", "fp32", "bf16", "fp16")),
                bias=rng.random() < 0.5)


def draw(rng):
    while True:
        case = _draw(rng)
        cost = work(case)
        fp32 = case.get("mode", case.get("dtype")) == "fp32" and case["kind"] in ("train", "linear")
        if cost["bytes"] <= _MAX_BYTES and cost["flops"] <= (_MAX_FLOPS_FP32 if fp32 else _MAX_FLOPS):
            return case


# ---- what a program holds before the call ----------------------------------------------------------------------------

def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(seed * 7919 + 17)


def _normal(g, shape, std, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=g.device).mul_(std).to(dtype)


def _activations(g, shape, dtype):
    """N(0, 1) with a thousandth of the entries twenty times as large, as hidden states have them."""
    x = torch.randn(shape, generator=g, device=g.device)
    x = torch.where(torch.rand(shape, generator=g, device=g.device) < 1e-3, x * 20, x)
    return x.to(dtype)


def _layer(g, n, k, bias):
    """A deployed layer from N(0, 0.02) masters, its weights laid out once as a server does at load time."""
    w = _normal(g, (n, k), 0.02)
    b = _normal(g, (n,), 0.01) if bias else None
    return nn.create_ternary_linear_inference(k, n, w, b)


def prepare(case, seed):
    g = _generator(seed, "cuda")
    kind = case["kind"]
    if kind == "linear":
        dt = _DTYPES[case["dtype"]]
        layer = _layer(g, case["n"], case["k"], case["bias"]).prepare_decode()
        x = _normal(g, (case["rows"], case["k"]), 1.0, dt)
        res = _normal(g, (case["rows"], case["n"]), 1.0, dt) if case["residual"] else None
        return dict(kind=kind, layer=layer, x=x, residual=res)
    if kind == "tensor_core":
        layer = _layer(g, case["n"], case["k"], case["bias"])
        return dict(kind=kind, w=layer.weight_packed, scale=layer.scale, bias=layer.bias, k=case["k"],
                    x=_activations(g, (case["rows"], case["k"]), _DTYPES[case["dtype"]]))
    if kind == "mlp":
        d, ffn, dt = case["d"], case["ffn"], _DTYPES[case["dtype"]]
        mlp = nn.TernarySwiGLU(_layer(g, ffn, d, False), _layer(g, ffn, d, False), _layer(g, d, ffn, False),
                               compute=case["compute"], fuse_gate_up=True)
        mlp.gate_up.prepare_decode()
        mlp.down.prepare_decode()
        return dict(kind=kind, mlp=mlp, x=_normal(g, (case["rows"], d), 1.0, dt), norm=(1 + _normal(g, (d,), 0.1)).to(dt))
    if kind == "grouped":
        dt = _DTYPES[case["dtype"]]
        layers = [_layer(g, case["n"], case["k"], True).prepare_decode() for _ in range(case["units"])]
        shape = (case["units"], case["rows"], case["k"]) if case["int8"] else (case["units"], case["k"])
        return dict(kind="grouped_int8" if case["int8"] else kind, layers=layers, x=_normal(g, shape, 1.0, dt))
    if kind == "train":
        layer = nn.TernaryLinear(case["k"], case["n"], bias=case["bias"]).to("cuda")
        act = torch.float16 if case["mode"] == "amp" else _DTYPES[case["mode"]]
        with torch.no_grad():
            layer.weight.copy_(_normal(g, (case["n"], case["k"]), 0.02))
            if case["bias"]:
                layer.bias.copy_(_normal(g, (case["n"],), 0.01))
        if case["mode"] == "bf16":
            layer = layer.to(torch.bfloat16)
        return dict(kind=kind, layer=layer, amp=case["mode"] == "amp", x=_normal(g, (case["rows"], case["k"]), 1.0, act).requires_grad_(),
                    grad=_normal(g, (case["rows"], case["n"]), 0.01, act))
    dt = _DTYPES[case["dtype"]]
    return dict(kind=kind, n=case["n"], k=case["k"], w=_normal(g, (case["n"], case["k"]), 0.02, dt),
                bias=_normal(g, (case["n"],), 0.01, dt) if case["bias"] else None)


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"], state["residual"])
    if kind == "tensor_core":
        return ops.ternary_linear_tensor_core_forward(state["x"], state["w"], state["scale"], state["k"], state["bias"], version=2)
    if kind == "mlp":
        return state["mlp"](state["x"], state["norm"], 1e-5, state["x"])
    if kind == "grouped":
        return ops.ternary_linear_grouped(state["layers"], state["x"])
    if kind == "grouped_int8":
        return ops.ternary_linear_int8_grouped(state["layers"], state["x"])
    if kind == "train":
        layer, x = state["layer"], state["x"]
        x.grad = layer.weight.grad = None
        if layer.bias is not None:
            layer.bias.grad = None
        if state["amp"]:
            with torch.autocast("cuda", dtype=torch.float16):
                y = layer(x)
        else:
            y = layer(x)
        y.backward(state["grad"])
        return y.detach(), x.grad, layer.weight.grad, None if layer.bias is None else layer.bias.grad
    layer = nn.create_ternary_linear_inference(state["k"], state["n"], state["w"], state["bias"])
    return layer.weight_packed, layer.scale, layer.bias


# ---- what a pass cannot do without, and how far another correct one may be off ---------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "mlp":
        rows, d, ffn = case["rows"], case["d"], case["ffn"]
        return {"bytes": 3 * d * ffn // 4 + 4 * (2 * ffn + d) + 2 * d + 2 * 2 * rows * d, "flops": 6.0 * rows * d * ffn}
    n, k = case["n"], case["k"]
    if kind == "convert":
        size = _SIZE[case["dtype"]]
        return {"bytes": size * n * k + n * k // 4 + size * n, "flops": 0.0}
    rows = case["rows"]
    if kind == "grouped":
        return {"bytes": case["units"] * (n * k // 4 + 8 * n + 2 * rows * (n + k)), "flops": 2.0 * case["units"] * rows * n * k}
    if kind == "train":
        act = 4 if case["mode"] == "fp32" else 2
        master = 2 if case["mode"] == "bf16" else 4
        return {"bytes": 2 * master * n * k + act * rows * (2 * n + 2 * k), "flops": 6.0 * rows * n * k}
    size = _SIZE[case["dtype"]]
    extra = size * rows * n if case.get("residual") else 0
    return {"bytes": n * k // 4 + 8 * n + size * rows * (n + k) + extra, "flops": 2.0 * rows * n * k}


def tolerance(case):
    """Four times what the path's outputs differ from the same path in 64 bits: the rounding of the outputs' data type,
    and of the sums in fp32.  Packed weights and their scales are the same bytes."""
    kind = case["kind"]
    if kind == "convert":
        return "exact"
    dt = {"amp": "fp16"}.get(case.get("mode"), case.get("mode", case.get("dtype")))
    rel = {"fp32": 1e-5, "fp16": 1.2e-3, "bf16": 7e-3}[dt]
    if kind == "mlp":  # three layers, each reading rounded values
        rel *= 3
    return {"rel": rel}
