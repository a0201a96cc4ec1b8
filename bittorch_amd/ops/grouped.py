"""``ternary_linear_grouped`` / ``ternary_linear_int8_grouped``: G decode-shape products of same-shaped inference
layers in ONE kernel launch.

No counterpart in ``bittorch.ops``: the reference's packed kernel serves one matrix per launch
(``csrc/kernels/ternary_gemm_production.cu:286-362``, called from ``bittorch/nn/ternary_linear_infer.py:78-104``).  A
4 MiB weight matrix streams in less time than a kernel takes to start and drain, so a decode step that has several
independent GEMVs of one shape -- q, k and v of a block kept as separate layers, the same projection of several
models or adapters, one row per user times per-user layers -- pays that start once for all of them here
(``bt_ternary_gemv_grouped``).  Every unit's output equals ``layer(x_row)`` bit for bit for fp16 rows; bf16 rows are
summed exactly (each row scaled by its own largest exponent) and agree with the single call's fp32 sums to their
rounding.  Whatever the grouped kernel does not take (CPU tensors, fp32 rows, K % 16 != 0, layers without a natural
tiled copy) runs as single calls, same results as ``layer(x)``.

``ternary_linear_int8_grouped`` is the same for the int8 path with up to 16 rows per layer (a batched decode step;
``bt_ternary_gemm_i8_grouped``): per-row int8 activations, int32 accumulators on the matrix cores, every unit equal to
``layer.forward_int8`` on its rows bit for bit.
"""

from __future__ import annotations

import os
from collections import OrderedDict
from operator import attrgetter, itemgetter
from typing import List, Optional, Sequence, Union

import torch
from torch import Tensor

_MAX_K = 16384     # the grouped kernel keeps a row's digit planes in LDS
_PLANS: "OrderedDict[tuple, _Plan]" = OrderedDict()
_MAX_PLANS = 16
# Tables that captured graphs read (a few kilobytes each): a graph's launches hold their addresses alone, and how long it lives
# is not known here.  One entry for each set of layers and buffers that has been captured.
_CAPTURED: dict = {}


class _Plan:
    """Pointer tables of one set of layers (device arrays of G addresses), rebuilt when a layer's buffers move."""

    def __init__(self, layers):
        from .. import _C
        # (scales and biases go to the kernel in their own dtype, as the single call hands them over: same bits)
        self.tiled = [L.tiled_weights() for L in layers]       # keeps the copies alive
        self.scales = [L.scale.contiguous() for L in layers]
        self.biases = None if layers[0].bias is None else [L.bias.contiguous() for L in layers]
        self.held = [(L.scale, L.bias) for L in layers]        # (no other tensor takes their place in the key meanwhile)
        self.key = _fingerprint(layers)
        self.w_tab = _C.pointer_table(self.tiled)
        self.s_tab = _C.pointer_table(self.scales)
        self.b_tab = None if self.biases is None else _C.pointer_table(self.biases)
        self.own = [t for t in (self.w_tab, self.s_tab, self.b_tab) if t is not None]
        self.own += [v for v, L in zip(self.scales, layers) if v is not L.scale]
        self.own += [v for v, L in zip(self.biases or (), layers) if v is not L.bias]
        self.streams = {torch.cuda.current_stream(self.w_tab.device).cuda_stream}
        self.io_tabs: "OrderedDict[tuple, tuple]" = OrderedDict()
        self.i8_tabs: "OrderedDict[tuple, tuple]" = OrderedDict()

    def io_tab(self, x: Tensor, y: Tensor, shared_x: bool):
        """Tables of the G row addresses of x [G, K] (or of one shared row) and y [G, N]."""
        return self._tables(self.io_tabs, y.shape[0], y.device, ((x.data_ptr(), 0 if shared_x else _unit_bytes(x)),
                                                                 (y.data_ptr(), _unit_bytes(y))))

    def i8_tab(self, q: Tensor, s_x: Tensor, y: Tensor):
        """Tables of the G units' addresses inside q [G, M, K], s_x [G, M] and y [G, M, N]."""
        return self._tables(self.i8_tabs, q.shape[0], q.device, tuple((t.data_ptr(), _unit_bytes(t)) for t in (q, s_x, y)))

    def _tables(self, held, g: int, device, key):
        """One table of G addresses for each (first address, bytes from one unit to the next) of ``key``; kept by the whole
        key (the same buffers may hold units of another size on the next call), so a decode loop whose buffers repeat (and
        a captured graph, whose buffers are fixed) builds them once."""
        entry = held.get(key)
        if entry is None:
            tabs = tuple(torch.tensor([base + u * step for u in range(g)], dtype=torch.int64, device=device) for base, step in key)
            entry = held[key] = (tabs, set())
            if len(held) > 8:
                held.popitem(last=False)
        else:
            try:
                held.move_to_end(key)
            except KeyError:  # (another host thread has just dropped it)
                pass
        if device.type == "cuda":
            stream = torch.cuda.current_stream(device)
            self._read_on(stream, entry[0], entry[1])
            self._read_on(stream, self.own, self.streams)
            if torch.cuda.is_current_stream_capturing():
                self._keep_for_graph(key, entry[0])
        return entry[0]

    @staticmethod
    def _read_on(stream, tables, streams) -> None:
        """Once for each stream: memory that this object drops is handed out again behind what that stream reads of it."""
        if stream.cuda_stream not in streams:
            streams.add(stream.cuda_stream)
            for t in tables:
                t.record_stream(stream)

    def _keep_for_graph(self, key, tabs) -> None:
        _CAPTURED[(self.w_tab.data_ptr(), key)] = (tabs, self.own)


def _unit_bytes(t: Tensor) -> int:
    return t.stride(0) * t.element_size()


_data_ptr, _numel, _is_contiguous = Tensor.data_ptr, Tensor.numel, Tensor.is_contiguous
_own_dict = attrgetter("__dict__")
_settings = itemgetter("_buffers", "_tiled", "in_features", "out_features", "decode_tiled", "_tile_order")
_vectors = itemgetter("scale", "bias")


def _fingerprint(layers):
    """Everything about the layers that the checks below and a plan's tables depend on, read past ``nn.Module``'s
    attribute lookup and one property of all layers at a time (with 128 layers the checks one by one took 1.2 ms of host
    time around a kernel of 87 us, this takes about as long as the kernel).  Tensors count as themselves, which fixes
    dtype and device (a plan keeps them alive); scales and biases may still be pointed elsewhere or shortened.  What is
    written into one is read where it lies, except where the tables hold a contiguous copy of it."""
    buffers, tiled, *settings = zip(*map(_settings, map(_own_dict, layers)))
    try:
        scales, biases = zip(*map(_vectors, buffers))
    except KeyError:  # (made Parameters)
        scales, biases = [L.scale for L in layers], [L.bias for L in layers]
    vectors = [*scales, *(b for b in biases if b is not None)]
    contiguous = list(map(_is_contiguous, vectors))
    return [list(map(type, layers)), settings, list(map(id, tiled)),
            # (weight_packed held beside the tiled copy: written or replaced, the copy is made again)
            [(i, w.data_ptr(), w._version) for i, b in enumerate(buffers) if (w := b.get("weight_packed")) is not None],
            list(map(id, vectors)), list(map(_data_ptr, vectors)), list(map(_numel, vectors)),
            contiguous if all(contiguous) else [(v.stride(), v._version) for v in vectors]]


def _known_plan(layers) -> Optional[_Plan]:
    """The plan of exactly these layers if nothing about them has changed since it was made (the layers then passed every
    check), or None."""
    try:
        ident = tuple(map(id, layers))
        plan = _PLANS.get(ident)
        if plan is None or plan.key != _fingerprint(layers):
            return None
        _PLANS.move_to_end(ident)
        return plan
    except (KeyError, AttributeError):  # (not an inference layer: the checks say so)
        return None


def _plan_for(layers) -> _Plan:
    plan = _known_plan(layers)
    if plan is not None:
        return plan
    plan = _Plan(layers)
    _PLANS[tuple(map(id, layers))] = plan
    if len(_PLANS) > _MAX_PLANS:
        _PLANS.popitem(last=False)
    return plan


def _check_layers(who: str, layers) -> None:
    from ..nn.ternary_linear_infer import TernaryLinearInference
    for L in layers:
        if not isinstance(L, TernaryLinearInference):
            raise TypeError(f"{who} takes TernaryLinearInference layers")
    k, n = layers[0].in_features, layers[0].out_features
    for L in layers:
        if (L.in_features, L.out_features) != (k, n):
            raise ValueError(f"{who}: every layer must have the same in_features and out_features")
        if (L.bias is None) != (layers[0].bias is None) or L.scale.numel() != layers[0].scale.numel():
            raise ValueError(f"{who}: layers must agree on having a bias and on the scale's length")


def _groupable(layers, x: Tensor) -> bool:
    L0 = layers[0]
    if not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16):
        return False
    if L0.in_features % 16 != 0 or L0.in_features > _MAX_K:
        return False
    kinds = (torch.float32, torch.float16, torch.bfloat16)
    for L in layers:
        if not (L.decode_tiled and L.tile_order == "natural" and L.scale.is_cuda):
            return False
        if L.scale.dtype != L0.scale.dtype or L.scale.dtype not in kinds:
            return False
        if L.bias is not None and (L.bias.dtype != L0.bias.dtype or L.bias.dtype not in kinds):
            return False
        if not L._tiled_fresh() and torch.cuda.is_current_stream_capturing():
            return False  # (a capture never builds the tiled copy)
    return _kernels_allowed()


def _kernels_allowed() -> bool:
    return os.environ.get("BITTORCH_KERNEL", "auto") != "generic"


def ternary_linear_grouped(layers: Sequence, xs: Union[Tensor, Sequence[Tensor]], out: Optional[Tensor] = None) -> Tensor:
    """``Y[u] = layers[u](xs[u])`` for ``G`` :class:`~bittorch_amd.nn.TernaryLinearInference` layers of one shape,
    one activation row each, in one launch.

    ``xs``: ``[G, K]`` (row ``u`` goes to layer ``u``), a single row ``[K]`` / ``[1, K]`` shared by every layer, or a
    sequence of ``G`` rows.  Returns ``[G, N]`` in the rows' dtype (written into ``out`` if given)."""
    layers = list(layers)
    if not layers:
        raise ValueError("ternary_linear_grouped: no layers")
    plan = _known_plan(layers)
    if plan is None:
        _check_layers("ternary_linear_grouped", layers)
    g, k, n = len(layers), layers[0].in_features, layers[0].out_features
    if not isinstance(xs, Tensor):
        xs = torch.stack([t.reshape(-1) for t in xs])
    shared = xs.numel() == k
    if shared:
        x = xs.reshape(1, k)
    else:
        if xs.dim() != 2 or xs.shape != (g, k):
            raise RuntimeError(f"input K doesn't match in_features: expected [{g}, {k}] or one row of {k}, got {tuple(xs.shape)}")
        x = xs
    if plan is not None and not (x.is_cuda and x.dtype in (torch.float16, torch.bfloat16) and _kernels_allowed()):
        plan = None  # (a call the grouped kernel does not take)
    if plan is None and any(L.scale.is_cuda != x.is_cuda for L in layers):
        raise RuntimeError("All tensors must be CUDA")
    if out is not None and (out.shape != (g, n) or out.dtype != x.dtype or out.device != x.device or out.stride(1) != 1):
        raise ValueError("ternary_linear_grouped: out must be [G, N] in the rows' dtype on their device, rows contiguous")
    if plan is None and not _groupable(layers, x):
        ys = [L(x if shared else x[u:u + 1]) for u, L in enumerate(layers)]
        y = torch.cat(ys, dim=0)
        return y if out is None else out.copy_(y)
    from .. import _C
    if x.stride(-1) != 1 or (x.data_ptr() % 16) or (not shared and (x.stride(0) * x.element_size()) % 16):
        x = x.contiguous()
    plan = plan or _plan_for(layers)
    y = out if out is not None else torch.empty((g, n), dtype=x.dtype, device=x.device)
    xt, yt = plan.io_tab(x, y, shared)
    _C.ternary_gemv_grouped(xt, plan.w_tab, plan.s_tab, plan.b_tab, yt, k, n,
                            scale_len=layers[0].scale.numel(), scale_dtype=layers[0].scale.dtype,
                            bias_dtype=torch.float32 if layers[0].bias is None else layers[0].bias.dtype,
                            x_dtype=x.dtype)
    return y


_MAX_K_I8 = 11264  # the grouped int8 kernel holds a wave's K slice of the 16 rows in registers
_MIN_G_I8 = 3  # below this the one-matrix kernel, one call per unit, is the faster route (persistent workgroups
               # that walk a single matrix leave most of the chip's request queues empty)


def ternary_linear_int8_grouped(layers: Sequence, xs: Optional[Tensor] = None, q: Optional[Tensor] = None,
                                s_x: Optional[Tensor] = None, out_dtype: Optional[torch.dtype] = None,
                                q_operand_order: bool = False, out: Optional[Tensor] = None) -> Tensor:
    """``Y[u] = layers[u].forward_int8(q[u], s_x[u])`` for ``G`` same-shaped layers with up to 16 activation rows each,
    in one launch.

    Either ``xs`` ``[G, M, K]`` float activations (quantized here per row, one launch for all units) or already
    quantized ``q`` ``[G, M, K]`` int8 with row scales ``s_x`` ``[G, M]`` (``q_operand_order`` as in
    :func:`ops.ternary_linear_int8`).  Returns ``[G, M, N]`` in ``out_dtype`` (default: ``xs.dtype``, or bf16)."""
    layers = list(layers)
    if not layers:
        raise ValueError("ternary_linear_int8_grouped: no layers")
    from .. import _C
    plan = _known_plan(layers)
    if plan is None:
        _check_layers("ternary_linear_int8_grouped", layers)
    g, k, n = len(layers), layers[0].in_features, layers[0].out_features
    if (xs is None) == (q is None) or (q is not None and s_x is None):
        raise ValueError("ternary_linear_int8_grouped: give xs, or q together with s_x")
    src = xs if xs is not None else q
    if src.dim() != 3 or src.shape[0] != g or src.shape[2] != k:
        raise RuntimeError(f"input K doesn't match in_features: expected [{g}, M, {k}], got {tuple(src.shape)}")
    m = src.shape[1]
    if not src.is_cuda:
        raise RuntimeError("All tensors must be CUDA")
    if out_dtype is None:
        out_dtype = xs.dtype if xs is not None and xs.dtype in (torch.float16, torch.bfloat16, torch.float32) else torch.bfloat16
    if xs is not None:
        q_operand_order = k % 16 == 0
        q2, s2 = _C.act_quant_int8(xs.reshape(g * m, k), q_operand_order)
        q, s_x = q2.view(g, m, k), s2.view(g, m)
    else:
        if q.dtype != torch.int8 or s_x.shape != (g, m) or s_x.dtype != torch.float32:
            raise RuntimeError("q must be int8 [G, M, K] and s_x fp32 [G, M]")
        q, s_x = q.contiguous(), s_x.contiguous()
    groupable = g >= _MIN_G_I8 and m <= 16 and k % 16 == 0 and k <= _MAX_K_I8 and (
        _kernels_allowed() if plan is not None else _groupable(layers, torch.empty(0, dtype=torch.float16, device=q.device)))
    if out is not None and (out.shape != (g, m, n) or out.dtype != out_dtype or not out.is_contiguous()):
        raise ValueError("ternary_linear_int8_grouped: out must be a contiguous [G, M, N] tensor of out_dtype")
    if not groupable:
        y = torch.stack([L.forward_int8(q[u], s_x[u], out_dtype, None, q_operand_order) for u, L in enumerate(layers)])
        return y if out is None else out.copy_(y)
    plan = plan or _plan_for(layers)
    y = out if out is not None else torch.empty((g, m, n), dtype=out_dtype, device=q.device)
    qt, st, yt = plan.i8_tab(q, s_x, y)
    _C.ternary_gemm_int8_grouped(qt, st, plan.w_tab, plan.s_tab, plan.b_tab, yt, m, k, n,
                                 scale_len=layers[0].scale.numel(), scale_dtype=layers[0].scale.dtype,
                                 bias_dtype=torch.float32 if layers[0].bias is None else layers[0].bias.dtype,
                                 out_dtype=out_dtype, q_operand_order=q_operand_order)
    return y
