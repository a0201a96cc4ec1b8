"""GPU-only ternary linear layer and its autograd function.

API mirror of ``bittorch/nn/ternary_linear_cuda.py:23-228``.  Forward: one fused
HIP kernel quantizes and packs the master weights, a second one multiplies the
activations with the packed weights (fp32 accumulation).  Backward is the
straight-through estimator, as in the reference (``:73-111``): fp32 layers run on
the library's gradient kernels, which read the packed bytes; the 16-bit dtypes have a kernel
for the weight gradient and use a torch matmul for the input's, on dense effective weights
rebuilt from the packed bytes instead of being kept alive from the forward.
"""

from __future__ import annotations

import os
from typing import Optional, Tuple

import torch
import torch.nn as nn
from torch import Tensor

from ..quant.ternary import ternary_quantize
from ._packed_cache import PackedWeightCache, cache_usable
from .ternary_linear import _init_linear_params


def _fp32_kernels_serve(g2: Tensor, x2: Tensor, packed: Optional[Tensor], scale: Tensor) -> bool:
    """Whether this backward runs on the library's gradient kernels: fp32 throughout, and no graph of the backward itself
    wanted (``create_graph=True``: the torch products below are differentiable).  A batched gradient
    (``is_grads_batched=True``, a vectorized Jacobian) has no memory of its own to hand to a kernel."""
    if packed is None or torch.is_grad_enabled() or g2.numel() == 0 or _batched(g2) or _generic_forced():
        return False
    if not (g2.dtype == x2.dtype == scale.dtype == torch.float32 and g2.is_cuda):
        return False
    n, k = g2.shape[1], x2.shape[1]
    # (up to 7 outputs: the input gradient is a sum of so few products that each one's rounding, dY * scale, shows: 4 outputs
    # 4.0e-8 against 3.7e-8 as torch products, 8 outputs 4.0e-8 against 5.2e-8, 128 outputs 5.7e-8 against 1.9e-7)
    return 8 <= n < 2 ** 23 and 4 <= k < 2 ** 23 and packed.numel() < 2 ** 32


def _generic_forced() -> bool:
    """``BITTORCH_KERNEL=generic``: no kernel but the shape-generic ones, in the backward either (read on every call)."""
    return os.environ.get("BITTORCH_KERNEL") == "generic"


def _batched(t: Tensor) -> bool:
    return torch._C._functorch.is_functorch_wrapped_tensor(t) or torch._C._functorch.is_legacy_batchedtensor(t)


def _to_half(t: Optional[Tensor]) -> Optional[Tensor]:
    """What autocast does with an argument: floating-point GPU tensors other than float64 become fp16."""
    return t.half() if t is not None and t.is_cuda and t.is_floating_point() and t.dtype != torch.float64 else t


def _scale_to_master(g: Tensor, scale: Tensor, master_dtype: torch.dtype) -> Tensor:
    """The 16-bit product ``dY^T X`` times its scale.  For fp32 masters (autocast) the scale and the widening that autograd
    would do next are one pass, with the same bits; a differentiated or batched backward stays on torch."""
    if (master_dtype == torch.float32 and g.dtype in (torch.float16, torch.bfloat16) and g.is_cuda and g.numel() > 0
            and not _generic_forced() and g.shape[0] * ((g.shape[1] + 2047) // 2048) < 2 ** 30 and not torch.is_grad_enabled() and not _batched(g)):
        from .. import _C
        return _C.scale_grad_weight(g, scale)
    return g * scale.reshape(-1, 1).to(g.dtype)


def _w16_kernel_serves(g2: Tensor, x2: Tensor, scale: Tensor) -> bool:
    """Whether the weight gradient is the library's 16-bit kernel: 16-byte rows of both operands as they lie, no graph of the
    backward itself and no batched gradient wanted.  Of fewer than 2^16 weights the product takes no longer than its launch
    (256 x 256: 15 us a call against 35 for the two torch operations; the torch product serves other strides too)."""
    if torch.is_grad_enabled() or _batched(g2) or _batched(x2) or _generic_forced() or g2.numel() == 0:
        return False
    if not (g2.is_cuda and g2.dtype == x2.dtype and g2.dtype in (torch.float16, torch.bfloat16)
            and scale.dtype in (torch.float32, torch.float16, torch.bfloat16)):
        return False
    n, k = g2.shape[1], x2.shape[1]
    return (n % 8 == 0 and k % 8 == 0 and 2 ** 16 <= n * k < 2 ** 40 and n < 2 ** 24 and k < 2 ** 24 and g2.shape[0] < 2 ** 40 // max(n, k)
            and g2.is_contiguous() and x2.is_contiguous() and g2.data_ptr() % 16 == 0 and x2.data_ptr() % 16 == 0)


class TernaryLinearCUDAFunction(torch.autograd.Function):
    """``y = x @ (ternary(weight) * scale).T + bias`` with STE gradients."""

    @staticmethod
    def forward(ctx, x: Tensor, weight: Tensor, bias: Optional[Tensor], threshold_factor: float,
                per_channel: bool, cached=None) -> Tensor:
        """``cached``: optional ``(packed_T, scale, tiled copy or None)`` of exactly these weights (see
        ``_packed_cache.py``); the quantize+pack kernel is skipped when it is given.  Under autocast the layer runs in
        fp16 with autocast off; fp32 masters are rounded as the quantizer reads them."""
        ctx.master_dtype = weight.dtype
        if not torch.is_autocast_enabled("cuda"):
            return TernaryLinearCUDAFunction._forward(ctx, x, weight, bias, threshold_factor, per_channel, cached, False)
        as_half = (cached is None and x.dtype != torch.float64 and weight.dtype == torch.float32 and weight.is_cuda)
        with torch.autocast("cuda", enabled=False):
            return TernaryLinearCUDAFunction._forward(ctx, _to_half(x), weight if as_half else _to_half(weight),
                                                      _to_half(bias), threshold_factor, per_channel, cached, as_half)

    @staticmethod
    def _forward(ctx, x, weight, bias, threshold_factor, per_channel, cached, as_half) -> Tensor:
        from .. import _C

        if weight.dtype == torch.float64 or x.dtype == torch.float64:
            w_tern, scale = ternary_quantize(weight, threshold_factor, per_channel)
            out = _C.ternary_linear_forward(x.contiguous(), w_tern.to(torch.int8),
                                            scale.reshape(-1).to(x.dtype),
                                            None if bias is None else bias.to(x.dtype))
            packed = None
            ctx.w_eff = w_tern * scale.reshape(-1, 1)
        else:
            tiled = None
            if cached is not None:
                packed, scale, tiled = cached
            else:
                packed, scale, _ = _C.ternary_quantize_pack(weight, threshold_factor, per_channel, as_half=as_half)
            b = None if bias is None else bias.to(x.dtype).contiguous()
            if (tiled is not None and x.dtype in (torch.float16, torch.bfloat16, torch.float32)
                    and not _generic_forced()):  # (the shape-generic kernel reads packed_T)
                out = _C.ternary_linear_tiled_forward(x.contiguous(), tiled, scale.reshape(-1).to(x.dtype), b,
                                                      weight.shape[1], weight.shape[0])
            else:
                out = _C.ternary_linear_packed_forward(x.contiguous(), packed, scale.reshape(-1).to(x.dtype), b,
                                                       weight.shape[1])
            ctx.w_eff = None
        ctx.save_for_backward(x, packed, scale)
        ctx.in_features = weight.shape[1]
        ctx.weight_dtype = torch.float16 if as_half else weight.dtype
        ctx.has_bias = bias is not None
        return out

    @staticmethod
    def backward(ctx, grad_output: Tensor):
        with torch.autocast("cuda", enabled=False):  # (as the forward)
            return TernaryLinearCUDAFunction._backward(ctx, grad_output)

    @staticmethod
    def _backward(ctx, grad_output: Tensor):
        from .. import _C

        x, packed, scale = ctx.saved_tensors
        g2 = grad_output.reshape(-1, grad_output.shape[-1])
        x2 = x.reshape(-1, x.shape[-1])
        grad_x = grad_w = grad_b = None
        want_bias = ctx.has_bias and ctx.needs_input_grad[2]
        if _fp32_kernels_serve(g2, x2, packed, scale):
            if ctx.needs_input_grad[0]:
                grad_x = _C.linear_grad_input(g2, packed, scale.reshape(-1), ctx.in_features).reshape(x.shape)
            if ctx.needs_input_grad[1]:
                grad_w, grad_b = _C.linear_grad_weight(g2, x2, scale.reshape(-1), want_bias)
            elif want_bias:
                grad_b = g2.sum(dim=0)
            return grad_x, grad_w, grad_b, None, None, None
        if ctx.needs_input_grad[0]:
            if packed is not None:
                w_eff = _C.unpack_dequant(packed, ctx.in_features, scale.reshape(-1),
                                          out_dtype=ctx.weight_dtype)
            else:
                w_eff = ctx.w_eff
            grad_x = (g2 @ w_eff.to(g2.dtype)).reshape(x.shape)
        if ctx.needs_input_grad[1]:
            # d(w_eff)/d(weight) = scale under the straight-through estimator
            if _w16_kernel_serves(g2, x2, scale):
                grad_w = _C.linear_grad_weight_16(g2, x2, scale, torch.float32 if ctx.master_dtype == torch.float32 else g2.dtype)
            else:
                grad_w = _scale_to_master(g2.t() @ x2, scale, ctx.master_dtype)
        if want_bias:
            grad_b = g2.sum(dim=0)
        return grad_x, grad_w, grad_b, None, None, None


class TernaryLinearCUDA(nn.Module):
    """Ternary linear layer that only accepts GPU tensors (reference ``:114-228``)."""

    def __init__(self, in_features: int, out_features: int, bias: bool = True,
                 threshold_factor: float = 0.05, per_channel: bool = True) -> None:
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.threshold_factor = threshold_factor
        self.per_channel = per_channel
        self.weight = nn.Parameter(torch.empty(out_features, in_features))
        if bias:
            self.bias = nn.Parameter(torch.empty(out_features))
        else:
            self.register_parameter("bias", None)
        self._packed = PackedWeightCache()
        self.reset_parameters()

    def reset_parameters(self) -> None:
        _init_linear_params(self.weight, self.bias)

    def forward(self, x: Tensor) -> Tensor:
        if not x.is_cuda:
            raise RuntimeError("TernaryLinearCUDA requires CUDA tensors. Use TernaryLinear for CPU.")
        cached = None
        if cache_usable(x, self.weight):
            cached = self._packed.get(self.weight, self.threshold_factor, self.per_channel)
        return TernaryLinearCUDAFunction.apply(x, self.weight, self.bias, self.threshold_factor,
                                               self.per_channel, cached)

    def invalidate_packed_cache(self) -> None:
        """Forget the cached packed weights (needed only after an evaluation-time write through ``weight.data``,
        which the version counter the cache is keyed on does not see)."""
        self._packed.clear()

    def extra_repr(self) -> str:
        return (f"in_features={self.in_features}, out_features={self.out_features}, "
                f"bias={self.bias is not None}, threshold_factor={self.threshold_factor}, "
                f"per_channel={self.per_channel}")

    def get_quantized_weight(self) -> Tuple[Tensor, Tensor]:
        with torch.no_grad():
            return ternary_quantize(self.weight, self.threshold_factor, self.per_channel)
