"""The native host side of the calls (csrc/calls.cpp) against the Python functions it stands in for: the same bits for every form it
takes, None for every other, and the Python function's answer or error then."""
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import announce

pytestmark = pytest.mark.gpu


class _AsksNobody:
    """In the place of the native module: no call is ordinary."""

    def __getattr__(self, name):
        return (lambda: False) if name == "generic_kernel_asked" else (lambda *a: None)


class _Counts:
    def __init__(self, real):
        self.real, self.taken = real, 0

    def __getattr__(self, name):
        def f(*a):
            r = getattr(self.real, name)(*a)
            self.taken += r is not None
            return r
        return f


def _same(a, b):
    if isinstance(a, (tuple, list)):
        return len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    if a is None or b is None:
        return a is b
    return a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous() == b.is_contiguous() and \
        a.requires_grad == b.requires_grad and torch.equal(a, b)


def _both(monkeypatch, f, native=True):
    """f with the native module (which takes the call, or does not) and without it"""
    from bittorch_amd import _C
    real = _C._N
    counts = _Counts(real)
    monkeypatch.setattr(_C, "_N", counts)
    got = f()
    assert (counts.taken > 0) == native
    monkeypatch.setattr(_C, "_N", _AsksNobody())
    want = f()
    monkeypatch.setattr(_C, "_N", real)
    assert _same(got, want)


def _make(dtype, lead, n, k):
    from bittorch_amd import _C
    g = torch.Generator("cuda").manual_seed(n + k)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    packed, scale, _ = _C.ternary_quantize_pack(r(n, k) * 0.02)
    return r(*lead, k).to(dtype), packed, _C.retile_weights(packed, k), scale, r(n) * 0.1, r(*lead, n).to(dtype), (1 + 0.1 * r(k)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lead", [(), (1,), (5,), (2, 3), (40,)])
def test_forwards(monkeypatch, dtype, lead):
    from bittorch_amd import _C
    n, k = 96, 200
    announce("native forwards", dtype, lead)
    x, packed, tiled, scale, bias, res, norm = _make(dtype, lead, n, k)
    up = x.flip(-1).contiguous()
    pairs = _C.retile_weights(packed, k, True)
    for sc in (scale, scale[:1].clone(), scale.to(dtype)):
        for b in (None, bias, bias.to(dtype)):
            _both(monkeypatch, lambda: _C.ternary_linear_packed_forward(x, packed, sc, b, k))
            _both(monkeypatch, lambda: _C.ternary_linear_packed_forward(x, packed, sc, b))
            for kw in ({}, {"residual": res}, {"norm": (norm, 1e-5)}, {"norm": (None, 1e-5), "residual": res}, {"swiglu_up": up}):
                _both(monkeypatch, lambda: _C.ternary_linear_tiled_forward(x, tiled, sc, b, k, n, **kw))
            _both(monkeypatch, lambda: _C.ternary_linear_tiled_forward(x, pairs, sc, b, k, n, natural_from_pairs=True))
            if dtype != torch.float32:
                _both(monkeypatch, lambda: _C.ternary_linear_tiled_forward(x, pairs, sc, b, k, n, norm=(norm, 1e-5), swiglu_pairs=True))
            if len(lead) == 1:
                _both(monkeypatch, lambda: _C.ternary_linear_tensor_core_forward(x, packed, sc, b, k, 2))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_quantizers_gradients_and_int8(monkeypatch, dtype):
    from bittorch_amd import _C
    n, k, m = 256, 256, 24
    announce("native quantizer and gradients", dtype)
    x, packed, tiled, scale, bias, res, norm = _make(dtype, (m,), n, k)
    w = torch.randn(n, k, device="cuda").to(dtype)
    for per_channel in (True, False):
        _both(monkeypatch, lambda: _C.ternary_quantize_pack(w, 0.05, per_channel))
    if dtype == torch.float32:
        _both(monkeypatch, lambda: _C.ternary_quantize_pack(torch.nn.Parameter(w), 0.1, True, as_half=True))
        _both(monkeypatch, lambda: _C.linear_grad_input(x, packed, scale, k))
        for want in (False, True):
            _both(monkeypatch, lambda: _C.linear_grad_weight(x, res, scale, want))
    else:
        for out in (dtype, torch.float32):
            _both(monkeypatch, lambda: _C.linear_grad_weight_16(x, res, scale, out))
    for out in (torch.float32, torch.float16, torch.bfloat16):
        _both(monkeypatch, lambda: _C.unpack_dequant(packed, k, scale.to(dtype), out))
    q, s = _C.rmsnorm(x, norm, 1e-5, store=False, quantize=True)
    for wt in (norm, None):
        _both(monkeypatch, lambda: _C.rmsnorm(x, wt, 1e-5, store=False, quantize=True, operand_order=True))
    wide = torch.cat([x, x.flip(0)], dim=1)
    _both(monkeypatch, lambda: _C.swiglu(wide[:, :k], wide[:, k:], store=False, quantize=True))
    for r in (None, res):
        _both(monkeypatch, lambda: _C.ternary_gemm_int8_tiled(q, s, tiled, scale, bias, k, n, dtype, residual=r))


def test_other_calls_go_to_python(monkeypatch):
    """Strides, alignment, other dtypes and devices, subclasses, modes and transforms: not the native call's."""
    from bittorch_amd import _C
    n, k, m = 64, 128, 6
    x, packed, tiled, scale, bias, res, norm = _make(torch.bfloat16, (m,), n, k)
    off = torch.empty(m * n + 1, dtype=torch.bfloat16, device="cuda")[1:].view(m, n).copy_(res)
    call = lambda **kw: _C.ternary_linear_tiled_forward(**{**dict(X=x, W_tiled=tiled, scale=scale, bias=bias, in_features=k, out_features=n), **kw})
    for kw in (dict(X=torch.cat([x, x], 1)[:, :k]), dict(X=x.t().contiguous().t()), dict(residual=off), dict(scale=scale.double()),
               dict(bias=torch.cat([bias, bias])[::2]), dict(norm=(norm.float(), 1e-5)), dict(norm=[norm, 1e-5]),
               dict(X=x.as_subclass(type("T", (torch.Tensor,), {})))):
        announce("python call", list(kw))
        _both(monkeypatch, lambda: call(**kw).as_subclass(torch.Tensor), native=False)
    for kw in (dict(in_features=k + 1), dict(scale=scale[:5]), dict(W_tiled=tiled[:-256]), dict(residual=res[:-1]), dict(X=x.cpu()),
               dict(X=x[:0]), dict(X=x.to(torch.int32)), dict(norm=(norm, 1e-5), swiglu_up=x), dict(swiglu_pairs=True, residual=res)):
        announce("refused call", list(kw))
        with pytest.raises(RuntimeError):
            call(**kw)

    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Dispatches(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatches):
        del seen[:]
        with mode():
            got = _C.ternary_linear_packed_forward(x, packed, scale, bias, k)
        assert seen and torch.equal(got, _C.ternary_linear_packed_forward(x, packed, scale, bias, k))
    with torch.autocast("cuda", dtype=torch.float16), torch.inference_mode():
        assert call().is_inference()
    assert not call(X=x.requires_grad_()).requires_grad


def test_streams_and_graphs():
    """The current stream, its capture, and scratch that the graph's pool holds."""
    from bittorch_amd import _C
    n, k, m = 256, 1000, 40  # (rows that are padded: scratch)
    x, packed, tiled, scale, bias, _, _ = _make(torch.float16, (m,), n, k)
    want = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
    side.synchronize()
    assert torch.equal(y, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
    for i in range(3):
        x.normal_()
        torch.empty(1 << 20, device="cuda").fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n))
