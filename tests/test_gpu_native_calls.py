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
    n, k, m = 320, 256, 24  # (three numbers, so that none stands for another)
    announce("native quantizer and gradients", dtype)
    x, packed, tiled, scale, bias, res, norm = _make(dtype, (m,), n, k)
    w = torch.randn(n, k, device="cuda").to(dtype)
    for per_channel in (True, False):
        _both(monkeypatch, lambda: _C.ternary_quantize_pack(w, 0.05, per_channel))
    if dtype == torch.float32:
        _both(monkeypatch, lambda: _C.ternary_quantize_pack(torch.nn.Parameter(w), 0.1, True, as_half=True))
        _both(monkeypatch, lambda: _C.linear_grad_input(res, packed, scale, k))
        for want in (False, True):
            _both(monkeypatch, lambda: _C.linear_grad_weight(res, x, scale, want))
    else:
        for out in (dtype, torch.float32):
            _both(monkeypatch, lambda: _C.linear_grad_weight_16(res, x, scale, out))
    for out in (torch.float32, torch.float16, torch.bfloat16):
        for sc in (scale.to(dtype), scale[:1].clone()):
            _both(monkeypatch, lambda: _C.unpack_dequant(packed, k, sc, out))
    for wt in (norm, None):
        for order in (False, True):
            _both(monkeypatch, lambda: _C.rmsnorm(x, wt, 1e-5, store=False, quantize=True, operand_order=order))
    wide = torch.cat([x, x.flip(0)], dim=1)
    for order in (False, True):
        _both(monkeypatch, lambda: _C.swiglu(wide[:, :k], wide[:, k:], store=False, quantize=True, operand_order=order))
        _both(monkeypatch, lambda: _C.act_quant_int8(x, order))
        q, s = _C.act_quant_int8(x, order)
        for r in (None, res):
            _both(monkeypatch, lambda: _C.ternary_gemm_int8_tiled(q, s, tiled, scale, bias, k, n, dtype, residual=r, q_operand_order=order))
    if dtype != torch.float32:  # (q in operand order)
        for sc, b in ((scale, None), (scale[:1].clone(), bias), (scale.to(dtype), bias.to(dtype))):
            _both(monkeypatch, lambda: _C.ternary_swiglu_int8_tiled(q, s, tiled, sc, b, k, n, dtype))


def test_refused_calls_are_refused_alike(monkeypatch):
    """What each function refuses, with the native module and without it: the same error (none of these reaches a launch)."""
    from bittorch_amd import _C
    n, k, m = 64, 128, 6
    x, packed, tiled, scale, bias, res, norm = _make(torch.bfloat16, (m,), n, k)
    f, fres = x.float(), res.float()
    q, s = _C.act_quant_int8(x, True)
    bf16, fp32 = torch.bfloat16, torch.float32
    calls = [
        (_C.ternary_linear_packed_forward, (x, packed, scale, bias, k),
         [(0, x[:0]), (0, x[:, :-8]), (0, x.int()), (0, x.cpu()), (1, packed[:-1]), (1, packed.to(torch.int8)), (1, packed[0]), (2, scale[:5]),
          (2, scale[None]), (3, bias[:-1]), (4, k + 1), (4, 0)]),
        (_C.ternary_linear_tiled_forward, (x, tiled, scale, bias, k, n),
         [(0, x[:0]), (0, x.int()), (0, x.cpu()), (1, tiled[:-256]), (1, tiled[1:]), (1, tiled.to(torch.int8)), (2, scale[:5]), (3, bias[:-1]),
          (4, k + 1), (5, n + 16), (5, 0), (5, -1)]),
        (lambda *a: _C.ternary_linear_tensor_core_forward(*a, 2), (x, packed, scale, bias, k),
         [(0, x[:0]), (0, x[0]), (0, x.int()), (0, x.cpu()), (1, packed[:-1]), (2, scale[:5]), (3, bias[:-1]), (4, k + 1)]),
        (_C.ternary_gemm_int8_tiled, (q, s, tiled, scale, bias, k, n, bf16, False, None, True),
         [(0, q[:0]), (0, q[0]), (0, x), (0, q.cpu()), (1, s[:-1]), (1, s.double()), (2, tiled[:-256]), (3, scale[:5]), (4, bias[:-1]), (5, k + 1),
          (6, n + 16), (7, torch.int32), (9, res[:-1]), (9, res.float())]),
        (_C.ternary_swiglu_int8_tiled, (q, s, tiled, scale, bias, k, n, bf16),
         [(0, q[:0]), (0, x), (0, q.cpu()), (1, s[:-1]), (1, s.double()), (2, tiled[:-256]), (3, scale[:5]), (4, bias[:-1]), (5, k + 1), (6, n - 16),
          (7, fp32)]),
        (_C.ternary_quantize_pack, (f,), [(0, f[0]), (0, f[:0]), (0, f.int()), (0, f.cpu())]),
        (lambda *a: _C.ternary_quantize_pack(*a, as_half=True), (f,), [(0, x)]),
        (_C.act_quant_int8, (x, True), [(0, x[0]), (0, x[:0]), (0, x.int()), (0, x.cpu()), (0, x[:, :-8].contiguous())]),
        (lambda *a: _C.rmsnorm(*a, store=False, quantize=True, operand_order=True), (x, norm, 1e-5),
         [(0, x[:0]), (0, x.int()), (0, x.cpu()), (0, x[:, :-8].contiguous()), (1, norm[:-1]), (1, norm[None])]),
        (lambda *a: _C.swiglu(*a, store=False, quantize=True, operand_order=True), (x, x),
         [(0, x[:0]), (0, f), (0, x.cpu()), (1, x[:-1]), (1, f)]),
        (lambda *a: _C.swiglu(*a, store=False, quantize=True, operand_order=True), (x[:, :40], x[:, :40]), [(0, x[:, :40])]),
        (_C.unpack_dequant, (packed, k, scale, fp32),
         [(0, packed[:-1]), (0, packed.to(torch.int8)), (0, packed.cpu()), (1, k + 4), (2, scale[:5]), (3, torch.int32)]),
        (_C.linear_grad_input, (fres, packed, scale, k),
         [(0, fres[:0]), (0, fres[0]), (0, res), (0, fres.cpu()), (0, fres[:, :-1]), (1, packed[:-1]), (1, packed.to(torch.int8)), (2, scale[:5]),
          (2, scale.double()), (3, k + 4)]),
        (_C.linear_grad_weight, (fres, f, scale), [(0, fres[:0]), (0, res), (0, fres[:-1]), (1, f[0]), (1, x), (1, f.cpu()), (1, f[:, :3].contiguous()), (2, scale[:5]),
                                                   (2, scale.double())]),
        (_C.linear_grad_weight_16, (res, x, scale, bf16),
         [(0, res[:0]), (0, fres), (0, res[:-1]), (0, res.half()), (1, x[0]), (1, x.cpu()), (1, x[:, :-1].contiguous()), (2, scale[:5]), (2, scale.double()),
          (3, torch.float16)]),
    ]
    real = _C._N
    for i, (call, args, changes) in enumerate(calls):
        for at, value in changes:
            announce("refused alike", i, at, tuple(value.shape) if isinstance(value, torch.Tensor) else value)
            errors = []
            for module in (real, _AsksNobody()):
                monkeypatch.setattr(_C, "_N", module)
                with pytest.raises((RuntimeError, IndexError)) as e:
                    call(*args[:at], value, *args[at + 1:])
                errors.append((e.type, str(e.value)))
            assert errors[0] == errors[1]
    monkeypatch.setattr(_C, "_N", real)


def test_other_calls_go_to_python(monkeypatch):
    """Strides, alignment, other dtypes, subclasses and modes: not the native call's."""
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
