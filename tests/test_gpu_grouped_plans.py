"""GPU: a grouped call on layers it has seen before notices whatever has changed about them since."""
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _layers(n=64, k=128, count=5, bias=True):
    from bittorch_amd import nn
    g = torch.Generator("cuda").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    return [nn.create_ternary_linear_inference(k, n, r(n, k) * 0.02, r(n) * 0.01 if bias else None).prepare_decode()
            for _ in range(count)]


def _check(layers, x, int8):
    from bittorch_amd import ops
    if int8:
        got = ops.ternary_linear_int8_grouped(layers, x[:, None])
        want = torch.stack([L.forward_int8(*ops.act_quant_int8(x[u:u + 1]), x.dtype) for u, L in enumerate(layers)])
    else:
        got = ops.ternary_linear_grouped(layers, x)
        want = torch.cat([L(x[u:u + 1]) for u, L in enumerate(layers)])
    assert torch.equal(got, want)


@pytest.mark.parametrize("int8", [False, True])
def test_changes_between_calls_are_seen(int8):
    from bittorch_amd import ops
    announce("grouped plans", int8)
    layers = _layers()
    x = torch.randn(5, 128, device="cuda").half()
    for change in (lambda: None, lambda: layers[3].scale.mul_(2), lambda: setattr(layers[1], "bias", layers[1].bias + 1),
                   lambda: layers[0].bias.zero_(), lambda: setattr(layers[2], "scale", layers[2].scale.clone() * 3),
                   lambda: layers.reverse(), lambda: layers.__setitem__(4, _layers(count=6)[5])):
        change()
        _check(layers, x, int8)
        _check(layers, x * 2, int8)
    call = ops.ternary_linear_int8_grouped if int8 else ops.ternary_linear_grouped
    xs = x[:, None] if int8 else x
    layers[2].bias = None
    with pytest.raises(ValueError):
        call(layers, xs)
    layers[2].bias = layers[1].bias
    _check(layers, x, int8)
    layers[2].scale = layers[2].scale[:1]
    with pytest.raises(ValueError):
        call(layers, xs)
    with pytest.raises(TypeError):
        call(layers[:2] + [torch.nn.Linear(128, 64)], xs[:3])
    with pytest.raises((RuntimeError, TypeError)):
        call(_layers(), xs.cpu())


def test_other_rows_types_and_strides_in_the_same_buffers():
    """A held plan whose next call finds other units at the addresses of the call before."""
    from bittorch_amd import _C, ops
    n, k, g = 64, 128, 5
    announce("grouped plans, same buffers", g, n, k)
    layers = _layers(n, k, g)
    xs, outs = torch.randn(g * 16 * k, device="cuda"), torch.empty(g * 16 * n, device="cuda")
    q, s = torch.empty(g * 16 * k, device="cuda", dtype=torch.int8), torch.empty(g * 16, device="cuda")
    for m, dtype in ((16, torch.float32), (5, torch.float32), (5, torch.bfloat16), (1, torch.float16), (16, torch.float32)):
        q1, s1 = _C.act_quant_int8(xs[:g * m * k].view(g * m, k))
        qv, sv = q[:g * m * k].view(g, m, k), s[:g * m].view(g, m)
        qv.copy_(q1.view(g, m, k))
        sv.copy_(s1.view(g, m))
        out = outs.view(dtype)[:g * m * n].view(g, m, n)
        want = torch.stack([L.forward_int8(qv[u], sv[u], dtype) for u, L in enumerate(layers)])
        assert torch.equal(ops.ternary_linear_int8_grouped(layers, q=qv, s_x=sv, out_dtype=dtype, out=out), want)
    h, outs = xs.half(), outs.view(torch.float16)
    for wide_x, wide_y in ((1, 1), (2, 1), (1, 2), (2, 2), (1, 1)):
        x, out = h[:g * wide_x * k].view(g, wide_x * k)[:, :k], outs[:g * wide_y * n].view(g, wide_y * n)[:, :n]
        want = torch.cat([L(x[u:u + 1]) for u, L in enumerate(layers)])
        assert torch.equal(ops.ternary_linear_grouped(layers, x, out=out), want)


@pytest.mark.parametrize("int8", [False, True])
def test_layers_whose_scales_and_biases_are_parameters(int8):
    announce("grouped plans, parameters", int8)
    layers = _layers()
    x = torch.randn(5, 128, device="cuda").half()
    for L in layers[1:3]:
        L.scale, L.bias = torch.nn.Parameter(L.scale.clone()), torch.nn.Parameter(L.bias.clone())
    with torch.no_grad():
        for change in (lambda: None, lambda: layers[1].scale.mul_(2), lambda: layers[2].bias.add_(1)):
            change()
            _check(layers, x, int8)
            _check(layers, x, int8)


@pytest.mark.parametrize("int8", [False, True])
def test_packed_weights_written_in_place_or_replaced(int8):
    from bittorch_amd import ops
    announce("grouped plans, packed weights", int8)
    layers = _layers()
    x = torch.randn(5, 128, device="cuda").half()
    wide = torch.rand(128, device="cuda")

    def scale_view(step):
        layers[4].scale = wide[:64 * step:step]

    for change in (lambda: None, lambda: layers[1].weight_packed.zero_(), lambda: layers[1].weight_packed[3].fill_(0x55),
                   lambda: layers[2].weight_packed, lambda: setattr(layers[2], "weight_packed", layers[1].weight_packed.clone()),
                   lambda: layers[2].drop_row_major(), lambda: scale_view(1), lambda: scale_view(2)):
        change()
        _check(layers, x, int8)
        _check(layers, x, int8)
    # written just before a capture: the captured call runs on the bytes as they are, copy or not
    call = (lambda: ops.ternary_linear_int8_grouped(layers, x[:, None])) if int8 else (lambda: ops.ternary_linear_grouped(layers, x))
    layers[1].weight_packed[5].fill_(0x11)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = call()
    want = call()
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(got.float(), want.float(), rtol=2e-3, atol=1e-4)  # (fp16 of fp32 sums in another order)


@pytest.mark.parametrize("int8", [False, True])
def test_a_graph_keeps_its_tables(int8):
    """Calls on other buffers and other layers after a capture, more than a plan and the plans hold."""
    from bittorch_amd import _C, ops
    announce("grouped plans, graph", int8)
    n, k, g = 64, 128, 5
    layers = _layers(n, k, g)
    layers[1].scale = torch.rand(2 * n, device="cuda")[::2]  # (a plan reads a contiguous copy of it)
    rows = torch.randn(g * 3, k, device="cuda").half()
    q, s = (t.view(g, 3, *t.shape[1:]) for t in _C.act_quant_int8(rows))
    x, out = rows[:g].clone(), torch.empty((g, 3, n) if int8 else (g, n), device="cuda", dtype=torch.float16)
    if int8:
        call = lambda ls, y: ops.ternary_linear_int8_grouped(ls, q=q, s_x=s, out_dtype=torch.float16, out=y)
    else:
        call = lambda ls, y: ops.ternary_linear_grouped(ls, x, out=y)
    want = call(layers, out).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(layers, out)
    others = [_layers(n, k, g) for _ in range(18)]
    outs = [torch.empty_like(out) for _ in range(12)]
    for y in outs:
        assert torch.equal(call(layers, y), want)
    for ls in others:
        call(ls, outs[0])
    fill = [torch.full((4096,), -1, dtype=torch.int64, device="cuda") for _ in range(64)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(call(layers, outs[1]), want)
    del fill


def test_calls_from_several_streams_and_threads():
    """One set of layers, each host thread on a stream and buffers of its own, more buffers than a plan keeps tables for."""
    import threading
    from bittorch_amd import ops
    announce("grouped plans, streams")
    layers, bad = _layers(), []
    x = torch.randn(5, 128, device="cuda").half()
    want = ops.ternary_linear_grouped(layers, x)
    torch.cuda.synchronize()

    def loop(stream):
        with torch.cuda.stream(stream):
            for i in range(60):
                outs = [torch.empty_like(want) for _ in range(3)]
                bad.extend(1 for y in outs if not torch.equal(ops.ternary_linear_grouped(layers, x, out=y), want))

    threads = [threading.Thread(target=loop, args=(torch.cuda.Stream(),)) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
