"""CPU: the address tables of the grouped calls (``ops/grouped.py``) follow the sizes, types and strides of a call's buffers,
also where a buffer's address is one seen before."""
from collections import OrderedDict

import pytest
import torch


def _plan():
    grouped = pytest.importorskip("bittorch_amd.ops.grouped")
    plan = object.__new__(grouped._Plan)  # (a plan's other tables hold device addresses of layers)
    plan.io_tabs, plan.i8_tabs = OrderedDict(), OrderedDict()
    return plan


def _addresses(t):
    return [t[u].data_ptr() for u in range(t.shape[0])]


def test_int8_tables_of_other_rows_and_types_at_the_same_addresses():
    plan, g, k, n = _plan(), 3, 64, 32
    q, s, y = torch.zeros(g * 16 * k, dtype=torch.int8), torch.zeros(g * 16), torch.zeros(g * 16 * n)
    for m, dtype in ((16, torch.float32), (5, torch.float32), (5, torch.bfloat16), (16, torch.bfloat16), (16, torch.float32)):
        views = (q[:g * m * k].view(g, m, k), s[:g * m].view(g, m), y.view(dtype)[:g * m * n].view(g, m, n))
        for tab, t in zip(plan.i8_tab(*views), views):
            assert tab.tolist() == _addresses(t)


def test_float_tables_of_other_strides_at_the_same_addresses():
    plan, g, k, n = _plan(), 4, 64, 32
    x, y = torch.zeros(g * 2 * k, dtype=torch.float16), torch.zeros(g * 2 * n, dtype=torch.float16)
    xs = [x[:g * k].view(g, k), x.view(g, 2 * k)[:, :k]]
    ys = [y[:g * n].view(g, n), y.view(g, 2 * n)[:, :n]]
    for i, j in ((0, 0), (1, 0), (0, 1), (1, 1), (0, 0)):
        xt, yt = plan.io_tab(xs[i], ys[j], False)
        assert xt.tolist() == _addresses(xs[i]) and yt.tolist() == _addresses(ys[j])
    row = x[:k].view(1, k)
    assert plan.io_tab(row, ys[0], True)[0].tolist() == [x.data_ptr()] * g


def test_tables_of_a_captured_call_outlive_the_plan():
    """A graph's launches hold the tables' addresses alone: other buffers' tables and other plans must not free them."""
    import gc
    import weakref
    plan, g = _plan(), 3
    grouped = pytest.importorskip("bittorch_amd.ops.grouped")
    plan.w_tab = torch.zeros(g, dtype=torch.int64)
    plan.own = [plan.w_tab, torch.zeros(g)]
    buffers = torch.zeros(100, g, 8)
    tabs = plan.io_tab(buffers[0], buffers[1], False)
    plan._keep_for_graph(((buffers[0].data_ptr(), 32), (buffers[1].data_ptr(), 32)), tabs)
    alive = [weakref.ref(t) for t in (*tabs, *plan.own)]
    for i in range(2, 50):
        plan.io_tab(buffers[i], buffers[i + 1], False)
    del tabs, plan
    gc.collect()
    assert all(r() is not None for r in alive)
    grouped._CAPTURED.clear()
    gc.collect()
    assert all(r() is None for r in alive)


def test_fingerprint_of_a_layer_whose_scale_and_bias_are_parameters():
    grouped = pytest.importorskip("bittorch_amd.ops.grouped")
    from bittorch_amd import nn
    layer = nn.create_ternary_linear_inference(64, 32, torch.randn(32, 64), torch.randn(32))
    held = [layer.scale, layer.bias]  # (as a plan does)
    keys = [grouped._fingerprint([layer])]
    for name in ("scale", "bias"):
        setattr(layer, name, torch.nn.Parameter(getattr(layer, name).clone()))
        held.append(getattr(layer, name))
        keys.append(grouped._fingerprint([layer]))
    assert all(a != b for i, a in enumerate(keys) for b in keys[:i])
    assert grouped._fingerprint([layer]) == keys[-1]


def test_fingerprint_sees_packed_weights_and_views():
    """A held ``weight_packed`` written in place or replaced; a scale or bias that is another view of the same address, that
    is shortened or pointed elsewhere, or that is written where the tables hold a contiguous copy of it."""
    grouped = pytest.importorskip("bittorch_amd.ops.grouped")
    from bittorch_amd import nn
    layer = nn.create_ternary_linear_inference(64, 32, torch.randn(32, 64), torch.randn(64)[:32])
    wide, held = torch.rand(64), []
    layer.scale = wide[:32]
    keys = [grouped._fingerprint([layer])]
    with torch.no_grad():
        for change in (lambda: layer.weight_packed.bitwise_xor_(1), lambda: setattr(layer, "weight_packed", layer.weight_packed.clone()),
                       lambda: setattr(layer, "bias", torch.as_strided(layer.bias, (32,), (2,))), lambda: layer.bias.add_(1),
                       lambda: setattr(layer.bias, "data", layer.bias.clone()), lambda: setattr(layer, "scale", wide[::2]),
                       lambda: setattr(layer.scale, "data", wide[:32]), lambda: setattr(layer.scale, "data", wide[:1]),
                       lambda: setattr(layer, "bias", None)):
            held += [layer.scale, layer.bias]
            change()
            keys.append(grouped._fingerprint([layer]))
    assert all(a != b for i, a in enumerate(keys) for b in keys[:i])
