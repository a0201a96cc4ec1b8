"""GPU: the weight gradient of a layer with fp32 masters under autocast, scaled and widened in one pass: the bits of the two
torch operations it stands for."""
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(1, 1), (3, 7), (5, 1023), (4, 1024), (6, 1027), (7, 2048), (3, 2051), (300, 4096), (33, 6145)])
def test_scale_and_widening_are_the_two_torch_operations(n, k, dtype):
    from bittorch_amd import _C
    announce("scale_grad_weight", n, k, dtype)
    gen = torch.Generator("cuda").manual_seed(n * 10007 + k)
    g = (torch.randn(n * k + 1, generator=gen, device="cuda") * 100).to(dtype)
    for at, v in enumerate((float("inf"), float("nan"), -0.0, 6.0e-8, 65504.0, float("-inf"))):
        g[at * 5::31] = v
    for rows in (g[:-1].view(n, k), g[1:].view(n, k)):  # (the second one starts off every wider alignment)
        for scale in (torch.rand(n, generator=gen, device="cuda") * 3, torch.full((1,), 0.0371, device="cuda"),
                      torch.zeros(n, device="cuda"), (torch.rand(n, generator=gen, device="cuda")).to(dtype)):
            want = (rows * scale.reshape(-1, 1).to(dtype)).float()
            got = _C.scale_grad_weight(rows, scale)
            assert got.dtype == torch.float32 and torch.equal(got.isnan(), want.isnan())
            assert torch.equal(got.nan_to_num(7.0, 1e38, -1e38).view(torch.int32), want.nan_to_num(7.0, 1e38, -1e38).view(torch.int32))


@pytest.mark.parametrize("per_channel", [True, False])
@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16])
def test_autocast_layer_gradients(per_channel, amp):
    """Through the layer: fp32 gradients equal to the unfused formula; a differentiated backward still works."""
    from bittorch_amd import nn
    announce("autocast gradients", per_channel, amp)
    layer = nn.TernaryLinear(200, 72, per_channel=per_channel).cuda()
    x = torch.randn(50, 200, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=amp):
        y = layer(x)
    gy = torch.randn_like(y)
    gx, gw, gb = torch.autograd.grad(y, (x, layer.weight, layer.bias), gy, retain_graph=True)
    assert gw.dtype == gx.dtype == gb.dtype == torch.float32
    from bittorch_amd import _C
    scale = _C.ternary_quantize_pack(layer.weight.detach().half(), layer.threshold_factor, per_channel)[1]
    # (the layer's own cast is to fp16 whatever the autocast dtype)
    want = ((gy.half().t() @ x.detach().half()) * scale.reshape(-1, 1).half()).float()
    assert torch.equal(gw, want)
    graphed = torch.autograd.grad(y, layer.weight, gy.clone().requires_grad_(), retain_graph=True, create_graph=True)[0]
    assert torch.equal(graphed, want)


@pytest.mark.parametrize("per_channel", [True, False])
@pytest.mark.parametrize("n,k", [(1, 1), (5, 7), (17, 130), (64, 256), (16, 4096), (48, 11008), (32, 5120), (300, 260), (8, 9000)])
def test_fp32_masters_quantized_as_their_fp16_copy(n, k, per_channel):
    """Rounded as they are read (both kernels, the tensor-wide maximum too): the bytes and scales of ``weight.half()``."""
    from bittorch_amd import _C
    announce("quantize as half", n, k, per_channel)
    gen = torch.Generator("cuda").manual_seed(n * 31 + k)
    w = torch.randn(n * k + 1, generator=gen, device="cuda") * 0.02
    w[::7] *= 1e-5                       # fp16 subnormals
    for rows in (w[:-1].view(n, k), w[1:].view(n, k), (w[:-1] * 1e-7).view(n, k), (w[:-1] * 3e5).view(n, k),
                 torch.full((n, k), 1e6, device="cuda")):  # (the last two overflow to infinities)
        for want_tern in (True, False):                    # (dense values come from the generic kernel only)
            got, want = (_C.ternary_quantize_pack(t, 0.05, per_channel, True, want_tern, as_half=half)
                         for t, half in ((rows, True), (rows.half(), False)))
            for a, b in zip(got, want):
                assert a is b is None or (a.dtype == b.dtype and torch.equal(a, b))
