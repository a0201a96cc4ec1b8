"""GPU: the weight gradient of 16-bit layers against fp32 sums of the same products, at the edges of its tiles and parts."""
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

# (rows, N, K): one tile, edges of 128 and 256, rows around a stage (32, 64) and a loop (128, 256), tails summed in parts (few
# tiles, many rows; the last part shorter), a whole round of tiles and a remainder in parts (11008 x 2048 holds 344 tiles of 256)
SHAPES = [(1, 256, 256), (31, 264, 248), (33, 128, 512), (65, 136, 520), (127, 8, 8192), (129, 8200, 8), (255, 1024, 1032),
          (300, 768, 776), (1025, 256, 264), (2100, 128, 640), (5000, 768, 768), (9001, 264, 520), (700, 11008, 2048), (2305, 11008, 2048)]


@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float32), (torch.bfloat16, torch.float32), (torch.float16, torch.float16),
                                       (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_weight_gradient(m, n, k, dtype, out):
    from bittorch_amd import _C
    announce("linear_grad_weight_16", m, n, k, dtype, out)
    gen = torch.Generator("cuda").manual_seed(m * 31 + n * 7 + k)
    gy = torch.randn(m, n, generator=gen, device="cuda").to(dtype)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    for scale in (torch.rand(n, generator=gen, device="cuda") + 0.01, torch.full((1,), 0.0371, device="cuda").to(dtype)):
        got = _C.linear_grad_weight_16(gy, x, scale, out)
        assert got.dtype == out and got.shape == (n, k)
        s = scale.reshape(-1, 1).to(dtype).float()
        sums = gy.float().t() @ x.float()
        # fp32 sums of m products differ by at most 2 m 2^-24 sum |dY X| with their order; then two roundings to the dtype
        eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
        bound = s * (2 * m * 2.0 ** -24 * (gy.abs().float().t() @ x.abs().float()) * (1 + 2 * eps) + 2.01 * eps * sums.abs()) + 1e-7
        assert bool(((got.float() - sums * s).abs() <= bound).all())


# What each kind of launch stores, with the scratch that shows which it is: parts x bytes of one (256 KiB for tiles of 256, 64 KiB
# for tiles of 128).  Tiles of 128 whole and in parts, tiles of 256 whole, a round and the rest in equal parts, in two unequal ones
# (an XCD's share of the tiles full and one short, columns and rows that end inside a tile)
BIG, SMALL = 256 << 10, 64 << 10
LAUNCHES = [((257, 2040, 2048), 0), ((600, 2048, 2048), 0), ((1025, 256, 264), 6 * 5 * SMALL), ((9001, 264, 520), 15 * 12 * SMALL),
            ((70, 2560, 6920), 0), ((300, 4104, 3840), 0), ((2305, 11008, 2048), 88 * 2 * BIG), ((2048, 2560, 6912), 14 * 4 * BIG),
            ((8192, 3072, 3072), 144 * 2 * BIG), ((6200, 3080, 3000), 156 * 2 * BIG), ((6000, 2056, 4200), 153 * 2 * BIG)]


@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("shape,scratch", LAUNCHES)
def test_every_launch_is_exact_on_small_integers(shape, scratch, dtype, out):
    """Sums of small whole numbers have one value in any order and any parts; it is rounded to the operands' dtype once."""
    from bittorch_amd import _C
    m, n, k = shape
    announce("exact sums", m, n, k, dtype)
    assert _C._L.bt_linear_grad_weight_16_workspace_bytes(m, n, k) == scratch
    gen = torch.Generator("cuda").manual_seed(m + n + k)
    gy = torch.randint(-2, 3, (m, n), device="cuda", generator=gen).to(dtype)
    x = torch.randint(-1, 2, (m, k), device="cuda", generator=gen).to(dtype)
    got = _C.linear_grad_weight_16(gy, x, torch.ones(n, device="cuda"), out)
    assert torch.equal(got, (gy.float().t() @ x.float()).to(dtype).to(out))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_small_integers_are_exact(dtype):
    """Sums of small whole numbers have one value in any order: every output, by row and column, of both tile sizes."""
    from bittorch_amd import _C
    for m, n, k in ((96, 520, 264), (64, 4104, 4096)):
        announce("exact sums", m, n, k, dtype)
        gy = torch.randint(-2, 3, (m, n), device="cuda").to(dtype)
        x = torch.randint(-1, 2, (m, k), device="cuda").to(dtype)
        got = _C.linear_grad_weight_16(gy, x, torch.ones(n, device="cuda"), torch.float32)
        assert torch.equal(got, gy.float().t() @ x.float())


def test_non_finite_rows_stay_in_their_outputs():
    from bittorch_amd import _C
    announce("non-finite")
    gy, x = torch.randn(70, 264, device="cuda").half(), torch.randn(70, 256, device="cuda").half()
    gy[69, 263], x[3, 5] = float("inf"), float("nan")
    got = _C.linear_grad_weight_16(gy, x, torch.ones(264, device="cuda"), torch.float32)
    want = torch.zeros(264, 256, dtype=torch.bool, device="cuda")
    want[263, :], want[:, 5] = True, True
    assert torch.equal(~got.isfinite(), want)


@pytest.mark.parametrize("form", ["contiguous", "expanded", "transposed", "offset"])
def test_layer_backward_takes_any_gradient(form):
    """Gradients and inputs of other strides and starts keep their way through torch; the values agree."""
    from bittorch_amd import nn
    announce("layer backward", form)
    layer = nn.TernaryLinear(264, 256, bias=False).cuda().bfloat16()
    x = torch.randn(96 * 264 + 8, device="cuda", dtype=torch.bfloat16)
    x = (x[1:96 * 264 + 1] if form == "offset" else x[:96 * 264]).view(96, 264).requires_grad_()
    y = layer(x)
    gy = {"expanded": lambda: torch.ones(1, 1, device="cuda", dtype=torch.bfloat16).expand(96, 256),
          "transposed": lambda: torch.randn(256, 96, device="cuda", dtype=torch.bfloat16).t()}.get(
              form, lambda: torch.randn(96, 256, device="cuda", dtype=torch.bfloat16))()
    gw, = torch.autograd.grad(y, layer.weight, gy)
    _, scale = layer.get_quantized_weight()
    want = (gy.float().t() @ x.detach().float()) * scale.reshape(-1, 1).bfloat16().float()
    assert gw.dtype == torch.bfloat16 and torch.allclose(gw.float(), want, rtol=2 ** -6, atol=2 ** -6 * float(want.std()))
