"""GPU: the fp32 matrix-core kernels of ``csrc/gemm_f32.hip`` (forward on row-major and tiled weights, input gradient,
weight and bias gradient) against float64.

Every product is formed from bf16 terms that are the operands exactly, and they are added in fp32.  With ``C`` products in
steps of 32, the largest terms of all products and, once a step each, the sums of the smaller ones are added to a sum of full
size: at most ``C + (kinds of terms - 1) ceil(C / 32)`` roundings of 2^-24 of the sum of the products' magnitudes, and as many
more as parts of the sum are added up or factors multiplied.  The weight gradient leaves out two kinds of terms of at most
2^-25 of a product each; over up to 8 rows it is formed of fp32 products.
"""
import pytest
import torch

from conftest import announce
from _util import set_option

gpu = pytest.mark.gpu
EPS = 2.0 ** -24

# edges of the tiles (64, 128, 256 outputs; contraction steps of 32, split over 4 or 8 waves), remainders, the smallest
SHAPES = [(1, 4, 4), (33, 4, 5), (40, 20, 33), (65, 64, 31), (64, 256, 32), (129, 132, 77), (200, 300, 258), (300, 100, 1000),
          (513, 1028, 96), (1000, 36, 2048), (2100, 768, 260), (4099, 516, 516), (16384, 192, 130)]


def _close(got, a, b, roundings, scale=1.0):
    """got against a @ b in float64, by the bound above; scale: a factor of the rows or columns that is rounded too"""
    ref = (a.double() @ b.double()) * scale
    bound = roundings * EPS * ((a.double().abs() @ b.double().abs()) * scale) + 1e-37
    assert torch.isfinite(got).all()
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


def _three_terms(c):
    """Of a sum of c products with a ternary operand: up to 8 parts, a rounded factor before and after, the last rounding."""
    return c + 2 * ((c + 31) // 32) + 11


def _six_terms(m):
    """Of a weight gradient over m rows (up to 8: fp32 products): parts of 256 rows or more, the scale."""
    return m + 1 if m <= 8 else m + 5 * ((m + 31) // 32) + (m + 255) // 256 + 2


def _case(m, n, k, per_channel=True):
    from bittorch_amd import _C
    g = torch.Generator("cuda").manual_seed(m * 7 + n * 3 + k)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    w = r(n, k) * 0.02
    packed, scale, tern = _C.ternary_quantize_pack(w, 0.05, per_channel, True, True)
    return r(m, k), r(m, n) * 0.01, packed, scale.reshape(-1), tern.float()


@gpu
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_fp32_products_against_float64(m, n, k):
    from bittorch_amd import _C
    announce("fp32 gradients", m, n, k)
    x, dy, packed, scale, tern = _case(m, n, k)
    _close(_C.linear_grad_input(dy, packed, scale, k), dy, tern * scale[:, None], _three_terms(n))
    dw, db = _C.linear_grad_weight(dy, x, scale, True)
    _close(dw, dy.t(), x, _six_terms(m), scale.double()[:, None])
    _close(db[:, None], dy.t(), torch.ones(m, 1, device="cuda"), m)
    assert torch.equal(_C.linear_grad_weight(dy, x, scale, True)[0], dw)  # a fixed order of the sums
    set_option("STREAM_MAX_ROWS", "1")  # (the kernel that splits in registers at any number of rows)
    if m > 1 and n % 4 == 0:
        y = _C.ternary_linear_packed_forward(x, packed, scale, None, k)
        _close(y, x, tern.t(), _three_terms(k), scale.double()[None, :])
        _close(_C.ternary_linear_tiled_forward(x, _C.retile_weights(packed, k), scale, None, k, n), x, tern.t(),
               _three_terms(k), scale.double()[None, :])


@gpu
@pytest.mark.parametrize("m,n,k", [(70, 24, 40), (1500, 130, 70)])
def test_fp32_gradients_one_scale_strides_and_alignment(m, n, k):
    """A per-tensor scale; operands that start 4 bytes into a buffer; an expanded (stride 0) output gradient."""
    from bittorch_amd import _C
    announce("fp32 gradients, views", m, n, k)
    x, dy, packed, scale, tern = _case(m, n, k, per_channel=False)
    off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view_as(t)
    _close(_C.linear_grad_input(off(dy), packed, scale, k), dy, tern * scale, _three_terms(n))
    _close(_C.linear_grad_weight(off(dy), off(x), scale)[0], dy.t(), x, _six_terms(m), float(scale))
    wide = dy[:, :1].expand(m, n)
    _close(_C.linear_grad_weight(wide, x, scale)[0], wide.t(), x, _six_terms(m), float(scale))


@gpu
@pytest.mark.parametrize("m", [1, 2, 8, 9, 31, 32, 33, 300])
def test_weight_gradient_of_few_rows(m):
    """Sums of few products, whose terms left out would show: operands over the whole range of significands, those with the
    largest terms behind the first (next to 1 + 2^-7 and 1 + 2^-8) among them."""
    from bittorch_amd import _C
    n, k = 260, 520
    announce("fp32 weight gradient, few rows", m)
    g = torch.Generator("cuda").manual_seed(m)
    values = lambda *s: torch.where(torch.rand(*s, generator=g, device="cuda") < 0.5, 1 + torch.rand(*s, generator=g, device="cuda"),
                                    1 + torch.rand(*s, generator=g, device="cuda") * 2.0 ** -6)
    dy, x, scale = values(m, n), values(m, k), torch.rand(n, generator=g, device="cuda") + 0.5
    x[:, :4], dy[:, :4] = 1.0077972, 1.0077972
    for sign in (1.0, -1.0):
        dy[:, 1::2] *= sign
        _close(_C.linear_grad_weight(dy, x, scale)[0], dy.t(), x, _six_terms(m), scale.double()[:, None])


@gpu
def test_weight_gradient_of_the_largest_values():
    """Next to the largest float, where an operand's first term or a product of terms is an infinity and the product is not."""
    from bittorch_amd import _C
    announce("fp32 weight gradient, largest values")
    m, n, k, top = 40, 36, 68, 3.4028234663852886e38
    dy, x, scale = torch.zeros(m, n, device="cuda"), torch.zeros(m, k, device="cuda"), torch.ones(n, device="cuda")
    dy[3], x[3] = 1.0, 1.0
    dy[3, 5], x[3, 7] = top, -top * (1 - 2.0 ** -12)       # beyond the largest bf16 value
    dy[3, 9], x[3, 11] = 1.9985 * 2.0 ** 63, 1.9985 * 2.0 ** 63  # (their first terms are 2^64)
    got = _C.linear_grad_weight(dy, x, scale)[0].double()
    want = (dy.double().t() @ x.double())
    want[want.abs() > top] *= float("inf")
    fin = torch.isfinite(want)
    assert torch.equal(got[~fin], want[~fin]) and bool(((got - want)[fin].abs() <= 2.0 ** -24 * want[fin].abs()).all())


@gpu
@pytest.mark.parametrize("per_channel", [True, False])
@pytest.mark.parametrize("m,n,k", [(300, 64, 96), (7, 100, 96), (16384, 100, 256), (1000, 1100, 640), (130, 4128, 516)])
def test_fp32_gradients_of_non_finite_values(m, n, k, per_channel):
    """An infinity or NaN in the output gradient (an overflown loss) leaves what the fp32 products leave: the same
    elements non-finite, infinities with their sign, everything else untouched."""
    from bittorch_amd import _C
    announce("fp32 gradients, non-finite", m, n, k, per_channel)
    x, dy, packed, scale, tern = _case(m, n, k, per_channel)
    dy[1, 5], dy[m // 3, 11], dy[m // 2, 40], dy[5, n - 1] = float("inf"), float("-inf"), float("nan"), float("inf")
    dy[m - 1, 3] = torch.tensor(0x7F800001).int().view(torch.float32).cuda()  # (a NaN whose upper half is an infinity's)
    x[m // 4, 3] = float("inf")
    for got, ref in ((_C.linear_grad_input(dy, packed, scale, k), dy.double() @ (tern * scale[:, None]).double()),
                     (_C.linear_grad_weight(dy, x, scale)[0], (dy.double().t() @ x.double()) * scale.double()[:, None])):
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        inf = torch.isinf(ref)
        assert torch.equal(got[inf].double(), ref[inf]) and inf.any()
        fin = torch.isfinite(ref)
        assert torch.allclose(got[fin].double(), ref[fin], rtol=1e-4, atol=1e-5 * float(ref[fin].abs().max()))


@gpu
def test_non_finite_gradients_take_the_time_of_a_few_products():
    """A diverged step is no hundred times slower than the others (a tile is computed again, not element by element)."""
    from bittorch_amd import _C
    m, n, k = 4096, 768, 768
    announce("fp32 gradients, non-finite, time", m, n, k)
    x, dy, packed, scale, _ = _case(m, n, k)

    def microseconds(g):
        times = []
        for _ in range(7):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            _C.linear_grad_input(g, packed, scale, k)
            _C.linear_grad_weight(g, x, scale, True)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1e3)
        return sorted(times)[3]

    finite, nan = microseconds(dy), microseconds(torch.full_like(dy, float("nan")))
    assert nan < 12 * finite, (finite, nan)  # (element by element: 60 times)


@gpu
def test_fp32_layer_backward_uses_the_kernels_and_keeps_double_backward():
    from bittorch_amd import nn
    announce("fp32 layer backward")
    layer = nn.TernaryLinear(96, 40).cuda()
    x = torch.randn(70, 96, device="cuda", requires_grad=True)
    gy = torch.randn(70, 40, device="cuda")
    plain = torch.autograd.grad(layer(x), (x, layer.weight, layer.bias), gy)
    gy2 = gy.clone().requires_grad_()
    graphed = torch.autograd.grad(layer(x), (x, layer.weight, layer.bias), gy2, create_graph=True)
    for a, b in zip(plain, graphed):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5 * float(b.detach().abs().max()))
    assert torch.autograd.grad(graphed[0].sum(), gy2)[0].shape == gy.shape


@gpu
def test_fp32_layer_batched_gradients():
    """Several output gradients in one backward (``is_grads_batched=True``): as one backward each."""
    from bittorch_amd import nn
    announce("fp32 layer, batched gradients")
    layer = nn.TernaryLinear(96, 40).cuda()
    x = torch.randn(70, 96, device="cuda", requires_grad=True)
    y, leaves = layer(x), (x, layer.weight, layer.bias)
    gys = torch.randn(3, 70, 40, device="cuda")
    batched = torch.autograd.grad(y, leaves, gys, retain_graph=True, is_grads_batched=True)
    for i in range(3):
        for a, b in zip(batched, torch.autograd.grad(y, leaves, gys[i], retain_graph=True)):
            assert torch.allclose(a[i], b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))


@gpu
def test_generic_kernels_forced_in_the_backward(monkeypatch):
    """``BITTORCH_KERNEL=generic`` keeps the backward off the matrix-core kernels too: the torch products, bit for bit."""
    from bittorch_amd import _C, nn
    announce("fp32 layer backward, generic")
    monkeypatch.setenv("BITTORCH_KERNEL", "generic")
    for name in ("linear_grad_input", "linear_grad_weight", "scale_grad_weight"):
        monkeypatch.setattr(_C, name, None)
    layer = nn.TernaryLinear(96, 40).cuda()
    x, gy = torch.randn(70, 96, device="cuda", requires_grad=True), torch.randn(70, 40, device="cuda")
    gx, gw, gb = torch.autograd.grad(layer(x), (x, layer.weight, layer.bias), gy)
    packed, scale, _ = _C.ternary_quantize_pack(layer.weight.detach(), layer.threshold_factor, True)
    assert torch.equal(gx, gy @ _C.unpack_dequant(packed, 96, scale, torch.float32))
    assert torch.equal(gw, (gy.t() @ x.detach()) * scale[:, None]) and torch.equal(gb, gy.sum(0))
    with torch.autocast("cuda", dtype=torch.float16):
        y = layer(x)
    assert torch.autograd.grad(y, layer.weight, gy.half())[0].dtype == torch.float32


@gpu
@pytest.mark.parametrize("n", [1, 4, 7, 8, 9])
def test_input_gradient_of_few_outputs(n):
    """Of a layer with few outputs: up to 7 the product of exact factors, from 8 on each product may have a rounding of its own."""
    from bittorch_amd import _C, nn
    announce("fp32 layer backward, few outputs", n)
    g = torch.Generator("cuda").manual_seed(n)
    layer = nn.TernaryLinear(260, n, bias=False).cuda()
    x, gy = torch.ones(600, 260, device="cuda", requires_grad=True), torch.randn(600, n, generator=g, device="cuda")
    got = torch.autograd.grad(layer(x), x, gy)[0]
    packed, scale, tern = _C.ternary_quantize_pack(layer.weight.detach(), layer.threshold_factor, True, True, True)
    _close(got, gy, tern.float() * scale[:, None], _three_terms(n))
    if n < 8:
        assert torch.equal(got, gy @ _C.unpack_dequant(packed, 260, scale, torch.float32))


@gpu
@pytest.mark.parametrize("m,n,k", [(16384, 64, 100), (600, 1028, 260)])
def test_fp32_forward_without_a_workspace(m, n, k):
    """Through the C ABI with the scratch its query asks for, none: both weight layouts, on the kernel that splits in registers;
    the SwiGLU output stage and the prologues still have what they need."""
    from bittorch_amd import _C, _lib
    announce("fp32 forward, no workspace", m, n, k)
    lib = _lib.load()
    set_option("STREAM_MAX_ROWS", "1")
    x, _, packed, scale, tern = _case(m, n, k)
    assert lib.bt_packed_forward_workspace_bytes(m, n, k, 0) == 0
    tiled, stream = _C.retile_weights(packed, k), torch.cuda.current_stream().cuda_stream
    rows, tiles = (torch.full((m, n), float("nan"), device="cuda") for _ in range(2))
    assert lib.bt_ternary_linear_packed_forward(x.data_ptr(), 0, packed.data_ptr(), scale.data_ptr(), 0, n, None, 0,
                                                rows.data_ptr(), m, n, k, None, 0, stream) == 0
    assert lib.bt_ternary_linear_tiled_forward(x.data_ptr(), k, 0, 0, None, 0, 0.0, tiled.data_ptr(), scale.data_ptr(), 0, n, None, 0,
                                               None, 0, tiles.data_ptr(), m, n, k, None, 0, stream) == 0
    for y in (rows, tiles):
        _close(y, x, tern.t(), _three_terms(k), scale.double()[None, :])
    assert torch.equal(rows, _C.ternary_linear_packed_forward(x, packed, scale, None, k))
    if n % 32 == 0:
        gu = _C.ternary_linear_packed_forward(x, packed, scale, None, k)
        pairs = _C.retile_weights(packed, k, True)
        h = _C.ternary_linear_tiled_forward(x, pairs, scale, None, k, n, swiglu_pairs=True)
        want = torch.nn.functional.silu(gu[:, :n // 2]) * gu[:, n // 2:]
        assert torch.allclose(h, want, rtol=1e-4, atol=1e-5)
    norm = _C.ternary_linear_tiled_forward(x, tiled, scale, None, k, n, norm=(None, 1e-5))
    xn = torch.nn.functional.rms_norm(x, (k,), None, 1e-5)
    assert torch.allclose(norm, (xn.double() @ (tern.double() * scale.double()[:, None]).t()).float(), rtol=1e-4, atol=1e-5)


@gpu
@pytest.mark.parametrize("m,n,k", [(33700, 250, 200), (33792, 120, 196), (49000, 256, 232), (34000, 510, 254), (49000, 120, 256),
                                   (49000, 118, 256), (49000, 256, 118)])
def test_fp32_remainder_tiles_shared_by_workgroups(m, n, k):
    """33 tiles of 128 x 256 an XCD leave one, 48 leave sixteen: each is shared by four or two workgroups of 32 or 64 rows.  Rows that
    end inside the last tile, the right half of the columns past the end (forward and input gradient, both numbers of workgroups,
    N % 4 != 0 too), a partial step."""
    from bittorch_amd import _C
    announce("fp32 remainder tiles", m, n, k)
    x, dy, packed, scale, tern = _case(m, n, k)
    _close(_C.linear_grad_input(dy, packed, scale, k), dy, tern * scale[:, None], _three_terms(n))
    for y in (_C.ternary_linear_packed_forward(x, packed, scale, None, k),
              _C.ternary_linear_tiled_forward(x, _C.retile_weights(packed, k), scale, None, k, n)):
        _close(y, x, tern.t(), _three_terms(k), scale.double()[None, :])
    bad = dy.clone()
    bad[m - 1, 0], bad[5, n - 1], bad[m // 2, 1] = float("inf"), float("nan"), float("-inf")
    got, want = _C.linear_grad_input(bad, packed, scale, k), (bad * scale) @ tern
    rows = [m - 1, 5, m // 2]
    for r in rows:
        assert torch.equal(got[r].isnan(), want[r].isnan()) and torch.equal(got[r].isinf(), want[r].isinf())
    assert torch.isfinite(got[[0, 6, m - 2]]).all()


@gpu
@pytest.mark.parametrize("m,n,k", [(33792, 120, 224), (49000, 256, 232), (49000, 118, 256), (16384, 768, 768)])
def test_fp32_rows_are_summed_alike_wherever_they_lie(m, n, k):
    """Equal rows of a call have equal bits, in tiles of their own and in shared ones, forward and input gradient."""
    from bittorch_amd import _C
    announce("fp32 equal rows", m, n, k)
    x, dy, packed, scale, _ = _case(m, n, k)
    place = torch.arange(m, device="cuda") % 8
    x, dy = x[:8][place].contiguous(), dy[:8][place].contiguous()
    for y in (_C.linear_grad_input(dy, packed, scale, k), _C.ternary_linear_packed_forward(x, packed, scale, None, k),
              _C.ternary_linear_tiled_forward(x, _C.retile_weights(packed, k), scale, None, k, n)):
        assert torch.equal(y, y[:8][place])
