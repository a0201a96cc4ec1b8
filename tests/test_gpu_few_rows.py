"""The kernel for a few tens of rows (few_rows.hip): 16-bit rows from 33 on, int8 rows in operand order."""
import pytest
import torch

from conftest import announce
from _util import set_option

pytestmark = pytest.mark.gpu
TILES = ["2,2", "2,4", "3,4", "4,4", "5,4"]


def _case(m, n, k, dtype, pairs=False):
    from bittorch_amd import _C
    g = torch.Generator("cuda").manual_seed(m * 7 + n * 3 + k)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    packed, scale, tern = _C.ternary_quantize_pack(r(n, k) * 0.02, 0.05, True, True, True)
    return r(m, k).to(dtype), packed, scale, tern.double(), r(n) * 0.1, r(m, n).to(dtype)


def _bound(x, tern, scale, bias, dtype):
    """|sum| off by a rounding of fp32 each for K products (in any order, parts added up), the scale and the bias, then one of the
    output's type: 2^-11 or 2^-8 of the value."""
    value = (x.double() @ tern.t()) * scale.double() + bias.double()
    mags = (x.double().abs() @ tern.abs().t()) * scale.double() + bias.double().abs()
    fp32 = (x.shape[1] + 12) * 2.0 ** -24 * mags
    return fp32 + 2.0 ** (-11 if dtype == torch.float16 else -8) * (value.abs() + fp32) + 2.0 ** -25  # (2^-25: half of fp16's smallest)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(33, 64, 64), (80, 65, 8), (81, 48, 72), (47, 1030, 1000), (130, 100, 576), (64, 16, 4096), (100, 257, 640)])
def test_products_against_float64(m, n, k, tile):
    """Rows and columns that end inside a tile, a last tile of columns past the matrix, fewer steps than waves, one and two steps more
    than the loads that are on their way, a partial step."""
    from bittorch_amd import _C
    set_option("ROWS_CFG", tile)
    for dtype in (torch.float16, torch.bfloat16):
        announce("few rows", tile, m, n, k, dtype)
        x, packed, scale, tern, bias, res = _case(m, n, k, dtype)
        tiled = _C.retile_weights(packed, k)
        got = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
        err = (got.double() - ((x.double() @ tern.t()) * scale.double() + bias.double())).abs()
        assert bool((err <= _bound(x, tern, scale, bias, dtype)).all()), float(err.max())
        assert torch.equal(_C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n, residual=res), got + res)
        if n % 4 == 0:  # row-major weights: the same sums
            assert torch.equal(_C.ternary_linear_packed_forward(x, packed, scale, bias, k, residual=res), got + res)
        assert torch.equal(_C.ternary_linear_tiled_forward(x, tiled, scale[:1], None, k, n),
                           _C.ternary_linear_tiled_forward(x, tiled, scale[:1].expand(n).contiguous(), None, k, n))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(33, 96, 100), (82, 160, 512), (64, 32, 1096)])
def test_gate_up_pairs(m, n, k, tile):
    """A pair-ordered copy read in natural order gives the natural copy's bits, and the SwiGLU output stage the SwiGLU kernel's;
    infinities and NaN stay in their rows (K = 100: rows that are padded)."""
    from bittorch_amd import _C
    set_option("ROWS_CFG", tile)
    for dtype in (torch.float16, torch.bfloat16):
        announce("few rows, pairs", tile, m, n, k, dtype)
        x, packed, scale, tern, bias, _ = _case(m, n, k, dtype)
        x[1, k - 1], x[m - 1, 0], x[2] = float("inf"), float("nan"), x[2] * 500
        natural, pairs = _C.retile_weights(packed, k), _C.retile_weights(packed, k, True)
        want = _C.ternary_linear_tiled_forward(x, natural, scale, bias, k, n)
        got = _C.ternary_linear_tiled_forward(x, pairs, scale, bias, k, n, natural_from_pairs=True)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        assert bool(torch.isfinite(want[[0] + list(range(3, m - 1))]).all()) and bool((~torch.isfinite(want[1])).all())
        h, ref = _C.ternary_linear_tiled_forward(x, pairs, scale, bias, k, n, swiglu_pairs=True), _C.swiglu(want[:, :n // 2], want[:, n // 2:])
        assert bool(((h == ref) | (h.isnan() & ref.isnan())).all())


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (2, 100, 192), (17, 64, 144), (33, 257, 80), (47, 1028, 1024), (80, 48, 16), (81, 160, 1168),
                                   (130, 96, 2064)])
def test_int8_accumulators_and_outputs(m, n, k):
    """The exact integers and the streaming kernel's outputs, bit for bit, on tiled and on row-major weights: rows and columns that end
    inside a tile, fewer steps than waves, K of half a step more, every output type, residual."""
    from bittorch_amd import _C
    x, packed, scale, tern, bias, res = _case(m, n, k, torch.bfloat16)
    tiled = _C.retile_weights(packed, k)
    q, sx = _C.act_quant_int8(x)
    qo, _ = _C.act_quant_int8(x, operand_order=True)
    want_acc = 127 * (q.cpu().double() @ tern.cpu().t()).to(torch.int32)
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        for r in (None, res.to(dtype)):
            set_option("ROWS_CFG", None)
            set_option("STREAM_MAX_ROWS", "2000000")
            want, acc = _C.ternary_gemm_int8_tiled(qo, sx, tiled, scale, bias, k, n, dtype, True, r, True)
            assert torch.equal(acc.cpu(), want_acc)
            set_option("STREAM_MAX_ROWS", None)
            for tile in ("1,4", "2,4", "3,4", "4,4", "5,4"):
                announce("few int8 rows", tile, m, n, k, dtype)
                set_option("ROWS_CFG", tile)
                for y, a in (_C.ternary_gemm_int8_tiled(qo, sx, tiled, scale, bias, k, n, dtype, True, r, True),
                             _C.ternary_gemm_int8(qo, sx, packed, scale, bias, k, dtype, True, r, True)):
                    assert torch.equal(a.cpu(), want_acc) and torch.equal(y, want)


@pytest.mark.parametrize("m,n,k", [(3, 64, 100), (40, 128, 8), (70, 64, 1290), (16, 7680, 130)])
def test_int8_rows_that_are_padded(m, n, k):
    """K that is no multiple of 16: rows of Q longer than the weights' K, on row-major weights whose last rows then do not exist."""
    from bittorch_amd import _C
    x, packed, scale, _, bias, _ = _case(m, n, k, torch.bfloat16)
    set_option("STREAM_MAX_ROWS", "2000000")
    want = _C.ternary_linear_tensor_core_forward(x, packed, scale, bias, k, 2)
    set_option("STREAM_MAX_ROWS", None)
    for tile in ("1,4", "2,4", "5,4"):
        announce("few padded int8 rows", tile, m, n, k)
        set_option("ROWS_CFG", tile)
        assert torch.equal(_C.ternary_linear_tensor_core_forward(x, packed, scale, bias, k, 2), want)


@pytest.mark.parametrize("m,n,k,here", [(77, 7680, 2560, True), (64, 2560, 2560, True), (128, 7680, 2560, True), (192, 16384, 1024, False), (2048, 512, 11008, False)])
def test_choice_by_size(m, n, k, here):
    """From 33 rows on the forward's results are this kernel's where it is the cheaper one, and not the tiled GEMM's, which sums in another
    order (its tiles all have the same bits, and so has the streaming kernel on eight waves: not told apart here); up to 32 rows the
    row-major weights'.  The last: rows that no L2 holds."""
    from bittorch_amd import _C
    announce("few rows, choice", m, n, k)
    x, packed, scale, _, bias, _ = _case(m, n, k, torch.bfloat16)
    tiled = _C.retile_weights(packed, k)
    got = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
    assert torch.equal(_C.ternary_linear_tiled_forward(x[:32], tiled, scale, bias, k, n), _C.ternary_linear_packed_forward(x[:32], packed, scale, bias, k))
    for option, value, same in (("ROWS_CFG", "3,4", here), ("STREAM_MAX_ROWS", "1", not here)):
        set_option(option, value)
        assert torch.equal(got, _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)) == same
        set_option(option, None)


def test_more_rows_than_its_grid_has_blocks():
    """65535 blocks of 32 rows and a few rows more: served by a kernel that slices such a call, whatever ROWS_CFG asks for."""
    from bittorch_amd import _C
    m, n, k = 65535 * 32 + 17, 64, 16
    x, packed, scale, tern, bias, _ = _case(m, n, k, torch.bfloat16)
    tiled = _C.retile_weights(packed, k)
    want, bound = (x.double() @ tern.t()) * scale.double() + bias.double(), _bound(x, tern, scale, bias, torch.bfloat16)
    for option in (None, "2,2"):
        announce("few rows, tall", option, m, n, k)
        set_option("ROWS_CFG", option)
        got = _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n)
        assert bool(((got.double() - want).abs() <= bound).all())
