"""GPU parity: the float forwards on sizes that fit no vector width: rows that start on any element, any number of columns,
activations that start anywhere, on both weight layouts, against float64."""
import pytest
import torch

from conftest import announce
from _util import random_ternary, seeded_acts

pytestmark = pytest.mark.gpu

_HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}

# rows of less than, exactly and just over a group of 8 values, a step of 32 / 64; columns around 4, a tile of 16, 64 and 256;
# rows around the streaming kernel's 16 and the tiled GEMMs' 32 / 64 / 128; sizes below and above the one that re-tiles weights
SHAPES = [(1, 5, 7), (1, 2049, 1031), (2, 4, 9), (16, 6, 24), (17, 255, 40), (33, 257, 63), (33, 260, 65), (37, 2050, 1047),
          (130, 259, 1029), (129, 1023, 1040), (300, 2051, 1040), (700, 2052, 1033), (1030, 1026, 2055), (40, 513, 8201), (1, 4098, 4112), (5, 4097, 4111), (20, 2050, 4103), (3, 131, 4103)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_float_forward_on_any_size(m, n, k):
    from bittorch_amd import _C
    announce("float forward, ragged", m, n, k)
    w = random_ternary(n, k, seed=n + k).cuda()
    w_t = _C.pack_ternary_int8(w)
    tiled = _C.retile_weights(w_t, k)
    assert torch.equal(_C.untile_weights(tiled, n, k), w_t)
    g = torch.Generator().manual_seed(m)
    scale, bias = (torch.rand(n, generator=g) * 0.02 + 0.001).cuda(), torch.randn(n, generator=g).cuda()
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        x = seeded_acts(m, k, seed=m + n + k, dtype=dtype).cuda()
        res = seeded_acts(m, n, seed=7, dtype=dtype).cuda()
        xo = torch.empty(m * k + 1, dtype=dtype, device="cuda")[1:].view(m, k).copy_(x)
        lin = x.double() @ w.double().t() * scale.double() + bias.double()
        # the output's rounding, and fp32 sums of K terms of any order: K half-ulps of the sum of magnitudes
        size = (x.double().abs() @ w.double().abs().t()) * scale.double() + bias.double().abs()
        bound = _HALF_ULP[dtype] * 1.01 * lin.abs() + (k + 4) * 2.0 ** -24 * size
        got = {"rows": _C.ternary_linear_packed_forward(x, w_t, scale, bias, k),
               "rows, off": _C.ternary_linear_packed_forward(xo, w_t, scale, bias, k),
               "tiles": _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n),
               "tiles, off": _C.ternary_linear_tiled_forward(xo, tiled, scale, bias, k, n)}
        for name, y in got.items():
            assert bool(((y.double() - lin).abs() <= bound).all()), (dtype, name)
        # with a residual: the same sums, one rounding more
        for y, yr in ((got["rows"], _C.ternary_linear_packed_forward(x, w_t, scale, bias, k, res)),
                      (got["tiles"], _C.ternary_linear_tiled_forward(x, tiled, scale, bias, k, n, res))):
            assert torch.equal(yr, y + res), dtype


@pytest.mark.parametrize("m,n,k", [(37, 2050, 1047), (300, 2051, 1040), (300, 259, 1029)])
def test_nothing_is_written_beside_ragged_outputs_and_no_workspace_is_needed(m, n, k):
    from bittorch_amd import _C
    announce("float forward, ragged, guards", m, n, k)
    w_t = _C.pack_ternary_int8(random_ternary(n, k, seed=n + k).cuda())
    scale = torch.full((n,), 0.01, device="cuda")
    for dtype, tag in ((torch.float32, 0), (torch.float16, 1), (torch.bfloat16, 2)):
        x = seeded_acts(m, k, seed=3, dtype=dtype).cuda()
        want = _C.ternary_linear_packed_forward(x, w_t, scale, None, k)
        full = _C._L.bt_packed_forward_workspace_bytes(m, n, k, tag)
        for nbytes in (full, 0):
            y = torch.full((m * n + 64,), -3.0, dtype=dtype, device="cuda")
            ws = torch.full((nbytes + 256,), 0x5A, dtype=torch.uint8, device="cuda")
            assert _C._L.bt_ternary_linear_packed_forward(
                x.data_ptr(), tag, w_t.data_ptr(), scale.data_ptr(), 0, n, None, 0, y[32:].data_ptr(), m, n, k,
                ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream) == 0
            torch.testing.assert_close(y[32:-32].view(m, n), want, rtol=2e-2 if dtype != torch.float32 else 1e-4, atol=1e-2)
            assert (y[:32] == -3).all() and (y[-32:] == -3).all() and (ws[nbytes:] == 0x5A).all()
