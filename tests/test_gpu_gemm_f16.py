"""GPU: the tiled 16-bit GEMM (``csrc/gemm_f16.hip``) against float64 at the edges of its tiles and stages.

Rows 128 / 64 / 32 a tile and 256 columns, the last round of a launch in halves or quarters of tiles (bit for bit the sums of
tiles of 128 rows); stages of 64 k with a remainder of any
multiple of 8, fewer stages than are in flight; row-major weights with N a multiple of 16 and of 4 only, and the tiled copy.
The products are exact and summed in fp32: the error before the output's rounding is at most (K + 8) 2^-24 of the sum of the
products' magnitudes, the scale and the output round once each.
"""
import pytest
import torch

from conftest import announce
from _util import random_ternary, set_option

pytestmark = pytest.mark.gpu

SHAPES = [(33, 260, 64), (40, 1000, 8), (70, 1028, 200), (129, 4096, 336), (999, 2564, 1032), (2000, 1296, 120),
          (1025, 16388, 72), (4111, 4356, 264), (8200, 2304, 328), (4100, 5380, 136)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiled_float_gemm_against_float64(m, n, k, dtype):
    from bittorch_amd import _C
    announce("gemm_f16", m, n, k, dtype)
    set_option("STREAM_MAX_ROWS", "1")
    g = torch.Generator("cuda").manual_seed(m + n + k)
    w = random_ternary(n, k, seed=m).cuda()
    wt = _C.ternary_quantize_pack(w.float(), 0.05, True)[0]  # (the entries are -1, 0, 1: kept as they are)
    tiled = _C.retile_weights(wt, k)
    w = torch.where(w.abs().amax(1, keepdim=True) > 0, w, 0).double()
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    scale = torch.rand(n, generator=g, device="cuda") + 0.5
    res = torch.randn(m, n, generator=g, device="cuda").to(dtype)
    ref = (x.double() @ w.t()) * scale.double()
    mags = (x.double().abs() @ w.t().abs()) * scale.double()
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for r in (None, res):
        set_option("GEMM_TAIL_SPLIT", None)
        y = _C.ternary_linear_packed_forward(x, wt, scale, None, k, residual=r)
        yt = _C.ternary_linear_tiled_forward(x, tiled, scale, None, k, n, residual=r)
        assert torch.equal(y, yt)
        set_option("GEMM_TAIL_SPLIT", "0")
        assert torch.equal(_C.ternary_linear_packed_forward(x, wt, scale, None, k, residual=r), y)
        want = ref if r is None else ref + r.double()
        bound = (k + 8) * 2.0 ** -24 * mags + unit * (want.abs() + (0 if r is None else ref.abs())) + 2e-7
        assert bool(((y.double() - want).abs() <= bound).all())


def test_infinities_past_the_end_of_a_row_stay_in_their_row():
    """K not a multiple of the stage: what lies behind a row's end is the next row, and must not reach it."""
    from bittorch_amd import _C
    m, n, k = 200, 256, 72
    announce("gemm_f16 tail", m, n, k)
    set_option("STREAM_MAX_ROWS", "1")
    w = torch.ones(n, k, device="cuda")
    wt = _C.ternary_quantize_pack(w, 0.05, True)[0]
    x = torch.ones(m, k, device="cuda", dtype=torch.float16)
    x[7, 0], x[9, 64], x[150, 71] = float("inf"), float("nan"), float("-inf")
    scale = torch.ones(n, device="cuda")
    for y in (_C.ternary_linear_packed_forward(x, wt, scale, None, k),
              _C.ternary_linear_tiled_forward(x, _C.retile_weights(wt, k), scale, None, k, n)):
        assert bool((y[7] == float("inf")).all()) and bool(y[9].isnan().all()) and bool((y[150] == float("-inf")).all())
        rest = torch.ones(m, dtype=torch.bool)
        rest[[7, 9, 150]] = False
        assert bool((y[rest.cuda()] == k).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(33, 260, 1536), (97, 1004, 1544), (250, 516, 1480), (640, 5000, 1608), (129, 1024, 2112), (70, 1030, 1800),
                                   (129, 1024, 1608), (300, 4096, 1576)])
def test_stages_in_two_groups(m, n, k, dtype):
    """Launches of at most one tile a compute unit, 24 stages and more: an even and an odd number of stages, a remainder of K in the
    second group, rows that end in either group's half of a tile, tiles of 32 and 64 rows, N % 4 != 0; N % 16 == 0 (row-major weights
    16 bytes a lane) with a remainder of K.  Bound as above."""
    from bittorch_amd import _C
    announce("gemm_f16 two groups", m, n, k, dtype)
    set_option("STREAM_MAX_ROWS", "1")
    g = torch.Generator("cuda").manual_seed(m + n + k)
    w = random_ternary(n, k, seed=m).cuda()
    wt = _C.ternary_quantize_pack(w.float(), 0.05, True)[0]
    tiled = _C.retile_weights(wt, k)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    scale = torch.rand(n, generator=g, device="cuda") + 0.5
    res = torch.randn(m, n, generator=g, device="cuda").to(dtype)
    w = w.double()
    ref = (x.double() @ w.t()) * scale.double()
    mags = (x.double().abs() @ w.t().abs()) * scale.double()
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for r in (None, res):
        want = ref if r is None else ref + r.double()
        bound = (k + 8) * 2.0 ** -24 * mags + unit * (want.abs() + (0 if r is None else ref.abs())) + 2e-7
        y = _C.ternary_linear_packed_forward(x, wt, scale, None, k, residual=r)
        yt = _C.ternary_linear_tiled_forward(x, tiled, scale, None, k, n, residual=r)
        assert torch.equal(y, yt)
        assert bool(((y.double() - want).abs() <= bound).all())
