"""GPU: the tiled int8 GEMM on operand-order activations (``csrc/gemm_i8_dma.hip``), bit for bit against the kernel that reads
row-major activations and against exact integer sums, at the edges of its tiles and stages.

Rows 128 / 64 / 32 a tile and 256 columns, the last round of a launch in halves or quarters of tiles or whole; stages of 64 k (a remainder of 16, 32 or 48 in the last one), fewer stages than the
five in flight; a last row block that is partly or wholly past M; row-major, tiled and field-layout weights.
"""
import pytest
import torch

from conftest import announce
from _util import random_ternary, set_option

pytestmark = pytest.mark.gpu

SHAPES = [(33, 260, 64), (40, 1000, 48), (70, 1028, 208), (129, 4096, 336), (999, 2564, 1040), (2000, 1300, 112),
          (1025, 16388, 192), (4111, 4356, 320), (8200, 2304, 704), (4100, 5380, 256), (4111, 4356, 384)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_operand_order_equals_row_major_activations(m, n, k, dtype):
    from bittorch_amd import _C
    announce("gemm_i8 operand order", m, n, k, dtype)
    set_option("STREAM_MAX_ROWS", "1")
    g = torch.Generator("cuda").manual_seed(m + n + k)
    w = random_ternary(n, k, seed=m).cuda()
    wt = _C.ternary_quantize_pack(w.float(), 0.05, True)[0]  # (the entries are -1, 0, 1: kept as they are)
    tiled = _C.retile_weights(wt, k)
    x = torch.randn(m, k, generator=g, device="cuda")
    x[m // 2] = 0
    scale = torch.rand(n, generator=g, device="cuda") + 0.5
    bias = torch.randn(n, generator=g, device="cuda").to(dtype)
    res = torch.randn(m, n, generator=g, device="cuda").to(dtype)
    q, s = _C.act_quant_int8(x, False)
    qo, so, rowsum = _C.act_quant_int8(x, True, return_rowsum=True)
    fields = _C.retile_fields(tiled, k, n) if k % 128 == 0 else None
    s[m // 3] = so[m // 3] = 2.0 ** -125  # below the range of the two-operation division
    exact = (127 * (q.double() @ w.double().t())).int()
    for residual in (None, res):
        kw = dict(out_dtype=dtype, return_acc=True, residual=residual)
        y, acc = _C.ternary_gemm_int8(q, s, wt, scale, bias, k, **kw)
        yr, ar = _C.ternary_gemm_int8(qo, so, wt, scale, bias, k, q_operand_order=True, **kw)
        yt, at = _C.ternary_gemm_int8_tiled(qo, so, tiled, scale, bias, k, n, q_operand_order=True, **kw)
        assert torch.equal(acc, exact) and torch.equal(ar, exact) and torch.equal(at, exact)
        assert torch.equal(yr, y) and torch.equal(yt, y)
        if fields is not None:
            yf, af = _C.ternary_gemm_int8_fields(qo, so, rowsum, fields, scale, bias, k, n, q_operand_order=True, **kw)
            assert torch.equal(af, exact) and torch.equal(yf, y)
        set_option("GEMM_TAIL_SPLIT", "0")
        yw, aw = _C.ternary_gemm_int8(qo, so, wt, scale, bias, k, q_operand_order=True, **kw)
        set_option("GEMM_TAIL_SPLIT", None)
        assert torch.equal(aw, exact) and torch.equal(yw, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(33, 260, 1536), (97, 1004, 1552), (250, 516, 1584), (640, 5000, 1616), (129, 1024, 2112),
                                   (129, 1024, 1616), (300, 4096, 1584), (250, 516, 1664), (640, 5000, 1536), (1000, 2560, 6912)])
def test_stages_in_two_groups(m, n, k, dtype):
    """Launches of at most one tile a compute unit, 24 stages and more: even and odd numbers of stages, a remainder of K in the
    second group, rows that end in either group's half of a tile, tiles of 32 and 64 rows; N % 16 == 0 with a remainder of K; whole stages of
    128, where decode-tiled weights leave the other kernel for this one."""
    test_operand_order_equals_row_major_activations(m, n, k, dtype)
