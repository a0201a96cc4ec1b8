"""GPU parity: the int8 matrix-core forward on sizes that fit no vector width (any rows, any columns, any K, operands that
start anywhere).  Sums of integers, one fp32 epilogue: bit for bit the result of the int8 GEMM on separately quantized rows."""
import numpy as np
import pytest
import torch

from conftest import announce
from _util import BT_DT, f32np, random_ternary, seeded_acts

pytestmark = pytest.mark.gpu

# K around a group of 8 or 16 and a stage of 64, N around a group of 4, a tile of 16 and of 256, rows around the streaming
# kernel's 16, and the tiled one's 32 / 64 / 128; shapes above and below the size from which weights are re-tiled
SHAPES = [(1, 2049, 1031), (5, 4, 8), (16, 6, 24), (17, 255, 40), (33, 257, 63), (33, 258, 65), (70, 1023, 1000), (130, 260, 1029),
          (129, 259, 4097), (300, 2051, 1040), (77, 2050, 1033), (2049, 1025, 2055), (64, 513, 8201), (5, 4098, 4104), (20, 2049, 4111), (40, 1537, 16384), (3, 131, 16391)]


def _oracle(oracle, x, w, scale, bias, dtype):
    q, s = oracle.act_quant_i8(f32np(x))
    acc = q.astype(np.int64) @ w.numpy().astype(np.int64).T * 127
    y = ((acc.astype(np.float32) * s[:, None]) / np.float32(127)) * scale.numpy()[None, :]
    y = y + bias.numpy()[None, :]
    return torch.from_numpy(y).to(dtype)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tensor_core_forward_on_any_size(oracle, m, n, k):
    from bittorch_amd import _C
    announce("tensor core, ragged", m, n, k)
    w = random_ternary(n, k, seed=n + k)
    w_t = _C.pack_ternary_int8(w.cuda())
    g = torch.Generator().manual_seed(m)
    scale, bias = torch.rand(n, generator=g) * 0.02 + 0.001, torch.randn(n, generator=g)
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        x = seeded_acts(m, k, seed=m + n + k, dtype=dtype, outliers=True)
        want = _oracle(oracle, x, w, scale, bias, dtype)
        got = _C.ternary_linear_tensor_core_forward(x.cuda(), w_t, scale.cuda(), bias.cuda(), k, version=2)
        assert torch.equal(got.cpu(), want), dtype
        # the same rows starting at an odd place, outputs with guards, and the smallest workspace that was ever enough
        xs = torch.empty(m * k + 1, dtype=dtype, device="cuda")
        xs[1:] = x.cuda().reshape(-1)
        least = -(-m * k // 256) * 256 + -(-m * 4 // 256) * 256
        for nbytes in (_C._L.bt_tensor_core_workspace_bytes(m, n, k), least):
            y = torch.full((m * n + 64,), -3.0, dtype=dtype, device="cuda")
            ws = torch.full((nbytes + 256,), 0x5A, dtype=torch.uint8, device="cuda")
            assert _C._L.bt_ternary_linear_tensor_core_forward(
                xs[1:].data_ptr(), BT_DT[dtype], w_t.data_ptr(), scale.cuda().data_ptr(), 0, n, bias.cuda().data_ptr(), 0,
                y[32:].data_ptr(), m, n, k, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
            assert torch.equal(y[32:-32].reshape(m, n).cpu(), want), (dtype, nbytes)
            assert (y[:32] == -3).all() and (y[-32:] == -3).all() and (ws[nbytes:] == 0x5A).all()


@pytest.mark.parametrize("m,n,k", [(130, 259, 1040), (300, 1030, 2048), (40, 2049, 512)])
def test_tiled_int8_gemm_with_residual_and_accumulators_on_any_columns(oracle, m, n, k):
    """What only the entry point on tiled weights has: int32 accumulators and a residual, rows of N % 4 != 0."""
    from bittorch_amd import _C
    announce("tiled int8 GEMM, ragged columns", m, n, k)
    w = random_ternary(n, k, seed=n + k)
    w_t = _C.pack_ternary_int8(w.cuda())
    tiled = _C.retile_weights(w_t, k)
    scale = (torch.rand(n, generator=torch.Generator().manual_seed(1)) * 0.02 + 0.001).cuda()
    for dtype in (torch.bfloat16, torch.float32):
        x = seeded_acts(m, k, seed=3, dtype=dtype).cuda()
        res = seeded_acts(m, n, seed=4, dtype=dtype).cuda()
        q, s = _C.act_quant_int8(x, operand_order=True)
        y, acc = _C.ternary_gemm_int8_tiled(q, s, tiled, scale, None, k, n, dtype, True, None, True)
        q_nat, _ = _C.act_quant_int8(x)
        assert torch.equal(acc.cpu().long(), 127 * (q_nat.cpu().double() @ w.double().t()).long())
        plain = _C.ternary_gemm_int8(q_nat, s, w_t, scale, None, k, dtype)
        assert torch.equal(y, plain)
        assert torch.equal(_C.ternary_gemm_int8_tiled(q, s, tiled, scale, None, k, n, dtype, False, res, True), plain + res)
