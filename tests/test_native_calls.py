"""The native host side of the calls takes GPU tensors alone, and is bound to the library that is loaded."""
import torch

from bittorch_amd import _C, _lib


def test_cpu_tensors_and_wrong_arguments_are_left_to_python():
    x, w, s = torch.randn(2, 8), torch.zeros(2, 4, dtype=torch.uint8), torch.ones(4)
    n = _C._N
    assert n.packed_forward(x, w, s, None, 8) is None
    assert n.tensor_core_forward(x, w, s, None, 8) is None
    assert n.tiled_forward(x, w.reshape(-1), s, None, 8, 4, None, None, None, False, False) is None
    assert n.quantize_pack(torch.randn(4, 8), 0.05, True, False) is None
    assert n.grad_input(torch.randn(2, 4), w, s, 8) is None
    assert n.grad_weight(torch.randn(2, 4), x, s, True) is None
    assert n.grad_weight_16(torch.randn(2, 4).half(), x.half(), s, torch.float32) is None
    assert n.unpack_dequant(w, 8, s, torch.float32) is None
    assert n.rmsnorm_int8(x, None, 1e-5, False) is None
    assert n.swiglu_int8(x, x, False) is None
    assert n.gemm_i8_tiled(x.to(torch.int8), torch.ones(2), w.reshape(-1), s, None, 8, 4, torch.float32, None, False) is None
    for bad in ((), (None,) * 5, ("x", w, s, None, 8), (x, w, s, None, "8"), (x, w, s, None, 2 ** 70)):
        assert n.packed_forward(*bad) is None


def test_generic_kernel_is_read_on_every_call(monkeypatch):
    monkeypatch.setenv("BITTORCH_KERNEL", "generic")
    assert _C._N.generic_kernel_asked()
    monkeypatch.setenv("BITTORCH_KERNEL", "auto")
    assert not _C._N.generic_kernel_asked()
    monkeypatch.delenv("BITTORCH_KERNEL")
    assert not _C._N.generic_kernel_asked()


def test_bound_to_every_function_it_names():
    assert set(_C._N.names()) <= set(_lib.SIGNATURES)
