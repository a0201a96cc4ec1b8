"""The native host side of the calls takes GPU tensors alone, and is bound to the library that is loaded; the package works
without it."""
import importlib.util
import os
import re
import types

import pytest
import torch

from bittorch_amd import _C, _lib, build


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


def test_tensors_are_read_under_the_interpreter_lock():
    """Between letting go of the lock and taking it back, by a destructor, there is the library's call with values alone."""
    source = open(os.path.join(build.CSRC, "calls.cpp")).read()
    assert source.count("PyEval_SaveThread") == source.count("PyEval_RestoreThread") == 1
    assert re.search(r"~(\w+)\(\) \{ PyEval_RestoreThread\(state\); \}", source)
    assert re.search(r"const Unlocked unlocked;\s+rc = f\(args\.\.\.\);\s+\}", source) and source.count("Unlocked unlocked") == 1
    assert not re.search(r"call\(\s*\[", source)  # (a lambda's body would run in there)


def test_bound_to_every_function_it_names():
    assert set(_C._N.names()) <= set(_lib.SIGNATURES)


def _another_c():
    """bittorch_amd._C, imported once more with what _lib loads now."""
    spec = importlib.util.spec_from_file_location("bittorch_amd._C_again", _C.__file__)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_the_package_works_without_it(monkeypatch, tmp_path):
    """Hidden, no shared object, of another ABI, of another torch: a warning that says so, and every call is left to Python."""
    assert _lib.load_calls().stamp() == f"abi {_lib.ABI_VERSION}, {_lib.calls_build()}"
    (tmp_path / "_calls.so").write_bytes(b"no shared object")
    for attr, value, why in (("CALLS_PATH", str(tmp_path / "none.so"), "is missing"), ("CALLS_PATH", str(tmp_path / "_calls.so"), "_calls"),
                             ("ABI_VERSION", _lib.ABI_VERSION + 1, "compiled against"),
                             ("calls_build", lambda: "torch 9.9.9 abc, python 3.10", "compiled against .*, not .*9.9.9")):
        with monkeypatch.context() as m:
            m.setattr(_lib, "_calls", None)
            m.setattr(_lib, attr, value)
            with pytest.warns(RuntimeWarning, match=why):
                again = _another_c()
            assert again._N.packed_forward(None) is None and again._N.generic_kernel_asked() is False
            m.setenv("BITTORCH_KERNEL", "generic")
            assert again._N.generic_kernel_asked() is True
            with pytest.raises(RuntimeError, match="CUDA"):  # the Python function's own answer
                again.ternary_linear_packed_forward(torch.randn(2, 8), torch.zeros(2, 4, dtype=torch.uint8), torch.ones(4), None, 8)
    assert _C._N is _lib.load_calls() and not isinstance(_C._N, _lib._PythonCalls)


def test_the_library_is_built_without_it(monkeypatch, tmp_path, capsys):
    """No g++: the library is finished, what is missing is said, and no earlier file stays in its place."""
    monkeypatch.setattr(build, "OUT_DIR", str(tmp_path))
    monkeypatch.setattr(build, "LIB_PATH", str(tmp_path / "libbittorch_hip.so"))
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    monkeypatch.setattr(build.subprocess, "run", lambda *a, **k: types.SimpleNamespace(returncode=0, stdout="", stderr=""))
    (tmp_path / "_calls.so").write_bytes(b"an earlier one")
    assert build.build() == str(tmp_path / "libbittorch_hip.so")
    assert "g++ not found" in capsys.readouterr().err and not (tmp_path / "_calls.so").exists()
    with pytest.raises(RuntimeError, match="g\\+\\+ not found"):
        build.build(need_calls=True)
