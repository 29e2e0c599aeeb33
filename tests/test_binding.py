"""The Python binding where its module csrc/py_call.cpp cannot be had: the calls then go through ctypes, and the library builds without
what only the module needs.  CPU only: what a call on host tensors is refused with shows the way it took."""
import os
import sys
import types

import pytest

torch = pytest.importorskip("torch")
import fastertnn_amd
import fastertnn_amd.build as build
import fastertnn_amd.lib as lib
from fastertnn_amd import TNN


def _calls_on_host_tensors():
    i, f = torch.zeros(64, dtype=torch.int64), torch.zeros((1, 64, 2, 2))
    thr, u = torch.zeros(1), torch.zeros(64, dtype=torch.uint8)
    yield lambda: lib.mm(TNN, i, i, 1, 1, 1, 1, 4, 0.5, out=f)
    yield lambda: lib.mm_engine(lib.ENGINE_AUTO, TNN, i, i, 1, 1, 1, 1, 4, 0.5, out=f, scratch=u)
    yield lambda: lib.mm_expanded(lib.ENGINE_MFMA_F4, TNN, u, u, 1, 1, 1, 1, 4, 0.5, out=f)
    yield lambda: lib.conv(TNN, f, thr, i, 64, 1, 1, 0, 1, 0.5, scratch=u, out=f)
    yield lambda: lib.conv_prepared(TNN, f, thr, u, 64, 1, 1, 0, 1, 0.5, scratch=u, out=f)
    yield lambda: lib.conv_static(TNN, f, thr, i, 64, 1, 1, 0, 1, 0.5, f)


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(torch_version="0.4")], ids=("missing", "of another torch"))
def test_calls_without_the_module(monkeypatch, module):
    monkeypatch.setattr(lib, "_call", None)
    monkeypatch.delattr(fastertnn_amd, "_call", raising=False)
    monkeypatch.setitem(sys.modules, "fastertnn_amd._call", module)
    if module is not None:
        monkeypatch.setattr(fastertnn_amd, "_call", module, raising=False)
    with pytest.warns(RuntimeWarning, match="through ctypes"):
        assert lib._native().conv() is None
    for call in _calls_on_host_tensors():
        with pytest.raises(AssertionError, match="contiguous CUDA"):
            call()


def test_the_module_is_of_this_torch():
    assert lib._native().torch_version == torch.__version__


@pytest.mark.parametrize("lacking", ("compiler", "torch", "headers"))
def test_library_builds_without_what_the_module_needs(monkeypatch, tmp_path, lacking):
    """the last step of the build then says so, and leaves no module of another library behind"""
    old = tmp_path / "_call.so"
    old.write_bytes(b"")
    monkeypatch.setattr(build, "BINDING", str(old))
    if lacking == "compiler":
        monkeypatch.setenv("CXX", "no-such-compiler -m64")
    elif lacking == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)
    else:
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build_binding() is None
    assert not os.path.exists(old)
