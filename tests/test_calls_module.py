"""Building and loading the module of native calls where torch, Python's headers or the module itself are missing, or are others than it
was built for: everything else builds and every call still works, through ctypes."""
import importlib.util
import os

import pytest


@pytest.fixture
def capi(monkeypatch):
    from inferspore_amd import capi
    capi.lib()
    monkeypatch.setattr(capi, "_calls", None)
    return capi


def _left_to_ctypes(capi):
    with pytest.warns(RuntimeWarning, match="through ctypes"):
        calls = capi.calls()
    assert calls.rmsnorm(None, None, 1e-5) is None and calls.context_layer() is None
    assert capi.calls() is calls   # said once


def test_the_module_that_is_built_loads(capi):
    import torch
    assert capi.calls().built_for[0] == torch.__version__
    assert capi.calls().rmsnorm(torch.zeros(2, 8), torch.zeros(8), 1e-5) is None   # not on the GPU: left to the general path


def test_without_the_module(capi, monkeypatch, tmp_path):
    monkeypatch.setattr(capi, "CALLS_PATH", str(tmp_path / "_torch_calls.so"))
    _left_to_ctypes(capi)


def test_with_one_that_does_not_load(capi, monkeypatch, tmp_path):
    path = tmp_path / "_torch_calls.so"
    path.write_bytes(b"no library")
    monkeypatch.setattr(capi, "CALLS_PATH", str(path))
    _left_to_ctypes(capi)


def test_with_one_for_another_torch(capi, monkeypatch):
    import torch
    monkeypatch.setattr(torch, "__version__", "1.0")
    _left_to_ctypes(capi)


@pytest.mark.parametrize("missing", ["torch", "ATen.h", "libc10_hip.so", "Python.h"])
def test_building_without(missing, monkeypatch, tmp_path):
    from inferspore_amd import build
    stale = tmp_path / "_torch_calls.so"
    stale.write_bytes(b"of another torch")
    monkeypatch.setattr(build, "CALLS", str(stale))
    monkeypatch.setattr(build, "_run", lambda cmd: pytest.fail("compiles without " + missing))
    if missing == "torch":
        find = importlib.util.find_spec
        monkeypatch.setattr(importlib.util, "find_spec", lambda name, *a: None if name == "torch" else find(name, *a))
    else:
        exists = os.path.exists
        monkeypatch.setattr(os.path, "exists", lambda p: not str(p).endswith(missing) and exists(p))
    build._compile_calls()
    assert not os.path.lexists(str(stale))
