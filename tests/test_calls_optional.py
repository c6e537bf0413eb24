"""The native call path (_calls.so) only saves host time: without it, or with one built for another
torch or Python, the library loads all the same and every op is left to ctypes."""
import importlib.util
import os
import sys
import types

import pytest

import tileinfer_hip as ti
from tileinfer_hip import _lib


@pytest.fixture
def calls():
    ti.load_library()
    was = _lib.calls
    yield
    _lib.calls = was


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(built_for="torch 1.0.0, Python 3.9", bind=None)])
def test_load_without_native_calls(calls, monkeypatch, module):
    monkeypatch.setitem(sys.modules, "tileinfer_hip._calls", module)
    monkeypatch.setattr(sys.modules["tileinfer_hip"], "_calls", module, raising=False)
    if module is None:
        monkeypatch.delattr(sys.modules["tileinfer_hip"], "_calls")
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        L = _lib.load()
    assert L.ti_version().startswith(b"tileinfer_hip")
    n = _lib.native()
    assert {n.attention(), n.attention_inputs(), n.store_kv(), n.rope(), n.rmsnorm()} == {-1}


def test_build_without_torch(tmp_path, monkeypatch):
    """No torch: _calls.so is left out (and an older one removed), nothing raises."""
    src = os.path.join(os.path.dirname(_lib.HERE), "build.py")
    spec = importlib.util.spec_from_file_location("ti_build_test", src)
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    stale = tmp_path / "_calls.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "CALLS", str(stale))
    monkeypatch.setitem(sys.modules, "torch", None)
    assert build._build_calls() is False
    assert not stale.exists()
