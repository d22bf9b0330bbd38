"""The native extension's loading, on the CPU: what is there but does not fit
leaves the ctypes path in place."""

import subprocess
import types

import pytest
import torch

from kotodama_amd import _native
from kotodama_amd import build as kbuild


def _lookup(monkeypatch, path):
    monkeypatch.setattr(_native, "PATH", path)
    return _native._Native()


def test_absent_extension_leaves_the_calls_to_python(monkeypatch, tmp_path, recwarn):
    native = _lookup(monkeypatch, tmp_path / "none.so")
    assert all(getattr(native, fn)(1, 2) is None for fn in _native.FUNCTIONS)
    assert not recwarn.list
    with pytest.raises(AttributeError):
        native.other


@pytest.mark.parametrize("content", [b"", b"\x7fELF truncated", None], ids=["empty", "truncated", "no-module"])
def test_unloadable_extension_leaves_the_calls_to_python(monkeypatch, tmp_path, content):
    path = tmp_path / "_attnres_torch.so"
    if content is None:  # a shared object without the module's entry, as one built for another interface
        subprocess.run(["gcc", "-shared", "-x", "c", "-", "-o", str(path)], input=b"int unused;", check=True)
    else:
        path.write_bytes(content)
    native = _lookup(monkeypatch, path)
    with pytest.warns(RuntimeWarning, match="native call path is off"):
        assert native.route(1) is None
    assert native.merge(1) is None  # said once


def test_extension_of_another_torch_is_not_used(monkeypatch, tmp_path):
    path = tmp_path / "_attnres_torch.so"
    path.touch()

    class Loader:
        def __init__(self, name, where):
            pass

        def create_module(self, spec):
            return types.SimpleNamespace(torch_version="1.0", route=lambda *a: "native")

        def exec_module(self, mod):
            pass

    monkeypatch.setattr(_native.importlib.machinery, "ExtensionFileLoader", Loader)
    monkeypatch.setattr(_native.importlib.util, "module_from_spec", lambda spec: Loader("", "").create_module(spec))
    with pytest.warns(RuntimeWarning, match="built for torch 1.0"):
        assert _lookup(monkeypatch, path).route() is None


def test_names_agree_and_the_built_extension_loads(monkeypatch):
    assert kbuild.NATIVE_NAME == _native.NAME
    if not _native.PATH.exists():
        pytest.skip("the extension is not built")
    mod = _native._load(_native.PATH)
    assert mod.torch_version == torch.__version__
    assert all(callable(getattr(mod, fn)) for fn in _native.FUNCTIONS)
    assert mod.route(1, 2) is None  # not a call it takes
