"""The native extension's loading and building, on the CPU: what is there but
does not fit leaves the ctypes path in place, and the C-ABI library does not
depend on it."""

import subprocess
import sys
import types
from pathlib import Path

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


class _Proc:
    def __init__(self, cmd, fails, **kw):
        self.returncode = int(fails(cmd))
        if not self.returncode:
            Path(cmd[cmd.index("-o") + 1]).write_bytes(b"built")

    def communicate(self):
        return "", "c10/hip headers are missing"


def _fake_build(monkeypatch, out, fails=lambda cmd: False):
    cmds = []

    def start(cmd, **kw):
        cmds.append(cmd)
        return _Proc(cmd, fails, **kw)

    def run(cmd, cwd=None):
        kbuild._wait(cmd, start(cmd))

    monkeypatch.setattr(kbuild.subprocess, "Popen", start)
    monkeypatch.setattr(kbuild, "_run", run)
    kbuild.build(out_dir=out)
    return cmds


def test_library_is_in_place_when_the_extension_does_not_compile(monkeypatch, tmp_path):
    stale = tmp_path / "_attnres_torch.so"
    stale.write_bytes(b"an earlier build")
    with pytest.raises(RuntimeError, match="headers are missing"):
        _fake_build(monkeypatch, tmp_path, lambda cmd: any("attnres_torch.cpp" in str(c) for c in cmd))
    assert (tmp_path / kbuild.LIB_NAME).read_bytes() == b"built"
    assert not stale.exists()


@pytest.mark.parametrize("torch_there", ["cpu-only", "none"])
def test_library_needs_no_rocm_torch(monkeypatch, tmp_path, torch_there):
    (tmp_path / kbuild.NATIVE_NAME).write_bytes(b"an earlier build")
    if torch_there == "none":
        monkeypatch.setitem(sys.modules, "torch", None)  # import torch fails
    else:
        monkeypatch.setattr(torch.version, "hip", None)
    cmds = _fake_build(monkeypatch, tmp_path)
    assert [p.name for p in tmp_path.iterdir()] == [kbuild.LIB_NAME]
    assert not any("attnres_torch" in str(c) for cmd in cmds for c in cmd)


def test_extension_is_built_for_this_torch_and_python(monkeypatch, tmp_path):
    if torch.version.hip is None:
        pytest.skip("not a ROCm torch")
    cmds = _fake_build(monkeypatch, tmp_path)
    assert (tmp_path / kbuild.NATIVE_NAME).read_bytes() == b"built"
    (compile_cmd,) = [c for c in cmds if any("attnres_torch.cpp" in a for a in c)]
    assert f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}" in compile_cmd
    assert f'-DATTNRES_TORCH_VERSION="{torch.__version__}"' in compile_cmd
