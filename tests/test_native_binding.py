"""Loading and building the native operator binding, without a device."""

import importlib.util
import sys
from types import SimpleNamespace

import pytest
import torch

from conftest import ROOT
from kvx import _lib


def bind_with(monkeypatch, module):
    """_lib.bind() where importing kvx._bind gives `module` (None: not built)."""
    monkeypatch.setitem(sys.modules, "kvx._bind", module)
    monkeypatch.setattr(_lib, "_bind", None)
    return _lib.bind()


def test_the_built_binding_matches_the_library_and_this_torch():
    module = _lib.load_bind()
    assert (module.ABI_VERSION, module.TORCH_VERSION) == (_lib.ABI_VERSION, torch.__version__)


def test_operators_run_through_ctypes_without_a_binding(monkeypatch):
    with pytest.warns(RuntimeWarning, match="ctypes"):
        binding = bind_with(monkeypatch, None)
    assert binding.store() is None and binding.codec() is None and binding.blocks() is None
    assert _lib.bind() is binding  # one warning only


def test_a_binding_of_another_torch_is_not_used(monkeypatch):
    other = SimpleNamespace(ABI_VERSION=_lib.ABI_VERSION, TORCH_VERSION="0.0")
    with pytest.warns(RuntimeWarning, match="built for torch 0.0"):
        assert bind_with(monkeypatch, other).store() is None


def test_a_binding_of_another_libkvx_is_refused(monkeypatch):
    other = SimpleNamespace(ABI_VERSION=_lib.ABI_VERSION - 1, TORCH_VERSION=torch.__version__)
    with pytest.raises(RuntimeError, match="ABI"):
        bind_with(monkeypatch, other)


def test_a_failed_build_leaves_the_pair_that_was_there(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("kvx_build_test", ROOT / "kv-cache-offloading_amd" / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    monkeypatch.setattr(build, "OUTPUT", tmp_path / "libkvx.so")
    monkeypatch.setattr(build, "BIND_OUTPUT", tmp_path / "_bind.so")
    for output in (build.OUTPUT, build.BIND_OUTPUT):
        output.write_text("old")
    fails = []

    def compiler(cmd, **kwargs):
        if cmd[0] in fails:
            return SimpleNamespace(returncode=1, stdout="", stderr="")
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")
        return SimpleNamespace(returncode=0, stdout="", stderr="")

    monkeypatch.setattr(build.subprocess, "run", compiler)
    fails.append("g++")
    with pytest.raises(RuntimeError, match="failed"):
        build.build()
    assert [p.read_text() for p in (build.OUTPUT, build.BIND_OUTPUT)] == ["old", "old"]
    fails.clear()
    build.build()
    assert [p.read_text() for p in (build.OUTPUT, build.BIND_OUTPUT)] == ["new", "new"]
