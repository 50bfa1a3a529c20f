"""Building the library and its native operator binding, without a device."""

import importlib.util
from types import SimpleNamespace

import pytest

from conftest import ROOT


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
