"""woq_call.so is an extra: the build and the package do without it wherever it cannot be built."""
import importlib.util
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture
def build(tmp_path, monkeypatch):
    """build.py with its outputs in a folder of their own, one translation unit and no compiler run but g++'s."""
    path = os.path.join(ROOT, "tensorrt-llm_amd", "build.py")
    spec = importlib.util.spec_from_file_location("woq_build_under_test", path)
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    monkeypatch.setattr(b, "HERE", str(tmp_path))
    monkeypatch.setattr(b, "OBJ", str(tmp_path / "build"))
    monkeypatch.setattr(b, "LIB", str(tmp_path / "libwoq.so"))
    monkeypatch.setattr(b, "_compile", lambda src: src + ".o")
    return b


@pytest.mark.parametrize("how", ["g++ fails", "no g++", "no torch"])
def test_the_library_is_built_without_the_native_call(build, tmp_path, monkeypatch, capsys, how):
    linked = []

    def run(cmd, **kw):
        if cmd[0] == "g++":
            if how == "no g++":
                raise FileNotFoundError(2, "No such file or directory", "g++")
            return subprocess.CompletedProcess(cmd, 1, "", "cannot find -ltorch_hip")
        linked.append(cmd)
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build.subprocess, "run", run)
    if how == "no torch":
        monkeypatch.setitem(__import__("sys").modules, "torch", None)
    (tmp_path / "woq_call.so").write_bytes(b"of an earlier build")
    assert build.build_lib(verbose=False) == str(tmp_path / "libwoq.so")
    assert len(linked) == 1 and not (tmp_path / "woq_call.so").exists()
    assert "woq_call.so" in capsys.readouterr().err
