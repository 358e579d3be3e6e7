"""The pair of libraries, built together (no GPU): a failed link leaves the old pair in place."""

import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "xlstm-metal_amd")


def test_failed_link_keeps_both_libraries(tmp_path, monkeypatch):
    spec = importlib.util.spec_from_file_location("xlstm_build_test", os.path.join(PKG, "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    libs = tmp_path / "lib"
    libs.mkdir()
    b.BUILD, b.LIBDIR = str(tmp_path / "_build"), str(libs)
    b.LIB, b.OPS_LIB = str(libs / "libxlstm_hip.so"), str(libs / "libxlstm_torch.so")
    for p in (b.LIB, b.OPS_LIB):
        open(p, "w").write("old")
    monkeypatch.setattr(b, "_compile", lambda src: src)
    monkeypatch.setattr(b, "_compile_ops", lambda: "ops.o")

    def run(cmd, **kw):
        if cmd[0] == "g++":
            return subprocess.CompletedProcess(cmd, 1, "", "no such symbol")
        open(cmd[cmd.index("-o") + 1], "w").write("new")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(b.subprocess, "run", run)
    with pytest.raises(RuntimeError, match="link failed"):
        b.build(verbose=False)
    assert [open(p).read() for p in (b.LIB, b.OPS_LIB)] == ["old", "old"]
