"""The pair of libraries, built and loaded together (no GPU): a failed link leaves the old pair in place, and operators
built against another C ABI than the library beside them refuse to run instead of passing it wrong arguments."""

import ctypes
import importlib.util
import os
import re
import shutil
import subprocess
import sys

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


# python_too: Python's declarations were rebuilt with the library, the operators alone were not
@pytest.mark.parametrize("python_too", [False, True])
def test_operators_of_another_abi_refuse(tmp_path, python_too):
    from xlstm_hip import _lib
    pkg = tmp_path / "xlstm_hip"
    shutil.copytree(os.path.join(PKG, "xlstm_hip"), pkg, ignore=shutil.ignore_patterns("*.so", "__pycache__"))
    os.makedirs(pkg / "lib", exist_ok=True)
    shutil.copy(_lib.OPS_PATH, pkg / "lib" / "libxlstm_torch.so")
    stub = "".join(f"int {n}(void) {{ return {99 if n == 'xl_abi_version' else -1}; }}\n" for n in _lib.SIGNATURES)
    (tmp_path / "stub.c").write_text(stub)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(pkg / "lib" / "libxlstm_hip.so"), str(tmp_path / "stub.c")],
                   check=True)
    if python_too:
        src = (pkg / "_lib.py").read_text()
        (pkg / "_lib.py").write_text(re.sub(r"^ABI_VERSION = \d+", "ABI_VERSION = 99", src, flags=re.M))
    code = "import xlstm_hip; print(xlstm_hip.ops.unavailable)"
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                         env={**os.environ, "PYTHONPATH": str(tmp_path)}, cwd=tmp_path)
    assert out.returncode == 0, out.stderr
    assert "ABI" in out.stdout and "build both libraries again" in out.stdout


def test_operators_without_their_library(tmp_path):
    """Half a build imports, and every op says what to do."""
    from xlstm_hip import _lib
    pkg = tmp_path / "xlstm_hip"
    shutil.copytree(os.path.join(PKG, "xlstm_hip"), pkg, ignore=shutil.ignore_patterns("*.so", "__pycache__"))
    os.makedirs(pkg / "lib", exist_ok=True)
    shutil.copy(_lib.OPS_PATH, pkg / "lib" / "libxlstm_torch.so")
    out = subprocess.run([sys.executable, "-c", "import xlstm_hip; print(xlstm_hip.ops.unavailable)"], capture_output=True,
                         text=True, timeout=120, env={**os.environ, "PYTHONPATH": str(tmp_path)}, cwd=tmp_path)
    assert out.returncode == 0, out.stderr
    assert "build it with" in out.stdout


def test_constants_are_the_librarys():
    """The padding tokens and the lm_head's limits, which the tests and the routing read, are the ones the native
    operators use."""
    from xlstm_hip import _lib, ops
    lib = ctypes.CDLL(_lib.OPS_PATH)
    assert (ops._PAD_I, ops._PAD_F) == tuple(ctypes.c_double.in_dll(lib, n).value for n in ("xl_pad_i", "xl_pad_f"))
    assert (ops.LM_HEAD_MAX_ROWS, ops.LM_HEAD_MAX_LDS) == tuple(
        ctypes.c_int64.in_dll(lib, n).value for n in ("xl_lm_head_max_rows", "xl_lm_head_max_lds"))
