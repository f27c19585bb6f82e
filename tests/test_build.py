"""The two libraries are published as one, and a native call path that cannot
be loaded leaves the operators to their Python wrappers (CPU only)."""
import os
import subprocess
import sys

import pytest

from bytes_amd import _lib
from bytes_amd import build as B


@pytest.fixture
def folder(tmp_path, monkeypatch):
    """A build in a folder of its own whose compilers only write their output."""
    for name, path in (("LIB", "libbytes_amd.so"), ("NATIVE", "_native.so"), ("OBJ", "_build")):
        monkeypatch.setattr(B, name, str(tmp_path / path))
    monkeypatch.setattr(B, "_compile", lambda src: str(tmp_path / "x.o"))
    (tmp_path / "libbytes_amd.so").write_text("old")
    (tmp_path / "_native.so").write_text("old")

    def run(cmd, **kw):
        native = any(str(a).endswith("native.cpp") for a in cmd)
        if native and run.fail:
            return subprocess.CompletedProcess(cmd, 1, "", "no compiler")
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    run.fail = False
    monkeypatch.setattr(B.subprocess, "run", run)
    return tmp_path, run


def test_failed_host_compile_publishes_nothing(folder):
    path, run = folder
    run.fail = True
    with pytest.raises(RuntimeError, match="no compiler"):
        B.build()
    assert (path / "libbytes_amd.so").read_text() == "old" and (path / "_native.so").read_text() == "old"


def test_build_replaces_both(folder):
    path, _ = folder
    B.build()
    assert (path / "libbytes_amd.so").read_text() == "new" and (path / "_native.so").read_text() == "new"


def test_unloadable_native_path_falls_through(monkeypatch):
    """A missing or mismatched _native.so: one warning that names the build
    command, and every call goes on in the Python wrapper."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} not built (run python -m bytes_amd.build)")
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setitem(sys.modules, "bytes_amd._native", None)
    with pytest.warns(RuntimeWarning, match="python -m bytes_amd.build"):
        n = _lib.native()
    assert n.dense(1, 2, 3) is None
    assert _lib.native() is n
