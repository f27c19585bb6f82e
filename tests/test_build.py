"""The two libraries are published as one (CPU only)."""
import subprocess

import pytest

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
