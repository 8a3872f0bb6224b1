"""The build's two products apart from each other: the C ABI library needs hipcc alone, the native
launchers need torch, its headers and a C++ compiler.  Compilers are replaced by a recorder."""

from __future__ import annotations

import shutil
import sys
from pathlib import Path

import pytest

from picotron_amd import build as builder


@pytest.fixture
def recorder(monkeypatch, tmp_path):
    """Builds into a folder of its own with commands that only write their output file."""

    commands = []

    def run(cmd):
        commands.append(cmd)
        Path(cmd[cmd.index("-o") + 1]).write_bytes(b"")
        return ""

    monkeypatch.setattr(builder, "_run", run)
    monkeypatch.setattr(builder, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(builder, "BUILD_DIR", tmp_path / "obj")
    monkeypatch.setattr(builder, "LIB_PATH", tmp_path / "libpicotron_hip.so")
    monkeypatch.setattr(builder, "NATIVE_PATH", tmp_path / "_native.so")
    return commands


def test_builds_both(recorder):
    assert builder.build(jobs=2).exists() and builder.NATIVE_PATH.exists()


@pytest.mark.parametrize("missing", ["torch", "compiler"])
def test_library_builds_without(recorder, monkeypatch, capsys, missing):
    if missing == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)  # import torch raises ImportError
    else:
        monkeypatch.delenv("CXX", raising=False)
        monkeypatch.setattr(shutil, "which", lambda name: None)
    builder.NATIVE_PATH.write_bytes(b"an earlier build's")
    assert builder.build(jobs=2).exists()
    assert not builder.NATIVE_PATH.exists()
    assert "_native.so not built" in capsys.readouterr().err
    links = [cmd for cmd in recorder if cmd[0] == "hipcc" and "-shared" in cmd]
    assert len(links) == 1
    del recorder[:]
    assert builder.ensure_built() == builder.LIB_PATH and recorder == []  # the library is not rebuilt


def test_a_failing_compilation_raises_after_the_library_is_there(recorder, monkeypatch):
    def broken():
        raise RuntimeError("command failed")

    monkeypatch.setattr(builder, "build_native", broken)
    with pytest.raises(RuntimeError, match="command failed"):
        builder.build(jobs=2)
    assert builder.LIB_PATH.exists()
