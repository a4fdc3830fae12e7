"""What the operators' native host side is built from, and that nothing else is used in its place."""
import importlib.machinery
import subprocess
import warnings
from pathlib import Path

import pytest
import torch

from timeviper_amd import _capi, _native, build


def test_what_is_loaded_is_built_from_this_tree():
    build.ensure_built()
    assert _native.ops.built_from == build.native_id() == build.NATIVE_ID.read_text()
    assert any(build.NATIVE.name == "_tv_native" + s for s in importlib.machinery.EXTENSION_SUFFIXES)


@pytest.mark.parametrize("what,value", [("NATIVE_FLAGS", ["-O3"]), ("NATIVE_LIBS", ["-lc10"]), ("CXX", "c++"), ("NATIVE", build.NATIVE.with_name("_tv_native.cpython-399-x.so"))])
def test_a_change_of_what_it_is_built_with_is_another_build(what, value, monkeypatch):
    before = build.native_id()
    monkeypatch.setattr(build, what, value)
    assert build.native_id() != before and not build.native_is_current()


def test_another_torch_is_another_build(monkeypatch):
    before = build.native_id()
    monkeypatch.setattr(torch, "__version__", "0.0")
    assert build.native_id() != before


def test_a_binary_of_other_sources_is_not_used(monkeypatch):
    """not even with the tree's id beside it: a warning, and kernels.py goes its own way"""
    monkeypatch.setattr(build, "native_id", lambda: "another")
    monkeypatch.setattr(build, "native_is_current", lambda: True)
    ops = _native._Ops()
    with pytest.warns(RuntimeWarning, match="other sources"):
        assert ops.rms_norm(1, 2, 3, 4, 5) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert ops.rms_norm() is None and ops.scan() is None and ops.native is None


@pytest.mark.parametrize("broken", ["missing", "no extension", "another library"])
def test_without_it_the_operators_go_through_ctypes(broken, tmp_path, monkeypatch):
    if broken == "another library":
        monkeypatch.setattr(_capi, "lib_path", lambda: tmp_path / "none.so")
    else:
        monkeypatch.setattr(build, "NATIVE", tmp_path / "none.so")
        monkeypatch.setattr(build, "native_id", lambda n=build.native_id(): n)
        if broken == "no extension":
            (tmp_path / "none.so").write_bytes(b"no ELF")
    with pytest.warns(RuntimeWarning, match="through ctypes"):
        assert _native._Ops().rms_norm() is None


def test_a_build_without_a_host_compiler_makes_the_library(tmp_path, monkeypatch, capfd):
    monkeypatch.setattr(build, "CXX", str(tmp_path / "no-compiler"))
    monkeypatch.setattr(build, "NATIVE", tmp_path / "_tv_native.so")
    monkeypatch.setattr(build, "NATIVE_ID", tmp_path / "_tv_native.id")
    assert build.ensure_built() == build.LIB and not build.NATIVE.exists()
    assert "go through ctypes" in capfd.readouterr().err


def test_a_build_never_shows_half_a_file(tmp_path, monkeypatch):
    """while the linker writes, and where it fails, what was there before stays"""
    there, tag = tmp_path / build.NATIVE.name, tmp_path / build.NATIVE_ID.name
    there.write_bytes(b"the old one")
    monkeypatch.setattr(build, "NATIVE", there)
    monkeypatch.setattr(build, "NATIVE_ID", tag)
    seen = []

    def linker(cmd, **k):
        out = Path(cmd[cmd.index("-o") + 1])
        out.write_bytes(b"half")
        seen.append(there.read_bytes())
        return subprocess.CompletedProcess(cmd, len(seen) == 1, "", "")
    monkeypatch.setattr(build.subprocess, "run", linker)
    with pytest.raises(RuntimeError):
        build.build_native()
    assert there.read_bytes() == b"the old one" and not tag.exists()
    build.build_native()
    assert seen == [b"the old one"] * 2 and there.read_bytes() == b"half" and tag.read_text() == build.native_id() and len(list(tmp_path.iterdir())) == 2
