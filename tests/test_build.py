"""build.py without a compiler run: what is linked when the Python binding, which
the mirror can do without, cannot be built, and which binding belongs to which
Python and torch."""
import os

import pytest

import __graft_entry__


@pytest.fixture
def b(monkeypatch, tmp_path):
    """The build script with its outputs under tmp_path; compiling and linking
    only note their arguments."""
    b = __graft_entry__._load_build_script()
    for name in ("OBJ_DIR", "LIB_DIR"):
        monkeypatch.setattr(b, name, str(tmp_path))
    for name in ("LIB_PATH", "BENCH_LIB_PATH"):
        monkeypatch.setattr(b, name, str(tmp_path / os.path.basename(getattr(b, name))))
    b.compiled = []
    monkeypatch.setattr(b, "_compile", lambda src: b.compiled.append(src) or src)
    monkeypatch.setattr(b, "_link", lambda objs, path: open(path, "w").close())
    return b


def _no_gxx(*a, **k):
    raise FileNotFoundError("g++")


def _gxx_fails(cmd, **k):
    return type("R", (), dict(returncode=1, stdout="", stderr="Python.h: No such file or directory"))


@pytest.mark.parametrize("run", [_no_gxx, _gxx_fails])
def test_library_without_the_binding(b, monkeypatch, capsys, run):
    monkeypatch.setattr(b.subprocess, "run", run)
    with open(b.binding_path(), "w") as f:
        f.write("built from other sources")
    assert b.build() == b.LIB_PATH
    assert os.path.exists(b.LIB_PATH) and os.path.exists(b.BENCH_LIB_PATH)
    assert not os.path.exists(b.binding_path())
    assert "not built" in capsys.readouterr().err
    # and the missing binding does not make the libraries stale
    b.compiled.clear()
    b.build(force=False)
    assert b.compiled == []


def test_binding_is_named_after_torch(b, pkg, monkeypatch, tmp_path):
    """The name build.py gives is the one the loader looks for; with another torch
    installed the binding is stale, and the new one replaces it."""
    import torch
    assert os.path.basename(b.binding_path()) == os.path.basename(pkg._binding_path())
    assert torch.__version__ in b.binding_path()
    b._build_binding = lambda path: open(path, "w").close()
    b.build()
    assert not b.binding_stale()
    other = tmp_path / "torch"
    other.mkdir()
    (other / "version.py").write_text("__version__ = '9.9.0'\ngit_version = '0123456789ab'\n")
    monkeypatch.setattr(b, "torch_dir", lambda: str(other))
    assert b.binding_stale()
    before = set(os.listdir(tmp_path))
    b.compiled.clear()
    b.build(force=False)
    assert b.compiled == []
    (new,) = set(os.listdir(tmp_path)) - before
    assert new.endswith(".torch-9.9.0-01234567.so")
    assert len([f for f in os.listdir(tmp_path) if f.startswith("_q4_binding")]) == 1
