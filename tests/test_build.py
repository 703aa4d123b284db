"""build.py without a compiler run: what is linked when the Python binding, which
the mirror can do without, cannot be built."""
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
    for name in ("LIB_PATH", "BENCH_LIB_PATH", "BINDING_PATH"):
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
    with open(b.BINDING_PATH, "w") as f:
        f.write("built from other sources")
    assert b.build() == b.LIB_PATH
    assert os.path.exists(b.LIB_PATH) and os.path.exists(b.BENCH_LIB_PATH)
    assert not os.path.exists(b.BINDING_PATH)
    assert "not built" in capsys.readouterr().err
    # and the missing binding does not make the libraries stale
    b.compiled.clear()
    b.build(force=False)
    assert b.compiled == []
