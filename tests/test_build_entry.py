"""The build entry point: the product's library is built and imported whatever becomes of the CPU emulation,
which is test infrastructure; a failure of the product's own build is one of the entry point."""
import sys

import pytest

import __graft_entry__ as entry


@pytest.fixture
def steps(monkeypatch):
    import oracle
    from cpu_emu import build_emu
    from ellipticforest_amd import build as efbuild
    done = []
    monkeypatch.setattr(sys, "path", list(sys.path))
    monkeypatch.setattr(efbuild, "build", lambda verbose=False: done.append("library"))
    monkeypatch.setattr(oracle, "build", lambda force=False: done.append("oracle"))
    monkeypatch.setattr(build_emu, "build", lambda: done.append("emulator"))
    return done, efbuild, build_emu


def fail():
    raise RuntimeError("no compiler for it here")


def test_build_survives_the_emulator(steps, monkeypatch, capsys):
    done, _, build_emu = steps
    monkeypatch.setattr(build_emu, "build", fail)
    entry.build()
    assert done == ["library", "oracle"]
    assert "not built: no compiler for it here" in capsys.readouterr().out


def test_build_fails_with_the_library(steps, monkeypatch):
    done, efbuild, _ = steps
    monkeypatch.setattr(efbuild, "build", lambda verbose=False: fail())
    with pytest.raises(RuntimeError, match="no compiler"):
        entry.build()
    assert done == []


def test_build_makes_everything(steps):
    entry.build()
    assert steps[0] == ["library", "oracle", "emulator"]
