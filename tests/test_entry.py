"""build() makes the checker library only where the reference's sources are."""
import subprocess

import pytest

import __graft_entry__ as entry
from fftcorr_amd import build as lib_build


@pytest.mark.parametrize("present", [False, True])
def test_build_needs_no_reference(tmp_path, monkeypatch, present):
    if present:
        (tmp_path / "cc" / "array").mkdir(parents=True)
        (tmp_path / "cc" / "array" / "array_ops.cc").write_text("")
    made = []
    monkeypatch.setattr(entry, "REFERENCE", str(tmp_path))
    monkeypatch.setattr(lib_build, "build", lambda: None)
    monkeypatch.setattr(subprocess, "run", lambda *a, **k: made.append(a))
    entry.build()
    assert len(made) == int(present)
