"""The build takes every listed source or fails, and the library needs no symbol
of its own from elsewhere."""
import os
import subprocess

import pytest

from shady_thinker_amd import build


def test_missing_source_fails(monkeypatch, tmp_path):
    monkeypatch.setattr(build, "SOURCES", ["runtime.hip", "no_such_kernel.hip"])
    monkeypatch.setattr(build, "OBJ", str(tmp_path))
    monkeypatch.setattr(build, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(build, "_compile", lambda src: pytest.fail(f"compiled {src}"))
    with pytest.raises(RuntimeError, match="no_such_kernel.hip"):
        build.build()


def test_sources_are_the_hip_files():
    assert sorted(build.SOURCES) == sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip"))


def test_library_defines_its_symbols():
    out = subprocess.run(["nm", "-D", "--undefined-only", build.LIB], check=True, capture_output=True, text=True).stdout
    assert not [l for l in out.split() if l.startswith(("_ZN2st", "st_"))]
