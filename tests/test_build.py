"""The library, its probe and its timing program are built whatever becomes of the Python layer's extension module."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from conftest import ROOT
from orin_qwen_lossless_amd import build

BUILT = os.path.exists(os.path.join(build.OBJ, "capi.cpp.o")) and os.path.exists(build.LIB)
pytestmark = pytest.mark.skipif(not BUILT, reason="links the objects of a build")


def test_without_torch():
    code = "import sys; sys.modules['torch'] = None; from orin_qwen_lossless_amd import build; print(build.build())"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=600)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == build.LIB and "needs torch" in r.stderr


def test_with_a_compiler_that_fails_on_the_module(monkeypatch, tmp_path):
    for name in ("LIB", "PROBE", "BENCH", "HOST"):
        monkeypatch.setattr(build, name, str(tmp_path / os.path.basename(getattr(build, name))))
    monkeypatch.setenv("CXX", "false")
    with pytest.raises(RuntimeError, match="building _host"):
        build.build()
    assert sorted(os.listdir(tmp_path)) == sorted(os.path.basename(p) for p in (build.LIB, build.PROBE, build.BENCH))
