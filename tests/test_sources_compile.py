"""Every HIP source is accepted by the compiler as it stands, whatever library
happens to be built: both passes, syntax and semantics only, with the build's
own flags. A name in a shared header that clashes with one of a source that was
not rebuilt shows here."""
from __future__ import annotations

import glob
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("levo_build", os.path.join(ROOT, "levo2.cpp_amd", "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)
SOURCES = sorted(glob.glob(os.path.join(build.CSRC, "*.hip")) + glob.glob(os.path.join(build.PKG, "bench", "*.hip")))


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("src", SOURCES, ids=[os.path.basename(s) for s in SOURCES])
@pytest.mark.parametrize("side", ["host", "device"])
def test_compiles(src, side):
    r = subprocess.run([build.HIPCC, *build.COMMON, *build.DEVICE, f"--cuda-{side}-only", "-fsyntax-only", "-x", "hip", src],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
