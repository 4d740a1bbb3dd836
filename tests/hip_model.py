"""Runs Python over libtgx.so and the stand-in for HIP's host calls (tests/hip_model.cpp) in a process
of its own: the stand-in is loaded first with its symbols global, so that the library's HIP calls
resolve to it and no device is needed."""

import subprocess
import sys
import textwrap
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

PRELUDE = """
import ctypes, sys
for p in {paths!r}:
    sys.path.insert(0, p)
model = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
import numpy as np
import tgx
import tgx.runtime as rt
ctx = tgx.Context(0)
assert ctx.report()["arch"] == "gfx950" and model.hip_model_graphs() == 0
"""


def build(folder: Path) -> Path:
    lib = folder / "libhip_model.so"
    cmd = ["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", "-w", str(ROOT / "tests" / "hip_model.cpp"), "-o", str(lib)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return lib


def run(lib: Path, code: str) -> None:
    """`code` behind the prelude (model, np, tgx, rt and a context ctx); its assertions are the caller's."""
    paths = [str(ROOT / "tests"), str(ROOT / "oracle"), str(ROOT / "tgtts-v4_amd")]
    script = PRELUDE.format(paths=paths, lib=str(lib)) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
