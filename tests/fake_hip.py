"""Runs code in a child process with a library between libsvo and the HIP runtime: fake_hip.cpp in the
runtime's place, for host code on the CPU, or launch_spy.cpp before it.  The child loads that library
(``fake``), then libsvo, and runs the code given (``svo``, ``B`` and ``cm``, a context, are there)."""
from __future__ import annotations

import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

TESTS = Path(__file__).resolve().parent

PRELUDE = f"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
if hasattr(fake, "fake_limit"):
    fake.fake_limit.argtypes = [ctypes.c_size_t]
    fake.fake_used.restype = fake.fake_launches.restype = ctypes.c_size_t
sys.path.insert(0, {str(TESTS.parent / "svo-tracer_amd")!r})
import _loader
import numpy as np
svo = _loader.load()
B, cm = svo.BufferName, svo.ComputeManager(0)
MiB = 1 << 20
"""


def build(folder: Path, name: str = "fake_hip") -> Path:
    lib = folder / f"lib{name}.so"
    hip = Path(shutil.which("hipcc") or "/opt/rocm/bin/hipcc").resolve().parents[1]
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{hip}/include",
                    f"-I{TESTS.parent / 'svo-tracer_amd' / 'csrc'}", f"-I{TESTS.parent / 'include'}",
                    str(TESTS / f"{name}.cpp"), "-o", str(lib), "-ldl"], check=True)
    return lib


def run(lib: Path, code: str) -> None:
    res = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), str(lib)], capture_output=True,
                         text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
