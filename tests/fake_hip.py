"""Runs host code of the library on the CPU over fake_hip.cpp: a child process loads the fake
runtime, then the library, and runs the code given (``svo``, ``fake``, ``B`` and ``cm``, a context,
are there)."""
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
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_used.restype = fake.fake_launches.restype = ctypes.c_size_t
sys.path.insert(0, {str(TESTS.parent / "svo-tracer_amd")!r})
import _loader
import numpy as np
svo = _loader.load()
B, cm = svo.BufferName, svo.ComputeManager(0)
MiB = 1 << 20
"""


def build(folder: Path) -> Path:
    lib = folder / "libfakehip.so"
    hip = Path(shutil.which("hipcc") or "/opt/rocm/bin/hipcc").resolve().parents[1]
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{hip}/include",
                    str(TESTS / "fake_hip.cpp"), "-o", str(lib)], check=True)
    return lib


def run(lib: Path, code: str) -> None:
    res = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), str(lib)], capture_output=True,
                         text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
