"""Writes stray_cones.npz: frames of cones whose blocks are those they entered and not those their
location names (NaN, vanishing and huge directions), which the oracle, looking blocks up by the
location, does not cover.  The expected outputs are those of the trace kernel before it had a
second step form (the library of commit 05664df, on an MI355X): run from the repo root on the
device with SVO_LIB naming that build.  Full arrays of the hit blocks and visit counts, digests of
the rest; per camera the plain frame, one with a short stack of two levels, and the composited
layers of four."""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[2]
sys.path[:0] = [str(ROOT / "svo-tracer_amd"), str(ROOT / "oracle"), str(ROOT / "tests")]
OUT = Path(__file__).resolve().parent

if __name__ == "__main__":
    import _loader
    from test_fast_steps import BEYOND_ORACLE, stray_outputs

    svo = _loader.load()
    arrays = {}
    with svo.ComputeManager(0) as cm:
        for name in BEYOND_ORACLE:
            for key, value in stray_outputs(svo, cm, name).items():
                arrays[f"{name}/{key}"] = value
    path = Path(sys.argv[1]) if len(sys.argv) > 1 else OUT / "stray_cones.npz"
    np.savez_compressed(path, **arrays)
    print(f"wrote {path}: {len(arrays)} arrays")
