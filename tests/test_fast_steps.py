"""The trace kernel's fast steps and its general steps against the oracle, bit for bit, at the
edges between them: cones that are not ordinary (a direction component of 0 or NaN, a start on
the face they move towards, an enormous or degenerate field of view), cameras with depth of
field, cones nearer than 2^-6 to the camera (the footprint's exact form), levels beyond 30 and
frames that refill lanes early."""
from __future__ import annotations

import hashlib
import math
from pathlib import Path

import numpy as np
import pytest

from frame_helpers import assert_frame_matches, gpu_frame, tree_arrays

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).parent / "golden"
IDENT = [1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0]


def axis_camera(svo, eye, forward=0, fov=math.radians(60.0), size=(64, 48)):
    """Looks along axis `forward` (negated for forward >= 3): the middle column and row of an odd
    image have direction components of exactly 0."""
    rows = np.eye(3)[[forward % 3, (forward + 1) % 3, (forward + 2) % 3]] * (-1.0 if forward >= 3 else 1.0)
    return svo.scenes.trace_input(eye, [float(v) for v in rows.reshape(-1)], size[0], size[1], fov,
                                  fov * size[1] / size[0], 4)


def cameras(svo):
    yield "zero components", axis_camera(svo, (-0.5, 0.5, 0.5), size=(65, 49))
    yield "zero components, moving down", axis_camera(svo, (1.5, 0.5, 0.5), forward=3, size=(65, 49))
    yield "inside, on cell faces", axis_camera(svo, (0.5, 0.25, 0.125), forward=4)
    yield "on the volume's faces", axis_camera(svo, (0.0, 1.0, 0.0), forward=5)
    yield "corner, moving out", axis_camera(svo, (0.0, 0.0, 0.0), forward=3)
    cam = svo.scenes.config1_camera(64, 48)
    cam.facing[1] = math.nan
    cam.origin[0], cam.origin[1], cam.origin[2] = 0.5, 0.05, 0.5
    yield "NaN in the facing", cam
    cam = svo.scenes.config1_camera(64, 48)
    for k in range(9):
        cam.facing[k] = cam.facing[k] * 1e-30
    yield "tiny directions", cam
    cam = svo.scenes.config1_camera(64, 48)
    for k in range(9):
        cam.facing[k] = cam.facing[k] * 3e7
    yield "huge directions", cam
    cam = svo.scenes.config1_camera(64, 48)
    cam.dof[0], cam.dof[1] = 0.02, 0.6
    yield "depth of field", cam
    cam = svo.scenes.config1_camera(64, 48)
    cam.fov[0] = -cam.fov[0]
    yield "negative field of view", cam
    cam = svo.scenes.config1_camera(64, 48)
    cam.fov[0] = 1e-6
    yield "narrow field of view", cam
    eye = (0.5 + 0.425, 0.5, 0.5)  # beside the sphere's surface
    yield "near the camera", svo.scenes.trace_input(eye, svo.scenes.look_at(eye, (0.5, 0.7, 0.6)), 64, 48,
                                                    math.radians(60.0), math.radians(45.0), 4)


BEYOND_ORACLE = ["NaN in the facing", "tiny directions", "huge directions"]
NAMES = ["zero components", "zero components, moving down", "inside, on cell faces", "on the volume's faces",
         "corner, moving out", "depth of field", "negative field of view", "narrow field of view", "near the camera"]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("refill", [0, 24])
def test_cameras(svo, orc, gpu, name, refill):
    cam = dict(cameras(svo))[name]
    tree, bases, blocks = tree_arrays(svo, svo.scenes.config1_scene())
    usages = tree.initial_usages(0)
    ref_usages = usages.copy()
    ref = orc.trace_frame(cam, bases, blocks, ref_usages, request_capacity=6000, threads=8)
    out = gpu_frame(svo, gpu, bases, blocks, usages, cam, refill_lanes=refill)
    assert_frame_matches(out, ref, usages_ref=ref_usages)


@pytest.mark.parametrize("name", NAMES + BEYOND_ORACLE)
def test_both_forms_agree(svo, gpu, name):
    """With early refills every step is a general one; otherwise ordinary cones take fast steps."""
    cam = dict(cameras(svo))[name]
    tree, bases, blocks = tree_arrays(svo, svo.scenes.config1_scene())
    a, b = (gpu_frame(svo, gpu, bases, blocks, tree.initial_usages(0), cam, refill_lanes=r) for r in (0, 24))
    for key in ("hit", "visits", "status", "hash", "depth", "location", "usages", "requests"):
        assert np.array_equal(a[key], b[key]), key
    assert np.array_equal(a["rgba"], b["rgba"]) and a["request_count"] == b["request_count"]


def stray_outputs(svo, cm, name, **opts):
    """A stray camera's outputs: hits and visits, and digests of the other arrays, of a frame, of one
    with a stack of two levels (keys s2-) and of four composited layers (key layers)."""
    cam = dict(cameras(svo))[name]
    tree, bases, blocks = tree_arrays(svo, svo.scenes.config1_scene())

    def digest(a):
        return np.array(hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest())

    out = {}
    for prefix, extra in (("", {}), ("s2-", {"stack_levels": 2})):
        o = gpu_frame(svo, cm, bases, blocks, tree.initial_usages(0), cam, **opts, **extra)
        out[prefix + "hit"], out[prefix + "visits"] = o["hit"], o["visits"]
        out[prefix + "request_count"] = np.array(o["request_count"])
        for key in ("status", "hash", "depth", "location", "usages", "requests"):
            out[prefix + key] = digest(o[key])
        # (a NaN's bits are not the frame's to define)
        out[prefix + "rgba"] = digest(np.where(np.isnan(o["rgba"]), np.float32(-1), o["rgba"]))
    if not opts:
        B, n = svo.BufferName, cam.screen_size[0] * cam.screen_size[1]
        cm.InitBuffer(B.LeafParams, np.random.default_rng(4).random((blocks.size, 4), np.float32))
        cm.InitDeviceBuffer(B.Layers, n, 16)
        cm.Composite([cam], layers=True)
        out["layers"] = digest(cm.ReadBuffer(B.Layers, np.uint32, 4 * n))
        for buffer in (B.LeafParams, B.Layers):
            cm.ReleaseBuffer(buffer)
    return out


@pytest.mark.parametrize("name", BEYOND_ORACLE)
@pytest.mark.parametrize("refill", [0, 24])
def test_stray_cones(svo, gpu, name, refill):
    """Stray cones (NaN, vanishing or huge directions), whose blocks are those they entered while the
    oracle looks a block up by the location, have the outputs of the kernel that knew one step form
    only (tests/golden/make_stray_fixture.py)."""
    want = np.load(GOLDEN / "stray_cones.npz")
    got = stray_outputs(svo, gpu, name, **({"refill_lanes": refill} if refill else {}))
    for key, value in got.items():
        assert np.array_equal(value, want[f"{name}/{key}"]), key
    assert (got["hit"] != 0xFFFFFFFF).any() or (got["visits"] > 0).any()


def deep_chain(svo, levels: int, at):
    """A pool (BaseDepth 1) whose only geometry is the cell of `at` on each level down to `levels`."""
    bits = [int(np.float32(v) * np.float32(2.0 ** 32)) for v in at]  # exact: multiples of 2^-32 below 1

    def octant(level):  # of the level-`level` cell of `at`
        return sum(((b >> (31 - level)) & 1 if level <= 31 else 0) << k for k, b in enumerate(bits))

    bases = np.full(8, 0x5555, np.uint16)
    bases[octant(0)] = 0x5555 & ~(3 << (2 * octant(1))) | 2 << (2 * octant(1))
    dense, n_groups = 8 ** 3, 8 ** 2 + levels
    blocks = np.zeros(8 * n_groups, dtype=svo.BLOCK_DTYPE)
    blocks["child"], blocks["chunk"] = 0xFFFFFFFF, 0x5555
    a = (octant(0) << 6) | (octant(1) << 3) | octant(2)
    for level in range(3, levels + 1):
        o = octant(level)
        blocks["chunk"][a] = 0x5555 & ~(3 << (2 * o)) | 2 << (2 * o)
        blocks["colour_r"][a] = level
        if level < levels:
            group = dense // 8 + level - 3
            blocks["child"][a] = 8 * group
            a = 8 * group + o
    usages = np.zeros(n_groups, dtype=svo.USAGE_DTYPE)
    usages["parent"], usages["tick"] = 0xFFFFFFFF, 1
    return bases, blocks, usages


@pytest.mark.parametrize("levels", [29, 30, 31, 32, 33, 40])
@pytest.mark.parametrize("stack_levels", [0, 2])
def test_levels_beyond_30(svo, orc, gpu, levels, stack_levels):
    """Cones aimed along an axis at one cell of each level down to `levels`: the steps change from
    the fast to the general form on the way (level 30)."""
    at = (0.59375, 0.296875, 0.6875)
    bases, blocks, usages = deep_chain(svo, levels, at)
    cam = svo.scenes.trace_input((0.25, at[1], at[2]), IDENT, 9, 9, 1e-12, 1e-12, 1, tick=7)
    ref_usages = usages.copy()
    ref = orc.trace_frame(cam, bases, blocks, ref_usages, request_capacity=100, threads=1)
    assert int(ref["depth"].max()) == levels, "some cones were meant to reach the deepest block"
    out = gpu_frame(svo, gpu, bases, blocks, usages, cam, request_capacity=100, max_tree_depth=levels,
                    stack_levels=stack_levels)
    assert_frame_matches(out, ref, usages_ref=ref_usages)
