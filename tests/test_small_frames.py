"""Frames around the sizes where their launch changes, against the oracle: how many cones a wave
takes (64 x 64 padded cones are the last of one a wave, each doubling after takes twice as many),
work-groups fewer than the chip holds, and the compaction's three forms (16 chunks of 4096 cones
are the last without a count pass, 1024 the last without a scan)."""
from __future__ import annotations

import numpy as np
import pytest

from frame_helpers import assert_frame_matches, gpu_frame, tree_arrays

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (7, 3), (9, 8), (64, 64), (65, 64), (128, 64), (129, 64), (181, 181), (256, 256), (257, 255),
         (256, 257), (513, 511), (641, 479)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("opts", [{}, {"workgroup_size": 64}, {"work_chunk": 128}, {"workgroup_size": 512}])
def test_sizes(svo, orc, gpu, size, opts):
    cam = svo.scenes.config1_camera(*size)
    tree, bases, blocks = tree_arrays(svo, svo.scenes.config1_scene())
    usages = tree.initial_usages(0)
    ref_usages = usages.copy()
    ref = orc.trace_frame(cam, bases, blocks, ref_usages, request_capacity=3000, threads=8)
    out = gpu_frame(svo, gpu, bases, blocks, usages, cam, request_capacity=3000, **opts)
    assert_frame_matches(out, ref, usages_ref=ref_usages)


@pytest.mark.parametrize("base_depth", [1, 2, 3, 5])
def test_staged_bases(svo, orc, gpu, base_depth):
    """Bases of 16 bytes up to the largest that fit the LDS, and larger (read from memory)."""
    spec = svo.scenes.sphere_noise_scene(seed=2, max_depth=max(5, base_depth + 2), base_depth=base_depth)
    spec.name += f"-b{base_depth}"
    cam = svo.scenes.config1_camera(80, 60)
    cam.base_depth = base_depth
    tree, bases, blocks = tree_arrays(svo, spec)
    ref = orc.trace_frame(cam, bases, blocks, None, request_capacity=3000, threads=8)
    out = gpu_frame(svo, gpu, bases, blocks, None, cam, request_capacity=3000)
    assert_frame_matches(out, ref)


def test_composite_spread_over_waves(svo, orc, gpu):
    """The compositing modes take the same launch rules: a frame of few cones a wave has the image,
    layers and loss of the same views in a batch large enough for whole waves."""
    B = svo.BufferName
    tree, bases, blocks = tree_arrays(svo, svo.scenes.config1_scene())
    views = [svo.scenes.config1_camera(48, 40)] + svo.scenes.config5_cameras(8, 256)
    n = [v.screen_size[0] * v.screen_size[1] for v in views]
    rng = np.random.default_rng(4)
    gpu.InitReadBuffer(B.Bases, bases)
    gpu.InitReadBuffer(B.Blocks, blocks)
    gpu.InitBuffer(B.LeafParams, rng.random((blocks.size, 4), np.float32))
    out = []
    for some in (views, views[:1]):
        cones = sum(v.screen_size[0] * v.screen_size[1] for v in some)
        for v in some:
            v.tick = 1
        gpu.InitDeviceBuffer(B.OutputImage, cones, 16)
        gpu.InitDeviceBuffer(B.Layers, cones, 16)
        gpu.InitBuffer(B.TargetImage, np.zeros((cones, 4), np.float32))
        gpu.Composite(some, layers=True)
        out.append((gpu.ReadBuffer(B.OutputImage, np.float32, 4 * n[0]), gpu.ReadBuffer(B.Layers, np.uint32, 4 * n[0])))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert (out[0][1] != 0xFFFFFFFF).any()
    for name in (B.TargetImage, B.LeafParams, B.Layers):
        gpu.ReleaseBuffer(name)
