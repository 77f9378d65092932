"""Device builds against the host builder, block for block, where their shared rules take another
form on the device: normals told apart without division (flat terrain, axis-aligned and vertical
normals, where the exact form decides), noise points that share a lattice cell (cells much smaller
than blocks, one octave, many), and levels without flags of their own (a tree that ends with its
dense level, one level below it)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def heightfield(svo, **k):
    spec = svo.scenes.config2_scene(max_depth=9, resolution=256)
    for name, v in k.items():
        setattr(spec.geometry, name, v)
    return spec


def noise(svo, **k):
    spec = svo.scenes.sphere_noise_scene(seed=5, max_depth=7, base_depth=2)
    for name, v in k.items():
        setattr(spec.geometry, name, v)
    return spec


CASES = {
    "flat terrain": lambda svo: heightfield(svo, z_min=0.4, z_max=0.4),
    "terrain clamped at both ends": lambda svo: heightfield(svo, gain=3.0, octaves=2),
    "steep terrain": lambda svo: heightfield(svo, z_min=0.05, z_max=0.95, frequency=16.0),
    "plain sphere": lambda svo: noise(svo, amplitude=0.0),
    "one octave": lambda svo: noise(svo, octaves=1, amplitude=0.2),
    "lattice cells smaller than blocks": lambda svo: noise(svo, octaves=2, frequency=300.0),
    "seven octaves": lambda svo: noise(svo, octaves=7, amplitude=0.1),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("below", [0, 1, 2])  # levels below the dense one
def test_equals_host_build(svo, gpu, name, below):
    spec = CASES[name](svo)
    depth = spec.base_depth + 2 + below
    ref = svo.build_tree(spec.geometry, spec.base_depth, depth, 0xFFFFFFFF // 8)
    count, tree = gpu.BuildTreeDevice(spec.geometry, spec.base_depth, depth, 0xFFFFFFFF // 8, with_usages=True,
                                      usage_tick=3, host_copy=True)
    assert count == ref.block_count
    assert np.array_equal(tree.bases, ref.bases)
    assert np.array_equal(tree.blocks.view(np.uint8), ref.blocks.view(np.uint8))
    B = svo.BufferName
    assert gpu.BufferSize(B.Blocks) == 16 * count
    assert np.array_equal(gpu.ReadBuffer(B.Blocks, np.uint8), ref.blocks.view(np.uint8))
    assert np.array_equal(gpu.ReadBuffer(B.Usages, svo.USAGE_DTYPE), ref.initial_usages(3))



def test_rebuilds_in_place(svo, gpu):
    """Builds over the last build's buffers (about the same size, nothing else holding them), over
    buffers that a kernel argument still holds (which are left alone), and of other sizes."""
    B, K = svo.BufferName, svo.KernelName
    big = 0xFFFFFFFF // 8

    def build(spec, depth, tick):
        ref = svo.build_tree(spec.geometry, spec.base_depth, depth, big)
        gpu.BuildTreeDevice(spec.geometry, spec.base_depth, depth, big, with_usages=True, usage_tick=tick)
        assert np.array_equal(gpu.ReadBuffer(B.Blocks, np.uint8), ref.blocks.view(np.uint8))
        assert np.array_equal(gpu.ReadBuffer(B.Bases, np.uint16), ref.bases)
        assert np.array_equal(gpu.ReadBuffer(B.Usages, svo.USAGE_DTYPE), ref.initial_usages(tick))

    hills, steep = heightfield(svo), heightfield(svo, seed=8, z_min=0.3, z_max=0.5)
    build(hills, 8, 1)
    first = gpu.DevicePointer(B.Blocks)
    build(hills, 8, 2)
    assert gpu.DevicePointer(B.Blocks) == first
    build(steep, 8, 3)
    gpu.SetArg(K.ResolveRemainders, "Blocks", B.Blocks)  # the argument holds this build's blocks
    held = gpu.DevicePointer(B.Blocks)
    build(hills, 8, 4)
    assert gpu.DevicePointer(B.Blocks) != held
    gpu.InitBuffer(B.PruningBlockData, np.zeros(1, svo.BLOCK_DTYPE))
    gpu.SetArg(K.ResolveRemainders, "Blocks", B.PruningBlockData)
    build(hills, 6, 5)
    build(steep, 9, 6)
    build(noise(svo), 5, 7)
