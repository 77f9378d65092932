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

