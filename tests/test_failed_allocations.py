"""What a refused device allocation leaves behind: nothing.  HIP keeps a failure as the thread's last
error until it is asked for, and the launches ask, so a failure that was already reported (or made
good by a smaller allocation) must not fail the next call."""
from __future__ import annotations

import numpy as np
import pytest

import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


def test_next_call_succeeds(fake):
    fake_hip.run(fake, """
        geometry = svo.scenes.sphere_noise_scene(seed=1, max_depth=4, base_depth=1).geometry
        try:
            cm.InitDeviceBuffer(B.OutputImage, 1 << 40, 16)
            raise SystemExit("an allocation beyond the device was accepted")
        except svo.SvoError as e:
            assert "out of memory" in str(e), e
        cm.BuildTreeDevice(geometry, 1, 4)
    """)


def test_build_falls_back_to_what_it_needs(fake):
    """A device with less room than the build's usual slabs, but enough for what it holds in them."""
    fake_hip.run(fake, """
        geometry = svo.scenes.sphere_noise_scene(seed=1, max_depth=4, base_depth=1).geometry
        fake.fake_limit(20 * MiB)
        cm.BuildTreeDevice(geometry, 1, 4)
        assert fake.fake_launches() > 5
    """)


@pytest.mark.gpu
def test_frame_after_a_refused_buffer(svo, gpu):
    B = svo.BufferName
    gpu.InitBuffer(B.ChildRequestID, np.full(1, 7, np.uint32))
    with pytest.raises(svo.SvoError):
        gpu.InitDeviceBuffer(B.PruningBlockData, 1 << 46, 16)  # 1 PiB
    assert gpu.ResetIDBuffer(B.ChildRequestID) == 7
    spec = svo.scenes.sphere_noise_scene(seed=1, max_depth=5, base_depth=2)
    with pytest.raises(svo.SvoError):
        gpu.InitDeviceBuffer(B.PruningBlockData, 1 << 46, 16)
    count, _ = gpu.BuildTreeDevice(spec.geometry, spec.base_depth, spec.max_depth)
    assert count == spec.build().block_count
