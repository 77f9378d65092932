"""What a refused device allocation leaves behind: nothing.  HIP keeps a failure as the thread's last
error until it is asked for, and the launches ask, so a failure that was already reported (or made
good by a smaller allocation) must not fail the next call."""
from __future__ import annotations

import textwrap

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


KEPT = """
    import threading
    geometry = svo.scenes.sphere_noise_scene(seed=1, max_depth=4, base_depth=1).geometry
    before = fake.fake_used()
    cm.BuildTreeDevice(geometry, 1, 4)
    kept = fake.fake_used() - before
    assert kept > 16 * MiB  # a build's temporaries stay for the next one
"""


@pytest.mark.parametrize("code", [
    """
    fake.fake_limit(fake.fake_used() + 8 * MiB)
    cm.InitDeviceBuffer(B.OutputImage, kept // 2, 1)  # a buffer of the same context
    assert fake.fake_used() < before + kept
    """, """
    other = svo.ComputeManager(0)
    fake.fake_limit(fake.fake_used() + 8 * MiB)
    other.InitDeviceBuffer(B.OutputImage, kept // 2, 1)  # of another one on the device
    cm.BuildTreeDevice(geometry, 1, 4)  # finds nothing kept
    """, """
    fake.fake_limit(fake.fake_used() + 8 * MiB)
    try:
        cm.InitDeviceBuffer(B.OutputImage, 64 * MiB, 1)  # does not fit without them either
        raise SystemExit("an allocation beyond the device was accepted")
    except svo.SvoError as e:
        assert "out of memory" in str(e), e
    """, """
    cm.ReleaseBuffer(B.Blocks)  # the scene goes, and what its build left with it
    assert fake.fake_used() < before + MiB
    """, """
    cm.Dispose()
    assert fake.fake_used() == before
    """, """
    others = [svo.ComputeManager(0) for _ in range(3)]
    fake.fake_limit(fake.fake_used() + 90 * MiB)  # for two builds and a buffer at a time
    failed = []
    def work(c, k):
        for _ in range(20):
            try:
                if k:
                    c.BuildTreeDevice(geometry, 1, 4)
                else:
                    c.InitDeviceBuffer(B.OutputImage, 60 * MiB, 1)
                    c.ReleaseBuffer(B.OutputImage)
            except svo.SvoError as e:
                if "out of memory" not in str(e): failed.append(e)  # both at once may not fit
    threads = [threading.Thread(target=work, args=(c, k)) for k, c in enumerate(others)]
    for t in threads: t.start()
    for t in threads: t.join()
    assert not failed, failed
    fake.fake_limit(1 << 32)
    for c in (cm, *others): c.Dispose()
    assert fake.fake_used() == 0
    """], ids=["same context", "another context", "too large", "release", "dispose", "threads"])
def test_kept_build_memory_is_given_back(fake, code):
    fake_hip.run(fake, textwrap.dedent(KEPT) + textwrap.dedent(code))


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
    count, _ = gpu.BuildTreeDevice(spec.geometry, spec.base_depth, spec.max_depth, spec.max_size)
    assert count == spec.build().block_count
