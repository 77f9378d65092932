"""A device build that fails leaves a defined state.  A build over the last tree's buffers destroys that
tree, so whichever call fails, either the tree is whole or none of its buffers is bound (frames are
then refused instead of walking a mixed tree), and the next build succeeds."""
from __future__ import annotations

import pytest

import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("call", ["hipMalloc", "hipMemsetAsync", "hipLaunchKernel", "hipMemcpyAsync",
                                  "hipStreamSynchronize", "hipDeviceSynchronize"])
@pytest.mark.parametrize("host_copy", [False, True])
def test_whole_or_unbound(fake, call, host_copy):
    # BaseDepth 1: 64 dense groups; launches do nothing, so the build finds no geometry
    fake_hip.run(fake, f"""
        geometry = svo.scenes.sphere_noise_scene(seed=1, max_depth=4, base_depth=1).geometry
        tree = {{B.Bases: 16, B.Blocks: 64 * 128, B.Usages: 64 * 8}}
        outcomes = set()
        for k in range(200):
            for name, size in tree.items():
                cm.InitBuffer(name, np.full(size, 0xa5, np.uint8))
            fake.fake_fail({call!r}.encode(), k)
            try:
                cm.BuildTreeDevice(geometry, 1, 4, with_usages=True, host_copy={host_copy})
                ok = True
            except svo.SvoError:
                ok = False
            if fake.fake_fail_pending():
                fake.fake_fail(b"", -1)
                assert ok
                break
            if ok:  # a failure that a smaller allocation made good
                outcomes.add("made good")
                continue
            bound = []
            for name in tree:
                try:
                    bound.append(cm.BufferSize(name) > 0)
                except svo.SvoError:
                    bound.append(False)
            assert all(bound) or not any(bound), (k, bound)
            if all(bound):
                outcomes.add("whole")
                for name, size in tree.items():
                    assert (cm.ReadBuffer(name, np.uint8) == 0xa5).all(), (k, name)
            else:
                outcomes.add("unbound")
            cm.BuildTreeDevice(geometry, 1, 4, with_usages=True)
        else:
            raise SystemExit("every build failed")
        assert outcomes, "no build failed"
        if {call!r} in ("hipMemsetAsync", "hipLaunchKernel", "hipMemcpyAsync"):
            assert outcomes == {{"whole", "unbound"}}, outcomes
    """)
