"""The cost a frame leaves for each tile is the most steps any of the tile's cones took, as the visit
counts have it, whether one wave ran the tile or several ran a part of it each; a frame's costs owe
nothing to the frame before.  A child process reads them where the launch keeps them."""
from __future__ import annotations

import pytest

import fake_hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spy(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("launch_spy"), "launch_spy")


COMMON = """
    import ctypes as C
    hip = C.CDLL("libamdhip64.so.7")
    spy = ctypes.CDLL(sys.argv[1])
    spy.spy_cost.restype = C.c_void_p

    def costs():
        cm.Wait()
        out = np.zeros(spy.spy_tiles(), np.uint32)
        assert hip.hipMemcpy(C.c_void_p(out.ctypes.data), C.c_void_p(spy.spy_cost()), C.c_size_t(out.nbytes), 2) == 0
        return out

    def most(cams):  # per tile of 8 x 8 cones, camera by camera
        visits, out = cm.ReadBuffer(B.VisitCounts, np.uint32, sum(w * h for w, h in cams)), []
        for w, h in cams:
            image = np.zeros((-(-h // 8) * 8, -(-w // 8) * 8), np.uint32)
            image[:h, :w] = visits[:w * h].reshape(h, w)
            visits = visits[w * h:]
            out.append(image.reshape(image.shape[0] // 8, 8, -1, 8).max(axis=(1, 3)).reshape(-1))
        return np.concatenate(out)

    spec = svo.scenes.sphere_noise_scene(seed=1, max_depth=7)
    cm.LoadTree(spec.build())

    def views(size, step):
        cam = svo.scenes.config1_camera(*size)
        for k in range(3):
            cam.origin[k] = cam.origin[k] + 0.02 * step * (k + 1)
        return cam
"""


@pytest.mark.parametrize("sizes,lanes", [([(64, 48)], 1), ([(65, 64)], 2), ([(160, 120)], 8), ([(300, 200)], 16),
                                         ([(401, 299)], 32), ([(641, 479)], 64), ([(33, 20), (160, 121)], 8)], ids=str)
@pytest.mark.parametrize("graph", [False, True])
def test_costs_are_the_most_steps(spy, sizes, lanes, graph):
    fake_hip.run(spy, COMMON + f"""
    sizes, lanes = {sizes!r}, {lanes}
    n = sum(w * h for w, h in sizes)
    cm.InitDeviceBuffer(B.OutputImage, n, 16)
    cm.InitDeviceBuffer(B.VisitCounts, n, 4)
    replay = cm.CaptureFrame([views(s, 0) for s in sizes]) if {graph} else None
    for step in (0, 1, 2, 1, 8):  # small moves (tiles in cost order), then a jump (raster order)
        cams = [views(s, step) for s in sizes]
        replay.Launch(cams) if replay else cm.TraceBatch(cams)
        got = costs()
        assert spy.spy_lanes() == lanes
        want = most(sizes)
        assert got.size == want.size and (step == 8 or want.max() > 20)
        assert np.array_equal(got, want), (step, int((got != want).sum()), got.size)
    """)
