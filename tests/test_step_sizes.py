"""A kernel-by-kernel step's appends around the sizes where they change: one work-group of 1024 items
(which appends by itself), a few, and more than 4096 (whose counts are scanned first); entries go
behind what a queue holds, in work-item order, and what a queue cannot hold is counted only."""
from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bind_init(svo, cm, n, queue_len):
    B, K = svo.BufferName, svo.KernelName
    for name, size in ((B.Origins, 16), (B.Directions, 16), (B.FoVs, 4), (B.Locations, 32), (B.Depths, 1),
                       (B.Weightings, 1), (B.ParentTraces, 4), (B.ColourRs, 1), (B.ColourGs, 1), (B.ColourBs, 1),
                       (B.FinalColourRs, 4), (B.FinalColourGs, 4), (B.FinalColourBs, 4), (B.FinalWeightings, 4)):
        cm.InitDeviceBuffer(name, n, size)
    for name in (B.BaseTraceQueue, B.BackgroundQueue):
        cm.InitDeviceBuffer(name, queue_len, 4)
    for name in (B.BaseTraceQueueID, B.BackgroundQueueID):
        cm.InitBuffer(name, np.zeros(1, np.uint32))
    for name in ("Origins", "Directions", "FoVs", "Locations", "Depths", "BaseTraceQueue", "BaseTraceQueueID",
                 "BackgroundQueue", "BackgroundQueueID", "ColourRs", "ColourGs", "ColourBs", "Weightings",
                 "ParentTraces", "FinalColourRs", "FinalColourGs", "FinalColourBs", "FinalWeightings"):
        cm.SetArg(K.Init, name, B[name])


@pytest.mark.parametrize("size", [(1, 1), (31, 33), (32, 32), (41, 25), (64, 64), (257, 129), (2049, 2048)])
def test_init_appends(svo, gpu, size):
    B, K = svo.BufferName, svo.KernelName
    n = size[0] * size[1]
    bind_init(svo, gpu, n, 2 * n)
    cam = svo.scenes.trace_input((-0.4, 0.5, 0.5), [1.0, 0, 0, 0, 1.0, 0, 0, 0, 1.0], *size, math.radians(120.0),
                                 math.radians(100.0), 4)
    gpu.SetArg(K.Init, "input", cam)
    for _ in range(2):  # the second step's entries follow the first's
        gpu.Enqueue(K.Init, list(size))
    ids = np.arange(n, dtype=np.uint32)
    inside = gpu.ReadBuffer(B.Depths, np.uint8, n) == 1
    if n >= 1024:
        assert inside.any() and not inside.all()
    for queue, counter, want in ((B.BaseTraceQueue, B.BaseTraceQueueID, ids[inside]),
                                 (B.BackgroundQueue, B.BackgroundQueueID, ids[~inside])):
        assert gpu.ResetIDBuffer(counter) == 2 * want.size
        assert gpu.ResetIDBuffer(counter) == 0
        assert np.array_equal(gpu.ReadBuffer(queue, np.uint32, 2 * want.size), np.concatenate([want, want]))


@pytest.mark.parametrize("size", [(24, 24), (129, 65)])
def test_full_queues_count_on(svo, gpu, size):
    B, K = svo.BufferName, svo.KernelName
    n = size[0] * size[1]
    bind_init(svo, gpu, n, 100)
    cam = svo.scenes.trace_input((0.5, 0.5, 0.5), [1.0, 0, 0, 0, 1.0, 0, 0, 0, 1.0], *size, 1.0, 1.0, 4)
    gpu.SetArg(K.Init, "input", cam)
    gpu.Enqueue(K.Init, list(size))
    assert gpu.ResetIDBuffer(B.BaseTraceQueueID) == n and gpu.ResetIDBuffer(B.BackgroundQueueID) == 0
    assert np.array_equal(gpu.ReadBuffer(B.BaseTraceQueue, np.uint32, 100), np.arange(100, dtype=np.uint32))
