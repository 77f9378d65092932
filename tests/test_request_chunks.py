"""The de-duplication takes requests in chunks of 1024, counted as it flags them: updates whose
stored requests end at, before and after a chunk's edge, and one far below it.  Bricks, grafts
and pool bit-exact against the oracle."""
from __future__ import annotations

import pytest

from stream_helpers import terrain_geometry
from test_stream_parity import _stream_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [False, True], ids=["child-requests", "kept-requests"])
@pytest.mark.parametrize("capacity", [1, 1023, 1024, 1025, 2049])
def test_capacity_at_chunk_edges(svo, orc, gpu, capacity, keep):
    geom = terrain_geometry(svo, 64)
    B, D = 2, 7
    cams = [svo.scenes.config3_camera(f, 96, 64, frames=3, base_depth=B) for f in range(3)]
    hold = svo.scenes.config3_camera(1, 96, 64, frames=3, base_depth=B)
    history, _, _ = _stream_and_compare(svo, orc, gpu, geom, B, D, 8 ** 3 + 700, cams, hold, 2, keep=keep,
                                        capacity=capacity, max_bricks=200, prune_age=3, gc_free_percent=0)
    assert any(h["requests"] > capacity for h in history) and any(h["bricks"] for h in history)
