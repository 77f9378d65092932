"""Edges of a tree dispatch's launches: walks that outlast the levels launched with them (what
follows waits for the host, and is launched again), requests appended once all the same, grafts
of one group with and without a child, and collections that end at a chunk's edge.  Pool and
statistics bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from test_tree_parity import Mirror, _stats_equal, _ui
from tree_helpers import U32MAX, check_pool, tiny_pool

pytestmark = pytest.mark.gpu

LEVELS = (1, 2, 3, 4, 5, 7, 8, 12)  # three go out with a dispatch, then four at a time


def _chains(svo, levels, roots=(100, 101, 300)):
    """A tiny pool with a chain of `levels` groups below each root."""
    bases, blocks, usages = tiny_pool(svo, 1, extra_groups=len(roots) * levels + 16)
    g = 64
    for k, a in enumerate(roots):
        for j in range(levels):
            blocks["child"][a] = 8 * g
            usages["tick"][g], usages["parent"][g] = 5, a
            a, g = 8 * g + (3 * k + j) % 8, g + 1
    return bases, blocks, usages, roots


@pytest.mark.parametrize("levels", LEVELS)
def test_prune_walk_lengths(svo, orc, gpu, levels):
    bases, blocks, usages, roots = _chains(svo, levels)
    surface = np.zeros(1, dtype=svo.BLOCK_DTYPE)
    surface["colour_r"], surface["child"] = 77, 5
    loc = np.zeros((2, 3), np.uint64)
    loc[1] = 1 << 63
    rec = np.zeros(len(roots) + 2, dtype=svo.PRUNING_DTYPE)
    rec["properties"][: len(roots)] = 1 | 8  # cull the children, write the surface record
    rec["depth"][: len(roots)] = 0xFF
    rec["address"][: len(roots)] = roots
    rec["child_address"] = U32MAX
    rec["depth"][-2:], rec["address"][-2:] = (6, 7), (0, 1)  # two misses: a child request each
    m = Mirror(svo, orc, gpu, bases, blocks, usages, count=1)
    got, ref = m.prune(_ui(orc, 1, 9), rec, surface, loc)
    _stats_equal(got, ref)
    assert ref["requests"] == 2
    m.compare(f"prune, {levels} levels")
    check_pool(m.ref.blocks, m.ref.usages, 1)


@pytest.mark.parametrize("levels", LEVELS)
def test_graft_walk_lengths(svo, orc, gpu, levels):
    bases, blocks, usages, roots = _chains(svo, levels)
    loc = np.zeros((1, 3), np.uint64)
    gb = np.zeros(16, dtype=svo.BLOCK_DTYPE)
    gb["child"], gb["chunk"], gb["colour_r"] = U32MAX, 0xAAAA, np.arange(16)
    gb["child"][6] = 8
    rec = np.zeros(len(roots) + 2, dtype=svo.GRAFTING_DTYPE)
    rec["graft_total_size"], rec["depth"] = 16, 0xFF
    rec["graft_address"][: len(roots)] = roots
    rec["graft_address"][-2] = roots[0]  # the later record of a target is linked
    rec["depth"][-1], rec["graft_address"][-1] = 6, 0  # a miss
    m = Mirror(svo, orc, gpu, bases, blocks, usages)
    got, ref = m.graft(_ui(orc, 1, 9), rec, gb, loc)
    _stats_equal(got, ref)
    assert ref["placed"] == len(roots) and ref["requests"] == 1
    m.compare(f"graft, {levels} levels")
    check_pool(m.ref.blocks, m.ref.usages, 1)


@pytest.mark.parametrize("child", [None, 0, 8, 4, U32MAX - 1], ids=str)
def test_one_group_grafts(svo, orc, gpu, child):
    """The middle of three one-group grafts names a child: invalid wherever it points."""
    bases, blocks, usages = tiny_pool(svo, 1, extra_groups=16)
    gb = np.zeros(24, dtype=svo.BLOCK_DTYPE)
    gb["child"], gb["colour_g"] = U32MAX, np.arange(24)
    if child is not None:
        gb["child"][8 + 5] = child
    rec = np.zeros(3, dtype=svo.GRAFTING_DTYPE)
    rec["graft_total_size"], rec["graft_data_address"], rec["depth"] = 8, (0, 8, 16), 0xFF
    rec["graft_address"] = (100, 200, 300)
    m = Mirror(svo, orc, gpu, bases, blocks, usages)
    got, ref = m.graft(_ui(orc, 1, 9), rec, gb, np.zeros((0, 3), np.uint64))
    _stats_equal(got, ref)
    assert ref["placed"] == (3 if child is None else 2)
    m.compare(f"one-group grafts, child {child}")


@pytest.mark.parametrize("need", [1, 959, 960, 961, 1984, 1985, 2936, 2937, 5000])
def test_collection_ends_at_chunk_edges(svo, orc, gpu, need):
    """3000 groups in chunks of 1024, the first 64 of them dense: 960 candidates in the first chunk."""
    bases, blocks, usages = tiny_pool(svo, 1, extra_groups=3000 - 64)
    m = Mirror(svo, orc, gpu, bases, blocks, usages)
    ui = _ui(orc, 1, 100, offset=0)
    got = gpu.Collect(ui, need)
    ref = m.ref.collect(ui, need)
    assert got.tolist() == ref.tolist() and len(ref) == min(need, 2936)
    m.compare(f"collect {need}")
