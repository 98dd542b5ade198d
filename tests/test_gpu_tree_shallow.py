"""Propagation of shallow trees through a plan of default shape, whose tiles take one
step of the last pass: sizes around a tile's end and around the line of 75,000 nodes.
World matrices and events against the oracle, bit for bit."""
import numpy as np
import pytest

from pipeline_amd import _lib, scenes

from test_gpu_tree import DeviceTree, oracle_world

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,kw", [(2_000, {"max_depth": 2, "roots": 20, "p": 0.01, "max_children": 200}), (20_000, {"max_depth": 2, "roots": 20, "p": 0.0005, "max_children": 5_000}),
                                      (74_999, {"max_depth": 3, "roots": 90, "p": 0.02, "max_children": 60}), (75_100, {"max_depth": 3, "roots": 90, "p": 0.02, "max_children": 60}),
                                      (5_000, {"max_depth": 2, "roots": 1_000, "p": 0.1, "max_children": 9}), (20_000, {})])
def test_shallow(orc, nodes, kw):
    ts = scenes.tree_scene(nodes, 3, **kw)
    t = DeviceTree(ts)
    plan = t.plan(0)[0]
    rng = np.random.default_rng(nodes)
    t.propagate(plan=plan)
    want, event = oracle_world(orc, ts)
    assert np.array_equal(t.world_by_slot()[1:].view(np.uint32), want[ts.index_of_slot][1:].view(np.uint32))
    assert np.array_equal(t.dirty_world.download()[1:ts.n_slots], event[ts.index_of_slot][1:])
    # a second frame with a few dirty nodes: unchanged matrices, an event for what lies below them
    dirty = (rng.random(ts.n_slots) < 0.02).astype(np.uint8)
    dirty[0] = 0
    t.dirty_world.fill_u32(0)
    t.propagate(dirty, plan=plan)
    assert np.array_equal(t.world_by_slot()[1:].view(np.uint32), want[ts.index_of_slot][1:].view(np.uint32))
    moved = dirty.copy()
    for a, b in zip(ts.level_offsets[:-1].astype(int), ts.level_offsets[1:].astype(int)):
        moved[a:b] |= moved[ts.parent_slot[a:b]]
    assert np.array_equal(t.dirty_world.download()[1:ts.n_slots], moved[1:])
    _lib.load().dpc_tree_plan_destroy(plan)
    t.free()
