"""The single-view cull over a long array whose objects share matrices, where a wave
takes two adjacent tiles: counts that end in the first or the second tile of a wave,
on both sides of the lines where that form is taken, and indices outside the matrix
array.  Masks, counts and changed indices against the oracle, bit for bit.  And the
line between workgroups of one wave and of many."""
import numpy as np
import pytest

from oracle import oracle as orc
from pipeline_amd import _lib, scenes
from pipeline_amd import device as dev

from gpu_util import mismatches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,share", [(1_399_999, 4), (1_400_000, 4), (1_400_001, 3), (1_400_064, 4), (1_400_065, 4),
                                     (1_400_127, 7), (1_400_128, 4), (1_400_129, 2), (1_500_033, 1_000)])
def test_cull_pair_matches_oracle(n, share):
    rng = np.random.default_rng(n + share)
    k = n // share
    lower, upper = scenes.random_boxes(rng, n, (-300.0, 300.0))
    mats = scenes.trs_matrices(rng, k)
    xform = np.minimum(np.arange(n) // share, k - 1).astype(np.uint32)
    xform[rng.random(n) < 0.001] = k + 3
    scene = dev.upload_scene(lower, upper, mats, xform)
    vps = [scenes.perspective_vp(rng.uniform(-50, 50, 3), rng.normal(size=3), 60.0, 1.5, 0.1, 900.0) for _ in range(2)]
    bad = xform >= k
    l4, e4 = scenes.extents(lower, upper)
    obbs = orc.obb_build_group(l4, e4, np.where(bad, 0, xform), mats)
    words = dev.mask_words(n)
    always = np.zeros(64 * words, np.uint8)
    always[:n] = bad
    always = np.packbits(always, bitorder="little").view(np.uint64)
    want = [orc.cull_obbs(obbs, vp) | always for vp in vps]
    got = dev.cull(scene, vps[0]).download()
    assert mismatches(got, want[0], n) == 0
    assert n % 64 == 0 or int(got[-1]) >> (n % 64) == 0
    # the same with the result's diff: from the first view's bits to the second's
    lib = _lib.load()
    old, mask = dev.DeviceArray(words, np.uint64), dev.DeviceArray(words, np.uint64)
    changed, count = dev.DeviceArray(n, np.uint32), dev.DeviceArray(1, np.uint32)
    ws = dev.DeviceArray((lib.dpc_cull_diff_workspace(n) + 7) // 8, np.uint64)
    old.upload(want[0])
    _lib.check(lib.dpc_cull_diff(scene.box_a.ptr, scene.box_b.ptr, scene.xform_addr, n, scene.planes.ptr, scene.ld,
                                 dev.vp_arg(vps[1]), mask.ptr, old.ptr, changed.ptr, count.ptr, 1, ws.ptr, None))
    assert mismatches(mask.download(), want[1], n) == 0 and mismatches(old.download(), want[1], n) == 0
    bits = np.unpackbits((want[0] ^ want[1]).view(np.uint8), bitorder="little")[:n]
    index = np.flatnonzero(bits).astype(np.uint32)
    assert int(count.download()[0]) == index.size
    assert np.array_equal(changed.download()[:index.size], index)


@pytest.mark.parametrize("share", [0, 4])
@pytest.mark.parametrize("n", [1, 64, 65, 899_999, 900_000, 900_001])
def test_cull_workgroup_sizes(n, share):
    rng = np.random.default_rng(n + share)
    k = max(n // share, 1) if share else n
    lower, upper = scenes.random_boxes(rng, n, (-300.0, 300.0))
    mats = scenes.trs_matrices(rng, k)
    xform = np.minimum(np.arange(n) // share, k - 1).astype(np.uint32) if share else None
    vp = scenes.perspective_vp((0, 0, 0), rng.normal(size=3), 60.0, 1.5, 0.1, 900.0)
    got = dev.cull(dev.upload_scene(lower, upper, mats, xform), vp).download()
    l4, e4 = scenes.extents(lower, upper)
    want = orc.cull_obbs(orc.obb_build_group(l4, e4, np.arange(n) if xform is None else xform, mats), vp)
    assert mismatches(got, want, n) == 0
    assert n % 64 == 0 or int(got[-1]) >> (n % 64) == 0
