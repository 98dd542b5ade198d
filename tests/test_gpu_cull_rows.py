"""The flat cull on both sides of the lines between workgroups of one wave and of 1024
threads: three quarters of a row of CUs, a whole row, and the ends of a workgroup.
Masks, and the fused diff's mask and count, against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as orc
from pipeline_amd import _lib, scenes
from pipeline_amd import device as dev

from gpu_util import mismatches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [191 * 1024, 191 * 1024 + 1, 192 * 1024, 192 * 1024 + 65, 256 * 1024, 256 * 1024 + 1, 384 * 1024, 383 * 1024 + 63])
def test_rows(n):
    rng = np.random.default_rng(n)
    lower, upper = scenes.random_boxes(rng, n, (-300.0, 300.0))
    mats = scenes.trs_matrices(rng, n)
    scene = dev.upload_scene(lower, upper, mats)
    vp = scenes.perspective_vp((0, 0, 0), rng.normal(size=3), 60.0, 1.5, 0.1, 900.0)
    l4, e4 = scenes.extents(lower, upper)
    want = orc.cull_obbs(orc.obb_build_group(l4, e4, np.arange(n), mats), vp)
    assert mismatches(dev.cull(scene, vp).download(), want, n) == 0
    lib, words = _lib.load(), dev.mask_words(n)
    old, mask = dev.DeviceArray(words, np.uint64), dev.DeviceArray(words, np.uint64)
    changed, count = dev.DeviceArray(n, np.uint32), dev.DeviceArray(1, np.uint32)
    ws = dev.DeviceArray((lib.dpc_cull_diff_workspace(n) + 7) // 8, np.uint64)
    old.fill_u32(0)
    _lib.check(lib.dpc_cull_diff(scene.box_a.ptr, scene.box_b.ptr, None, n, scene.planes.ptr, scene.ld, dev.vp_arg(vp), mask.ptr,
                                 old.ptr, changed.ptr, count.ptr, 1, ws.ptr, None))
    assert mismatches(mask.download(), want, n) == 0
    visible = np.flatnonzero(np.unpackbits(want.view(np.uint8), bitorder="little")[:n]).astype(np.uint32)
    assert int(count.download()[0]) == visible.size and np.array_equal(changed.download()[:visible.size], visible)
