"""The batched and the serving cull where the quick test leaves pairs undecided
(pipeline_amd/csrc/quick_cull.hpp): the queue of pairs that wait for the exact
test filling up within one work item, across items and at the end, frusta counts
on both sides of the LDS table, lists longer than a slice, and lanes with no
object or a matrix index outside the array.  Masks against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as orc
from pipeline_amd import _lib, scenes
from pipeline_amd import device as dev
from pipeline_amd.serving import Server

from gpu_util import mismatches

pytestmark = pytest.mark.gpu


def make_scene(n, undecided, seed):
    """n objects; a share `undecided` of the matrices has a last column of its own, which
    the quick test leaves to the exact one; some indices lie outside the matrix array."""
    rng = np.random.default_rng(seed)
    k = max(n // 2, 1)
    lower, upper = scenes.random_boxes(rng, n, (-50.0, 50.0), (0.1, 6.0))
    mats = scenes.trs_matrices(rng, k)
    odd = rng.random(k) < undecided
    mats[odd, :3, 3] = rng.normal(scale=0.01, size=(int(odd.sum()), 3)).astype(np.float32)
    xform = rng.integers(0, k, n).astype(np.uint32)
    xform[rng.random(n) < 0.01] = k + 5
    return lower, upper, mats, xform


def cameras(rng, count):
    return np.stack([scenes.perspective_vp(rng.uniform(-20, 20, 3), rng.normal(size=3), rng.uniform(30, 90), 16 / 9, 0.1,
                                           rng.uniform(20, 200)) for _ in range(count)]).astype(np.float32)


def oracle_masks(lower, upper, mats, xform, vps):
    l4, e4 = scenes.extents(lower, upper)
    bad = xform >= mats.shape[0]
    obbs = orc.obb_build_group(l4, e4, np.where(bad, 0, xform), mats)
    always = np.zeros((lower.shape[0] + 63) // 64 * 64, np.uint8)
    always[:lower.shape[0]] = bad
    always = np.packbits(always, bitorder="little").view(np.uint64)
    return [orc.cull_obbs(obbs, vp) | always for vp in vps]


@pytest.mark.parametrize("undecided", [0.0, 0.3, 1.0])
@pytest.mark.parametrize("n,frusta,cfg", [
    (1, 1, None), (63, 3, None), (64, 128, None), (65, 129, None), (4_097, 17, None), (40_001, 33, None),
    (4_097, 70, (1, 256, 1, 70)), (4_097, 129, (2, 64, 4, 0)), (1_000, 40, (2, 256, 2, 40)), (1_025, 130, (4, 128, 1, 130)),
    (5_000, 20, (4, 256, 8, 3)),
    (4_097, 15, None), (4_097, 16, (1, 256, 24, 64)), (1_000, 31, (2, 256, 16, 64)), (1_000, 32, (4, 256, 8, 64)),
    (200, 144, (1, 256, 24, 144))])
def test_batch_masks(n, frusta, cfg, undecided):
    rng = np.random.default_rng(n + frusta)
    lower, upper, mats, xform = make_scene(n, undecided, n)
    vps = cameras(rng, frusta)
    words = (n + 63) // 64
    scene = dev.upload_scene(lower, upper, mats, xform)
    plan = dev.BatchPlan([(0, 0, n)], [(f, 0, f * words) for f in range(frusta)], frusta,
                         None if cfg is None else _lib.BatchConfig(*cfg))
    plan.bind([scene])
    d_vps = dev.DeviceArray.from_host(vps.reshape(-1, 16))
    masks = dev.DeviceArray(frusta * words, np.uint64)
    masks.fill_u32(0xA5A5A5A5)
    plan.cull(d_vps, masks)
    got = masks.download().reshape(frusta, words)
    for f, want in enumerate(oracle_masks(lower, upper, mats, xform, vps)):
        assert mismatches(got[f], want, n) == 0, f"frustum {f}"
    plan.destroy()
    for d in (scene, d_vps, masks):
        d.free()


@pytest.mark.parametrize("lanes", [1, 2])
@pytest.mark.parametrize("undecided", [0.0, 1.0])
def test_serving_masks(lanes, undecided):
    rng = np.random.default_rng(lanes)
    sizes, counts = (1, 64, 10_007, 129, 3_000), (64, 1, 64, 33, 5)
    with Server(max_scenes=8, streams=2, objects_per_lane=lanes, hbm_budget_bytes=256 << 20) as srv:
        work = []
        for i, (n, frusta) in enumerate(zip(sizes, counts)):
            lower, upper, mats, xform = make_scene(n, undecided, 100 + i)
            sid = srv.add_scene(lower, upper, mats, xform)
            vps = cameras(rng, frusta)
            out = np.zeros(srv.mask_words(sid, frusta), np.uint64)
            work.append((srv.submit(sid, vps, out), n, out, oracle_masks(lower, upper, mats, xform, vps)))
        for rid, n, out, want in work:
            srv.wait(rid)
            for got, w in zip(out.reshape(len(want), -1), want):
                assert mismatches(got, w, n) == 0
