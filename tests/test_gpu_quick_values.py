"""The batched and the serving cull over what the quick test's bound is made for
(pipeline_amd/csrc/quick_cull.hpp), on the matrix cores and with the device's medians:
exact ties, boxes that graze a plane, every magnitude from denormal to overflow,
special values in objects and views, projective objects.  An object's point and edges
are the rows of its matrix (a unit box).  Masks against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as orc
from pipeline_amd import _lib, scenes
from pipeline_amd import device as dev
from pipeline_amd.serving import Server

from gpu_util import mismatches

pytestmark = pytest.mark.gpu
F = np.float32
N, VIEWS = 4_096, 48
ODD = np.array([0, -0.0, 1, -1, 1e-45, -1e-40, 2.0**-126, 2.0**-75, 2.0**-48, 2.0**-47, 2.0**55, 2.0**56, -(2.0**59), 2.0**60, 2.0**63,
                2.0**100, 3e38, -3e38, np.inf, -np.inf, np.nan], F)


def views(rng, ortho=True):
    out = []
    for _ in range(VIEWS):
        eye, direction = rng.uniform(-50, 50, 3), rng.normal(size=3)
        if ortho and rng.random() < 0.5:
            view = scenes.make_lookat(eye, eye + direction, rng.normal(size=3))
            e = rng.uniform(10, 500, 2)
            vp = scenes.view_projection(view, scenes.make_ortho(-e[0], e[0], -e[1], e[1], 0.1, rng.uniform(50, 3000)))
        else:
            vp = scenes.perspective_vp(eye, direction, rng.uniform(20, 120), 1.7, 0.1, rng.uniform(50, 3000))
        out.append(vp)
    return np.stack(out).astype(F)


def objects(rng, extent, size):
    """(N, 4, 4): three edges and the point."""
    m = np.zeros((N, 4, 4))
    m[:, :3, :3] = rng.uniform(-size, size, (N, 3, 3))
    m[:, 3, :3] = rng.uniform(-extent, extent, (N, 3))
    m[:, 3, 3] = 1
    return m.astype(F)


def make(kind, rng):
    with np.errstate(all="ignore"):
        if kind == "ties":  # integer boxes against planes through integers
            m = np.zeros((N, 4, 4), F)
            m[:, :, :3] = rng.integers(-3, 4, (N, 4, 3))
            m[:, 3, 3] = 1
            return m, rng.integers(-1, 2, (VIEWS, 4, 4)).astype(F)
        if kind == "large":
            return objects(rng, 100, 200), views(rng)
        if kind == "projective":
            m = objects(rng, 100, 20)
            m[:, :, 3] = np.where(rng.random((N, 4)) < 0.5, rng.uniform(-2, 2, (N, 4)), m[:, :, 3])
            return m, views(rng)
        if kind == "grazing":  # each box's nearest corner within a few rounding errors of a plane of one view
            m, vps = objects(rng, 500, 2).astype(np.float64), views(rng, False)
            v = vps[np.arange(N) % VIEWS].astype(np.float64)
            axis, sign = rng.integers(0, 3, N), np.where(rng.random(N) < 0.5, 1.0, -1.0)
            n = v[:, :, 3] + sign[:, None] * v[np.arange(N), :, axis]
            far = n[:, 3] + (n[:, :3] * m[:, 3, :3]).sum(1) + np.maximum((m[:, :3, :3] * n[:, None, :3]).sum(2), 0).sum(1)
            move = -far / np.maximum((n[:, :3] ** 2).sum(1), 1e-30) * (1 + rng.uniform(-2, 2, N) * 2.0**-22)
            m[:, 3, :3] += move[:, None] * n[:, :3]
            return m.astype(F), vps
        m, vps = objects(rng, 1000, 2), views(rng)
        if kind == "scaled":  # whole scenes and views by powers of two
            m[:, :, :3] = np.ldexp(m[:, :, :3], rng.integers(-130, 130, (N, 1, 1)))
            m[:, 3, 3] = np.where(rng.random(N) < 0.5, np.ldexp(F(1), rng.integers(-130, 130, N)), 1)
            shift = rng.integers(-130, 130, (VIEWS, 1, 1)) + np.where(rng.random((VIEWS, 4, 4)) < 0.75, 0, rng.integers(-20, 20, (VIEWS, 4, 4)))
            return m, np.ldexp(vps, np.where(np.arange(VIEWS)[:, None, None] % 2, shift, 0))
        if kind == "wild":  # every element by itself
            at, av = rng.random(m.shape) < 0.33, rng.random(vps.shape) < 0.33
            av[::2] = False
            return np.where(at, np.ldexp(m, rng.integers(-100, 100, m.shape)), m), np.where(av, np.ldexp(vps, rng.integers(-100, 100, vps.shape)), vps)
        # special values in any places
        m = objects(rng, 20, 5)
        at, av = rng.random(m.shape) < rng.choice([0.05, 0.2], (N, 1, 1)), rng.random(vps.shape) < 0.1
        av[::2] = False
        return np.where(at, rng.choice(ODD, m.shape), m), np.where(av, rng.choice(ODD, vps.shape), vps)


KINDS = ["ties", "grazing", "scaled", "wild", "odd", "projective", "large"]


def case(kind):
    rng = np.random.default_rng(KINDS.index(kind) + 7)
    m, vps = make(kind, rng)
    lower, upper = np.zeros((N, 3), F), np.ones((N, 3), F)
    l4, e4 = scenes.extents(lower, upper)
    m, vps = np.ascontiguousarray(m, F), np.ascontiguousarray(vps, F)
    obbs = orc.obb_build_group(l4, e4, np.arange(N), m.reshape(-1, 16))
    return lower, upper, m, vps, [orc.cull_obbs(obbs, vp) for vp in vps]


@pytest.mark.parametrize("cfg", [None, (2, 256, 8, 0), (4, 128, 8, 16)])
@pytest.mark.parametrize("kind", KINDS)
def test_batch(kind, cfg):
    lower, upper, m, vps, want = case(kind)
    scene = dev.upload_scene(lower, upper, m)
    plan = dev.BatchPlan([(0, 0, N)], [(f, 0, f * (N // 64)) for f in range(VIEWS)], VIEWS, None if cfg is None else _lib.BatchConfig(*cfg))
    plan.bind([scene])
    d_vps, masks = dev.DeviceArray.from_host(vps.reshape(-1, 16)), dev.DeviceArray(VIEWS * (N // 64), np.uint64)
    plan.cull(d_vps, masks)
    got = masks.download().reshape(VIEWS, -1)
    bad = [mismatches(got[f], want[f], N) for f in range(VIEWS)]
    assert sum(bad) == 0, bad
    plan.destroy()
    for d in (scene, d_vps, masks):
        d.free()


@pytest.mark.parametrize("kind", KINDS)
def test_serving(kind):
    lower, upper, m, vps, want = case(kind)
    with Server(max_scenes=1, hbm_budget_bytes=256 << 20) as srv:
        sid = srv.add_scene(lower, upper, m)
        out = np.zeros(srv.mask_words(sid, VIEWS), np.uint64)
        assert srv.wait(srv.submit(sid, vps, out), 60_000.0).status == 0
    got = out.reshape(VIEWS, -1)
    assert sum(mismatches(got[f], want[f], N) for f in range(VIEWS)) == 0
