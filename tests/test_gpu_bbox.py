"""dpc_bbox where its folds can differ from Box4f::update's comparisons: corners that
are NaN, infinite, denormal or zero of either sign, objects without a matrix, and
counts around a wave, a workgroup and a round.  Bit for bit against the oracle."""
import numpy as np
import pytest

from pipeline_amd import scenes

from test_gpu_reduce import gpu_bbox

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("kind", ["zeros", "denormal", "infinite", "nan", "none"])
@pytest.mark.parametrize("n", [1, 64, 65, 257, 40_001, 300_007])
def test_bbox_special_values(orc, n, kind):
    rng = np.random.default_rng(n)
    k = max(n // 3, 2)
    lower, upper = scenes.random_boxes(rng, n, (-10.0, 10.0))
    mats = scenes.trs_matrices(rng, k)
    xform = rng.integers(0, k, n)
    at = rng.random(n) < 0.3
    if kind == "zeros":  # a floor of zeros of both signs: every wave, lane and round has some
        mats[:, :3, :3] = np.eye(3, dtype=F)
        mats[:, 3, :3] = np.where(rng.random((k, 3)) < 0.5, F(-0.0), F(0.0))
        lower, upper = np.abs(lower), np.abs(lower) + np.abs(upper)
        lower[at] = np.where(rng.random((int(at.sum()), 3)) < 0.5, F(-0.0), F(0.0))
    elif kind == "denormal":
        mats[:, :3, :3] = np.eye(3, dtype=F)
        mats[:, 3, :3] = 0
        lower, upper = lower * F(1e-41), upper * F(1e-41)
    elif kind == "infinite":
        lower[at, rng.integers(0, 3)] = -np.inf
        upper[rng.random(n) < 0.2, 1] = np.finfo(F).max
    elif kind == "nan":
        lower[at] = np.nan
        mats[: k // 2, 0, 1] = np.inf
    else:  # no object has a matrix, or half of them
        xform[at | (n == 1)] = k + 7
    got = gpu_bbox(lower, upper, mats, xform.astype(np.uint32))
    keep = xform < k
    with np.errstate(all="ignore"):
        l4, e4 = scenes.extents(lower[keep], upper[keep])
    want = orc.bbox_group(l4, e4, xform[keep], mats)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
