"""dpc_bbox over matrices in order and in none: waves whose matrices lie apart read
them row by row, one to three rounds at once, the others round by round.
Orders of indices that choose either, or both within one call, with indices outside
the array, zeros of both signs, NaN and infinities.  Bit for bit against the oracle."""
import numpy as np
import pytest

from pipeline_amd import scenes

from test_gpu_reduce import gpu_bbox

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("order", ["random", "ascending", "spread", "half"])
@pytest.mark.parametrize("n", [65, 100_001, 300_007, 524_288, 524_289, 600_011, 1_100_003])
def test_bbox_scattered_matrices(orc, n, order, special):
    rng = np.random.default_rng(n)
    k = n // 3
    lower, upper = scenes.random_boxes(rng, n, (-10.0, 10.0))
    mats = scenes.trs_matrices(rng, k)
    xform = {"random": lambda: rng.integers(0, k, n),
             "ascending": lambda: np.arange(n) // 3,
             "spread": lambda: np.arange(n) * 8 % k,  # a line each, in order
             "half": lambda: np.where(np.arange(n) < n // 2, np.arange(n) // 3, rng.integers(0, k, n))}[order]()
    if special:
        mats[:, :3, :3] = np.eye(3, dtype=F)
        mats[:, 3, :3] = np.where(rng.random((k, 3)) < 0.5, F(-0.0), F(0.0))
        lower, upper = np.abs(lower), np.abs(lower) + np.abs(upper)
        zero = rng.random(n) < 0.1
        lower[zero] = np.where(rng.random((int(zero.sum()), 3)) < 0.5, F(-0.0), F(0.0))
        lower[rng.random(n) < 0.01, 1] = np.nan
        upper[rng.random(n) < 0.01, 2] = np.inf
        xform = np.where(rng.random(n) < 0.1, k + rng.integers(0, 9, n), xform)
    got = gpu_bbox(lower, upper, mats, xform.astype(np.uint32))
    keep = xform < k
    with np.errstate(all="ignore"):
        l4, e4 = scenes.extents(lower[keep], upper[keep])
    want = orc.bbox_group(l4, e4, xform[keep], mats)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
