"""The serving kernel's split of a batch: its (tile, frustum) pairs are divided
equally over the waves, so a wave's run may start and end inside a tile's list of
frusta and pass over several requests.  Batches whose totals leave a wave one pair,
a few, or several tiles, with sizes at the edges of a tile, against the oracle."""
import numpy as np
import pytest

from gpu_util import mismatches
from pipeline_amd import scenes as S
from pipeline_amd.serving import Server

pytestmark = pytest.mark.gpu

BATCHES = [
    [(1, 1)],
    [(64, 64)],
    [(65, 1), (1, 63), (127, 2), (129, 64)],
    [(9_999, 7), (1, 64), (20_033, 64), (64, 1)],
    [(300_000, 33), (2_000, 5), (150_007, 64)],
]


@pytest.mark.parametrize("per_lane", [1, 2])
@pytest.mark.parametrize("batch", BATCHES, ids=lambda b: "+".join(f"{n}x{f}" for n, f in b))
def test_serve_split_matches_oracle(orc, batch, per_lane):
    rng = np.random.default_rng(len(batch))
    with Server(max_scenes=8, max_batch_requests=8, streams=1, objects_per_lane=per_lane) as srv:
        requests, want = [], []
        for n, frusta in batch:
            lower = rng.uniform(-200, 200, (n, 3)).astype(np.float32)
            upper = lower + rng.uniform(0.1, 5.0, (n, 3)).astype(np.float32)
            mats = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
            mats[:, 3, :3] = rng.uniform(-20, 20, (n, 3))
            vps = np.stack([S.perspective_vp(rng.uniform(-50, 50, 3), rng.normal(size=3), 60.0, 1.5, 0.1, 500.0)
                            for _ in range(frusta)]).astype(np.float32)
            sid = srv.add_scene(lower, upper, mats)
            masks = np.full(srv.mask_words(sid, frusta), ~np.uint64(0), np.uint64)
            requests.append((sid, vps, masks, n))
            l4, e4 = S.extents(lower, upper)
            obbs = orc.obb_build_group(l4, e4, np.arange(n), mats.reshape(-1, 16))
            want.append([orc.cull_obbs(obbs, vp) for vp in vps])
        for rid in [srv.submit(sid, vps, masks) for sid, vps, masks, _ in requests]:
            assert srv.wait(rid, 60_000.0).status == 0
    for (_, vps, masks, n), rows in zip(requests, want):
        words = (n + 63) // 64
        for f, row in enumerate(rows):
            got = masks[f * words:(f + 1) * words]
            assert mismatches(got, row, n) == 0
            assert n % 64 == 0 or int(got[-1]) >> (n % 64) == 0
