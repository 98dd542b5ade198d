"""Serving requests of few frusta take the exact test at once, others the quick test
first.  Both sides of that line, alone and in one batch (a wave's run then passes from
one to the other), perspective, parallel and without any plane that the quick test could
use, at the edges of a tile and with many tiles a wave, against the oracle."""
import numpy as np
import pytest

from gpu_util import mismatches
from pipeline_amd import scenes as S
from pipeline_amd.serving import Server

pytestmark = pytest.mark.gpu

BATCHES = [
    [(1, 1)],
    [(64, 2), (65, 3)],
    [(127, 3), (128, 1), (129, 2), (1, 2), (63, 1)],
    [(9_999, 1), (64, 64), (20_033, 2), (10_001, 3)],
    [(700_001, 1)],
    [(500_003, 2), (300_007, 3), (400_001, 1)],
]


def frusta_of(count, rng, kind):
    if kind == "parallel":
        scale = np.diag([0.02, 0.015, 0.01, 1.0])
        vps = [scale @ np.linalg.qr(np.pad(rng.normal(size=(3, 3)), (0, 1)) + np.diag([0, 0, 0, 1.0]))[0]
               for _ in range(count)]
    else:
        vps = [S.perspective_vp(rng.uniform(-50, 50, 3), rng.normal(size=3), 60.0, 1.5, 0.1, 500.0)
               for _ in range(count)]
    vps = np.stack(vps).astype(np.float32)
    if kind == "zero":
        vps[0] = 0.0
    return vps


@pytest.mark.parametrize("kind", ["perspective", "parallel", "zero"])
@pytest.mark.parametrize("per_lane", [1, 2])
@pytest.mark.parametrize("batch", BATCHES, ids=lambda b: "+".join(f"{n}x{f}" for n, f in b))
def test_few_frusta_match_oracle(orc, batch, per_lane, kind):
    rng = np.random.default_rng(len(batch) + per_lane)
    with Server(max_scenes=8, max_batch_requests=8, streams=1, objects_per_lane=per_lane) as srv:
        requests, want = [], []
        for n, frusta in batch:
            lower = rng.uniform(-200, 200, (n, 3)).astype(np.float32)
            upper = lower + rng.uniform(0.1, 5.0, (n, 3)).astype(np.float32)
            mats = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
            mats[:, 3, :3] = rng.uniform(-20, 20, (n, 3))
            mats[::7, 0, 3] = 0.001  # some projective: the quick test leaves them out
            vps = frusta_of(frusta, rng, kind)
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
