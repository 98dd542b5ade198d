"""The serving loop's upload of a batch: deltas scattered out of the batch's arena,
64 matrices at a time, several requests' in one launch, by the kernel that reads the
host's arena itself or, for a batch of more than 1 MiB, after a copy.  Delta sizes at
the edges of the groups of 64, affine matrices and others, requests without a delta
among them; every scene's matrices are read back and equal the host's bit for bit."""
import numpy as np
import pytest

from pipeline_amd import scenes as S
from pipeline_amd.serving import Server

pytestmark = pytest.mark.gpu

BATCHES = [[1], [20_100], [20_200], [0, 63], [64, 65, 0, 127], [128, 129, 1, 4_097, 2], [70_001, 3], [150_000, 64, 40_001]]


@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("deltas", BATCHES, ids=lambda d: "+".join(map(str, d)))
def test_serve_stage_scatters_exactly(deltas, affine):
    rng = np.random.default_rng(len(deltas))
    with Server(max_scenes=8, max_batch_requests=8, streams=1) as srv:
        held = []
        for round_ in range(2):  # (the first request opens the batches; the second round runs on used arenas)
            for i, k in enumerate(deltas):
                if round_ == 0:
                    n = k + 70
                    lower = rng.uniform(-10, 10, (n, 3)).astype(np.float32)
                    mats = rng.normal(size=(n, 4, 4)).astype(np.float32)
                    held.append((srv.add_scene(lower, lower + 1, mats), mats))
                sid, mats = held[i]
                n = mats.shape[0]
                idx = rng.permutation(n)[:k].astype(np.uint32)
                new = rng.normal(size=(k, 4, 4)).astype(np.float32)
                if affine or i % 2:
                    new[:, :, 3] = [0, 0, 0, 1]
                mats[idx] = new
                vps = np.stack([S.perspective_vp((0, 0, 0), (0, 0, 1), 60.0, 1.5, 0.1, 100.0)]).astype(np.float32)
                masks = np.zeros(srv.mask_words(sid, 1), np.uint64)
                held[i] = (sid, mats, (sid, vps, masks, idx, new))
            for rid in [srv.submit(*h[2]) for h in held]:
                assert srv.wait(rid, 60_000.0).status == 0
            for sid, mats, _ in held:
                got = srv.read_matrices(sid)
                assert np.array_equal(got.view(np.uint32), mats.reshape(-1, 16).view(np.uint32))
            held = [h[:2] for h in held]
