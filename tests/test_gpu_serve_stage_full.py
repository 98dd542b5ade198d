"""A serving batch of as many requests as one can hold, each with a delta: one launch
scatters all of them.  Every scene's matrices are read back and equal the host's."""
import numpy as np
import pytest

from pipeline_amd import scenes as S
from pipeline_amd.serving import Server

pytestmark = pytest.mark.gpu

SCENES, WAVES, LONG = 64, 3, 1_000_000


@pytest.mark.parametrize("most", [3, 200, 900])  # 1.5 MB in all of 900: copied before the launch
def test_serve_stage_of_a_full_batch(most):
    rng = np.random.default_rng(most)
    vps = np.stack([S.perspective_vp((0, 0, 0), (0, 0, 1), 60.0, 1.5, 0.1, 100.0)]).astype(np.float32)
    with Server(max_scenes=SCENES, max_batch_requests=SCENES, streams=1, batches_per_stream=1) as srv:
        held = []
        for i in range(SCENES):
            n = most + int(rng.integers(1, 100)) if i else LONG
            lower = rng.uniform(-10, 10, (n, 3)).astype(np.float32)
            mats = rng.normal(size=(n, 4, 4)).astype(np.float32)
            mats[:, :, 3] = [0, 0, 0, 1]
            sid = srv.add_scene(lower, lower + 1, mats)
            held.append((sid, mats, np.zeros(srv.mask_words(sid, 1), np.uint64)))
        # a long first batch: all of the next requests wait for it, and the second takes
        # one of each scene
        sid, mats, masks = held[0]
        requests = [(sid, vps, masks, np.arange(LONG, dtype=np.uint32), mats.copy())]
        for _ in range(WAVES):
            for i, (sid, mats, masks) in enumerate(held):
                k = 1 + int(rng.integers(most))
                idx = rng.permutation(mats.shape[0])[:k].astype(np.uint32)
                new = rng.normal(size=(k, 4, 4)).astype(np.float32)
                if i % 3:
                    new[:, :, 3] = [0, 0, 0, 1]
                mats[idx] = new
                requests.append((sid, vps, masks, idx, new))
        done = [srv.wait(rid, 60_000.0) for rid in [srv.submit(*r) for r in requests]]
        assert all(d.status == 0 for d in done)
        assert max(d.batch_requests for d in done) == SCENES
        for sid, mats, _ in held:
            assert np.array_equal(srv.read_matrices(sid).view(np.uint32), mats.reshape(-1, 16).view(np.uint32))
