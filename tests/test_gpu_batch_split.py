"""dpc_batch_config.max_frusta_per_item: an explicit 0 splits no list, n cuts lists
into chunks of n at most, and only without a config does the plan choose."""
import numpy as np
import pytest

from pipeline_amd import _lib, scenes
from pipeline_amd import device as dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frusta", [1, 16, 17, 64, 65])
@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_chunks(lanes, frusta):
    rng = np.random.default_rng(frusta)
    n = 1_000
    tiles, words = -(-n // (64 * lanes)), (n + 63) // 64
    scene = dev.upload_scene(*scenes.random_boxes(rng, n, (-50.0, 50.0)), scenes.trs_matrices(rng, n))
    vps = np.stack([scenes.perspective_vp(rng.uniform(-20, 20, 3), rng.normal(size=3), 60, 1.5, 0.1, 100) for _ in range(frusta)]).astype(np.float32)
    d_vps = dev.DeviceArray.from_host(vps.reshape(-1, 16))
    results = []
    for cfg, items in ((_lib.BatchConfig(lanes, 256, 8, 0), tiles), (_lib.BatchConfig(lanes, 256, 8, 5), tiles * -(-frusta // 5)),
                       (_lib.BatchConfig(lanes, 256, 8, 1_000), tiles), (None, None)):
        plan = dev.BatchPlan([(0, 0, n)], [(f, 0, f * words) for f in range(frusta)], frusta, cfg)
        assert items is None or plan.items == items
        plan.bind([scene])
        masks = dev.DeviceArray(frusta * words, np.uint64)
        plan.cull(d_vps, masks)
        results.append(masks.download())
        plan.destroy()
        masks.free()
    assert all(np.array_equal(results[0], r) for r in results[1:])
    scene.free()
    d_vps.free()
