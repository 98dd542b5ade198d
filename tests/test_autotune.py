"""The lookup of tuned launch shapes, on the CPU: a shape that was measured, or one
about as large, gets its config; any other gets the plan's defaults."""
import pytest

from pipeline_amd import autotune


@pytest.fixture
def table(monkeypatch):
    entries = {"obj2^21-tests2^23-frusta64": {"config": [1, 256, 24, 16]}, "obj2^20-tests2^22-frusta32": {"config": [2, 128, 8, 4]}}
    monkeypatch.setattr(autotune, "load_table", lambda arch=None: {"batch": entries})


@pytest.mark.parametrize("objects,tests,frusta,want", [
    (1 << 21, 8_870_000, 64, 16), (2_500_000, 9_000_000, 50, 16), (1 << 20, 1 << 22, 32, 4), (1_000_000, 5_000_000, 20, 4),
    (20_000, 160_000, 8, None), (1 << 21, 8_870_000, 8, None), (1 << 21, 1 << 27, 64, None), (1 << 15, 1 << 21, 64, None), (0, 0, 0, None)])
def test_only_near_shapes_are_tuned(table, objects, tests, frusta, want):
    cfg = autotune.best_batch_config(objects, tests, frusta, "any")
    assert (cfg and cfg.max_frusta_per_item) == want


def test_no_table():
    assert autotune.best_batch_config(1 << 21, 1 << 23, 64, "an arch without a table") is None


def test_candidates_hold_whole_lists_and_the_plans_own_chunk():
    for quick in (False, True):
        chunks = {c[3] for c in autotune.batch_candidates(quick)}
        assert {0, 16} <= chunks
    assert 64 in {c[3] for c in autotune.batch_candidates()}


@pytest.mark.parametrize("default_us,want", [(36.5, [1, 256, 24, 16]), (37.0, [2, 256, 16, 0])])
def test_default_shape_wins_within_two_percent(default_us, want):
    rows = [{"config": c, "us": us} for c, us in (([2, 256, 16, 0], 36.0), ([1, 256, 24, 4], 50.0), ([1, 256, 24, 16], default_us))]
    assert autotune._best(rows)["config"] == want
