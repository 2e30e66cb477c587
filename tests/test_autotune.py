"""The autotuners' candidates: the row pass (configuration -1) among the tile
shapes, and no winner of a cache made without it."""
import json

import pytest
import torch

from openonda_amd import autotune as AT
from openonda_amd import physics as P


@pytest.mark.parametrize("fastest", [0, 1, 3])
def test_the_row_pass_is_a_candidate(monkeypatch, tmp_path, fastest):
    """Timings and sums replaced: whichever of (-1, 0, 1, 2) is fastest is kept."""
    asked, ms = [], iter([1.0 if k == fastest else 2.0 + k for k in range(4)])

    def forward(pos, alpha, sigma, nu, outputs, precision, sigma_mode, tile_config=None):
        if precision == "f32c":
            asked.append(tile_config)
        return {"vel": torch.ones((3, pos.shape[1]), dtype=torch.float64)}

    def timed(fn, reps):
        fn()
        return next(ms)

    monkeypatch.setattr(P, "require_gpu", lambda: None)
    monkeypatch.setattr(P, "tile_configs", lambda: [(512, 1, 512, 64, 0)] * 3)
    monkeypatch.setattr(P, "forward", forward)
    monkeypatch.setattr(AT, "_time", timed)
    x = torch.zeros((3, 1024), dtype=torch.float64)
    path = tmp_path / "cache.json"
    best, report = AT.tune(x, x, x[0], outputs=("vel",), path=path)
    assert asked == [-1, 0, 1, 2] and len(report) == 3
    assert best["config"] == fastest - 1
    assert AT.best_config(1024, ("vel",), path=path, default=99) == fastest - 1


def test_winners_among_tile_shapes_alone_do_not_apply(tmp_path):
    path = tmp_path / "cache.json"
    path.write_text(json.dumps({"fused|f32c|vel|uniform|2^10": {"config": 5},
                                "batch|f32c|mask3|pairs2^20|sets1": {"config": 4, "grid": 256}}))
    assert AT.best_config(1024, ("vel",), path=path) == -1
    assert AT.best_batch_config([1024], 3, path=path) is None


@pytest.mark.gpu
def test_tuned_rows_are_used(gpu, tmp_path):
    import numpy as np

    from openonda_amd import batch as B
    from openonda_amd import flow_models as FM

    sets = []
    for n in (200, 130):  # sets that the default leaves to the tiled launch
        x, a, s, _ = FM.random_cloud(n, seed=n)
        sets.append((x, a, s, np.full(n, 1e-3)))
    path = tmp_path / "cache.json"
    print("[autotune] rows and one shape", flush=True)
    best, report = AT.tune_batch(sets, configs=[-1, 4], grids=[0], reps=1, path=path)
    assert [(r["config"], r["grid"]) for r in report] == [(-1, 0), (4, 0)]
    assert all(r["rel_l2"] <= 1e-6 for r in report)
    bs = B.BatchedSystem(sets, dt=0.01, tile_config="auto", autotune_cache=path)
    assert bs.rows == (best["config"] == -1)
    cache = AT.load_cache(path)
    for e in cache.values():
        e.update(config=-1, grid=0)
    AT.save_cache(cache, path)
    assert B.BatchedSystem(sets, dt=0.01, tile_config="auto", autotune_cache=path).rows
    assert not B.BatchedSystem(sets, dt=0.01).rows
