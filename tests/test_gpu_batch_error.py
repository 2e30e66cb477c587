"""Length of the FP32 sums in the batched row pass.

A stage with the LES outputs sums runs of 64 sources in FP32, and the stages
without them do too: the velocity's rounding error against FP64 is then the
same in both.  Runs of 128 would carry up to sqrt(2) of it; the bar is half
way, 2^(1/4), on the mean over the sets.
"""
import numpy as np
import pytest

from openonda_amd import _lib as L
from openonda_amd import batch as B
from openonda_amd import flow_models as FM

pytestmark = pytest.mark.gpu

STAGES = [L.OUT_VEL | L.OUT_STRETCH, L.OUT_VEL | L.OUT_STRETCH | L.OUT_PSE]


def test_later_stages_sum_as_short_runs_as_the_first(gpu):
    sets = []
    for i, n in enumerate([4001, 6000, 9000, 12345, 5003, 7777, 10007, 8192]):
        x, a, s, _ = FM.random_cloud(n, seed=i) if i % 2 else FM.torus_ring(-(-n // 64))
        sets.append((x[:n], a[:n], s[:n], np.full(n, 1e-3)))
    bs, ref = (B.BatchedSystem(sets, dt=0.01, precision=p) for p in ("f32c", "f64"))
    ref.evaluate(ref.x, ref.a, ref.stage_mask, True, ref.stream.cuda_stream)
    ref.synchronize()

    def error(mask):
        bs.evaluate(bs.x, bs.a, mask, True, bs.stream.cuda_stream)
        bs.synchronize()
        e = [float((bs.vel[:, q] - ref.vel[:, q]).norm() / ref.vel[:, q].norm())
             for q in map(bs.set_slice, range(bs.nsets))]
        return np.exp(np.mean(np.log(e)))

    first = error(bs.stage_mask)
    for mask in STAGES:
        print(f"[batch-error] mask {mask}", flush=True)
        assert error(mask) <= 2 ** 0.25 * first, mask
