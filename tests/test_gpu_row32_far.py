"""Far chunks of the FP32-compensated row pass in sets without the moment form:
rows that sum in FP64 per pair do so on every chunk.

Parallel strengths have no stretching: alpha_i x alpha_j and alpha_i . (r x
alpha_j) vanish for every pair.  Summed in FP64 what is left is at most
n 2^-53 = 1e-12 of |alpha_i| sum_j g_ij |alpha_j| / (4 pi) for 9,000 particles
(each rounding of G, crossed with alpha_i; the triple product's share is of
the same order); summed in FP32 it is about 1e-8.  The radii are a hundredth
of the cloud, so almost every chunk is far.
"""
import numpy as np
import pytest
import torch

from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

ALL = ("vel", "stretch", "pse", "vort", "enstrophy")


@pytest.mark.parametrize("outputs,mode", [
    (("stretch",), "uniform"), (("stretch",), "general"), (("vel", "stretch"), "general"),
    (("vel", "stretch", "pse"), "general"), (("stretch", "vort", "enstrophy"), "general"),
    (("vel", "stretch", "vort", "enstrophy"), "general"), (ALL, "general")],
    ids=lambda v: "-".join(v) if isinstance(v, tuple) else v)
def test_parallel_strengths_do_not_stretch(gpu, outputs, mode):
    n = 9000
    rng = np.random.default_rng(5)
    x = rng.uniform(-1, 1, (n, 3))
    a = rng.uniform(0.5, 1.5, (n, 1)) * np.array([0.3, -0.7, 0.45]) / n
    s = np.full(n, 0.01) if mode == "uniform" else rng.uniform(0.005, 0.02, n)
    nu = np.full(n, 1e-3)
    print(f"[row32-far] {outputs} {mode}", flush=True)
    got = P.from_soa(P.forward(P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(),
                               torch.from_numpy(nu).cuda(), outputs=outputs, precision="f32c",
                               sigma_mode=mode)["stretch"])
    for i in range(0, n, 90):
        r2 = ((x[i] - x) ** 2).sum(1)
        sg = 0.5 * (s[i] + s)
        g = (r2 + 2.5 * sg ** 2) / (r2 + sg ** 2) ** 2.5
        g[i] = 0.0
        bound = np.linalg.norm(a[i]) * (g * np.linalg.norm(a, axis=1)).sum() / (4 * np.pi)
        assert np.linalg.norm(got[i]) <= 1e-12 * bound, i
