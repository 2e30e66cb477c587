"""A few sources at very many points: a row per wave, against the drop-in rows
of fewer points (pinned to the oracle elsewhere).  The same terms in another
order: rel-L2 <= 1e-13."""
import numpy as np
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [6143 * 64 + 1, 6150 * 64 + 65])  # 6144 rows, and a ragged last workgroup
@pytest.mark.parametrize("n", [0, 1, 3, 8, 9])
def test_points(gpu, n, m):
    rng = np.random.default_rng(n)
    x, a = P.to_soa(rng.uniform(-1, 1, (n, 3))), P.to_soa(rng.normal(size=(n, 3)))
    s = torch.from_numpy(rng.uniform(0.1, 0.3, n)).cuda()
    g = torch.Generator(device="cuda").manual_seed(n)
    y = torch.rand((3, m), dtype=torch.float64, device="cuda", generator=g)
    print(f"[few-sources] n={n} m={m}", flush=True)
    for f in (P.induced_velocity_at, P.vorticity_field_at,
              lambda *q: P.vorticity_field_at(*q, variant="cpu")):
        got = f(y, x, a, s)
        if n == 0:
            assert not got.any()
            continue
        half = m // 2
        ref = torch.cat([f(y[:, :half], x, a, s), f(y[:, half:], x, a, s)], 1)
        assert float((got - ref).norm() / ref.norm()) <= 1e-13


def test_gradient_of_very_many_particles_at_a_point(gpu):
    n = 6144 * 64 + 3
    g = torch.Generator(device="cuda").manual_seed(1)
    x, a = (torch.rand((3, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    s = torch.full((n,), 0.1, dtype=torch.float64, device="cuda")
    y = torch.rand((3, 2), dtype=torch.float64, device="cuda", generator=g)
    cot = torch.ones_like(y)
    print("[few-sources] gradient", flush=True)

    def grads(x, a, s):
        x, a = x.clone().requires_grad_(), a.clone().requires_grad_()
        return torch.autograd.grad(AG.probe_velocity(y, x, a, s), (x, a), cot)

    half = n // 2
    parts = [grads(x[:, q], a[:, q], s[q]) for q in (slice(0, half), slice(half, n))]
    for got, lo, hi in zip(grads(x, a, s), *parts):
        ref = torch.cat([lo, hi], 1)
        assert float((got - ref).norm() / ref.norm()) <= 1e-13
