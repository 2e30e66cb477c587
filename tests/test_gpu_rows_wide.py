"""FP64 rows, one per wave: sets whose component arrays lie 4 MiB apart.

The same particles behind a component stride of 2^19 run a row per wave and
packed ones the rows that share their sources among eight waves (pinned to the
oracle in test_gpu_rows): the same pair terms summed in another order, so
rel-L2 <= 1e-12 (scalars 1e-11).  Sizes: full workgroups, a last workgroup of
two rows, the second of a single target.
"""
import numpy as np
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

LD = 1 << 19
SIZES = [1 << 18, (1 << 18) + 65]


def rel(a, b):
    return float((a - b).norm() / b.norm())


def particles(n):
    rng = np.random.default_rng(n)
    pack = [torch.from_numpy(t).cuda() for t in
            (rng.uniform(-1, 1, (3, n)), rng.normal(0, 1 / n, (3, n)), rng.uniform(0.1, 0.3, n),
             rng.uniform(1e-4, 1e-2, n))]
    apart = []
    for t in pack[:2]:
        buf = torch.full((3, LD), float("nan"), dtype=torch.float64, device="cuda")
        buf[:, :n] = t
        apart.append(buf[:, :n])
    return pack, apart + pack[2:]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("outputs,mode", [(("vel", "stretch"), "uniform"),
                                          (("vel", "stretch", "pse", "vort", "enstrophy"),
                                           "general")])
def test_row_per_wave_forward(gpu, n, outputs, mode):
    print(f"[rows-wide] n={n} {outputs} {mode}", flush=True)
    pack, apart = particles(n)
    if mode == "uniform":
        pack[2].fill_(0.17)
    for splits in (0, 1):
        ref = P.forward(*pack, outputs=outputs, precision="f64", sigma_mode=mode)
        got = P.forward(*apart, outputs=outputs, precision="f64", sigma_mode=mode,
                        max_splits=splits)
        for k in outputs:
            assert rel(got[k], ref[k]) <= (1e-11 if k == "enstrophy" else 1e-12), (k, splits)


@pytest.mark.parametrize("n", SIZES)
def test_row_per_wave_plain_sums(gpu, n):
    print(f"[rows-wide] plain n={n}", flush=True)
    pack, apart = particles(n)
    for f in (lambda x, a, s, v: P.selfinduced_velocity(x, a, s),
              lambda x, a, s, v: P.strength_gradients(x, a, s),
              lambda x, a, s, v: P.vorticity_field_at(x, x, a, s)):
        assert rel(f(*apart), f(*pack)) <= 1e-12
    cot = torch.randn(3, n, dtype=torch.float64, device="cuda")
    grads = []
    for y in (pack[0], apart[0]):  # points as sources of the gradient's rows
        x, a = (pack[0] + 0.01).requires_grad_(), pack[1].clone().requires_grad_()
        grads.append(torch.autograd.grad(AG.probe_velocity(y, x, a, pack[2]), (x, a), cot))
    for g, r in zip(grads[1], grads[0]):
        assert rel(g, r) <= 1e-12
