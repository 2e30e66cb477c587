"""The FP64 adjoint rows at the edges of rows, waves and splits, for every
subset of cotangents, against torch.autograd of the FP64 oracle, in both
precisions (the FP32-compensated precision runs these rows up to 5,120).

Bar 1e-11, the one tests/test_gpu_adjoint.py holds the FP64 adjoint to.
"""
import itertools

import pytest
import torch

from oracle import vpm_torch as T
from openonda_amd import autograd as AG

pytestmark = pytest.mark.gpu

TOL = 1e-11
SUBSETS = [s for s in itertools.product((0, 1), repeat=3) if any(s)]


def particles(n):
    g = torch.Generator().manual_seed(n)
    x = 2 * torch.rand(n, 3, dtype=torch.float64, generator=g) - 1
    a = torch.randn(n, 3, dtype=torch.float64, generator=g) / n
    s = 0.2 + 0.2 * torch.rand(n, dtype=torch.float64, generator=g)
    nu = 1e-3 * (1 + 4 * torch.rand(n, dtype=torch.float64, generator=g))
    cots = [torch.randn(3, n, dtype=torch.float64, generator=g) for _ in range(3)]
    return x.cuda(), a.cuda(), s.cuda(), nu.cuda(), [c.cuda() for c in cots]


@pytest.mark.parametrize("subset", SUBSETS)
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 517, 1100])
def test_subsets_at_row_edges(gpu, n, subset):
    x, a, s, nu, cots = particles(n)
    cots = [c if f else None for c, f in zip(cots, subset)]
    tx, ta = x.clone().requires_grad_(True), a.clone().requires_grad_(True)
    outs = T.pair_sums(tx, ta, s, nu)
    loss = sum((c.t() * o).sum() for c, o in zip(cots, outs) if c is not None)
    ref = [r.t() for r in torch.autograd.grad(loss, (tx, ta))]
    d = (x.t().contiguous(), a.t().contiguous(), s, nu)
    for prec in ("f64", "f32c"):
        for kw in ({}, {"max_splits": 1}, {"max_splits": 3}):
            print(f"[adj64] n={n} {subset} {prec} {kw}", flush=True)
            got = AG.adjoint(*d, *cots, precision=prec, sigma_mode="general", **kw)
            for g, r in zip(got, ref):
                assert float((g - r).norm()) <= TOL * float(r.norm()), (prec, kw)
