"""The FP32-compensated adjoint rows at the edges of rows, chunks and splits,
for every subset of cotangents, against the FP64 adjoint.

Bar 2e-5, the one tests/test_gpu_adjoint.py holds the FP32-compensated adjoint
to: sparse rings cancel most of the stretching's gradient (4e-6 measured).
"""
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

TOL = 2e-5
SUBSETS = [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, 1, 1)]


def particles(layout, n, general, seed):
    x, a, s, _ = FM.torus_ring(-(-n // 64)) if layout == "ring" else FM.random_cloud(n, seed=seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = [P.to_soa(x[:n]), P.to_soa(a[:n]), torch.from_numpy(s[:n].copy()).cuda()]
    if general:
        d[2] = d[2] * (0.7 + 0.7 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g))
    d.append(1e-3 * (1 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g)))
    cots = [torch.randn(3, n, dtype=torch.float64, device="cuda", generator=g) for _ in range(3)]
    return d, cots


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("subset", SUBSETS)
@pytest.mark.parametrize("layout", ["cloud", "ring"])
def test_subsets_at_row_edges(gpu, layout, subset, general):
    mode = "general" if general else "uniform"
    for n in (2, 63, 65, 700, 4097, 5121, 5184, 5185, 12345):
        print(f"[adj32] {layout} n={n} {subset} general={general}", flush=True)
        d, cots = particles(layout, n, general, n)
        cots = [c if f else None for c, f in zip(cots, subset)]
        ref = AG.adjoint(*d, *cots, precision="f64", sigma_mode=mode)
        for kw in ({}, {"max_splits": 1}, {"max_splits": 3}):
            got = AG.adjoint(*d, *cots, precision="f32c", sigma_mode=mode, **kw)
            for g, r in zip(got, ref):
                assert float((g - r).norm()) <= TOL * float(r.norm()), (n, kw)


def test_one_particle_and_no_cotangents(gpu):
    d, cots = particles("cloud", 1, False, 1)
    for got in AG.adjoint(*d, *cots, precision="f32c", sigma_mode="uniform"):
        assert not got.any()
    d, _ = particles("cloud", 300, False, 2)
    for got in AG.adjoint(*d, precision="f32c", sigma_mode="uniform"):
        assert not got.any()


def test_same_bits_every_time(gpu):
    d, cots = particles("ring", 9001, False, 3)
    one = AG.adjoint(*d, *cots, precision="f32c", sigma_mode="uniform")
    two = AG.adjoint(*d, *cots, precision="f32c", sigma_mode="uniform")
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])
