"""The FP32-compensated adjoint rows above their first size (5,121 particles):
ragged and whole rows, waves that sweep more than one window of 64 chunks, and
no cotangent at all.  Bar 2e-5 against the FP64 adjoint, as in
tests/test_gpu_adj32.py.
"""
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

TOL = 2e-5


def particles(layout, n, general):
    x, a, s, _ = FM.torus_ring(-(-n // 64)) if layout == "ring" else FM.random_cloud(n, seed=n)
    g = torch.Generator(device="cuda").manual_seed(n)
    d = [P.to_soa(x[:n]), P.to_soa(a[:n]), torch.from_numpy(s[:n].copy()).cuda()]
    if general:
        d[2] = d[2] * (0.7 + 0.7 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g))
    d.append(1e-3 * (1 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g)))
    return d, [torch.randn(3, n, dtype=torch.float64, device="cuda", generator=g) for _ in range(3)]


# 8 waves x 64 chunks x 64 particles are the first window of an unsplit row
@pytest.mark.parametrize("n", [5183, 5248, 5249, 32768, 32769, 40000])
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("layout", ["cloud", "ring"])
def test_rows_and_windows(gpu, layout, general, n):
    print(f"[adj32-windows] {layout} n={n} general={general}", flush=True)
    mode = "general" if general else "uniform"
    d, cots = particles(layout, n, general)
    ref = AG.adjoint(*d, *cots, precision="f64", sigma_mode=mode)
    for kw in ({}, {"max_splits": 1}):
        got = AG.adjoint(*d, *cots, precision="f32c", sigma_mode=mode, **kw)
        for g, r in zip(got, ref):
            assert float((g - r).norm()) <= TOL * float(r.norm()), kw


def test_no_cotangents(gpu):
    d, _ = particles("cloud", 6001, False)
    for got in AG.adjoint(*d, precision="f32c", sigma_mode="uniform"):
        assert not got.any()
