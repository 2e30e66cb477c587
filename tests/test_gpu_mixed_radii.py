"""Per-particle radii that differ by many orders of magnitude: the FP32 passes
against the FP64 one.

The first particle's radius (the first of the caller's order and, in the
corner of the box, of the sorted one) is 1e-9 of the distances: lengths in
units of it would leave the range of FP32 in the kernels' fifth powers.  Its
own pairs are like any other's, since sigma_ij is the mean of two radii.
Bar: the passes' rel-L2 <= 1e-6.
"""
import numpy as np
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

TOL = 1e-6


def particles(n):
    rng = np.random.default_rng(n)
    x = rng.uniform(-1000, 1000, (n, 3))
    x[0] = -1000.0
    s = rng.uniform(80, 120, n)
    s[0] = 1e-6
    return (P.to_soa(x), P.to_soa(rng.normal(0, 1, (n, 3))), torch.from_numpy(s).cuda(),
            torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))


def rel(g, r):
    return float((g - r).norm() / r.norm())


@pytest.mark.parametrize("presorted", [False, True])
@pytest.mark.parametrize("outputs", [("vel",), ("stretch",), ("pse",), ("vort",), ("vel", "stretch"),
                                     ("vel", "stretch", "pse"), ("stretch", "vort"),
                                     ("vel", "stretch", "pse", "vort")], ids="-".join)
def test_forward(gpu, outputs, presorted):
    d = particles(9000)
    print(f"[mixed-radii] {outputs} presorted={presorted}", flush=True)
    got = P.forward(*d, outputs=outputs, precision="f32c", sigma_mode="general",
                    presorted=presorted)
    ref = P.forward(*d, outputs=outputs, precision="f64", sigma_mode="general")
    for k in outputs:
        assert rel(got[k], ref[k]) <= TOL, k


@pytest.mark.parametrize("outputs", [("vel",), ("vel", "stretch"), ("vel", "stretch", "pse")],
                         ids="-".join)
def test_gradient(gpu, outputs):
    n = 6000
    x, a, s, nu = particles(n)
    x.requires_grad_()
    a.requires_grad_()
    g = torch.Generator(device="cuda").manual_seed(1)
    cot = [torch.randn((3, n), dtype=torch.float64, device="cuda", generator=g) for _ in outputs]
    print(f"[mixed-radii] gradient {outputs}", flush=True)
    grads = [torch.autograd.grad(AG.pair_sums(x, a, s, nu, outputs, p, "general"), (x, a), cot)
             for p in ("f32c", "f64")]
    for g32, g64 in zip(*grads):
        assert rel(g32, g64) <= TOL
