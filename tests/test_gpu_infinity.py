"""A particle at infinity leaves PSE and vorticity sums, whose weights vanish
there, in every pass (its distance makes velocity, stretching and energy
inf/inf, as in the reference).

The FP32 passes are held to their 1e-6.  The sort sees an infinite box and
keeps the caller's order, so offsets are as large as the cloud: radii of half
its size bound a weight's error by 4.5 (2 |x| 2^-24 / sigma) + 9 roundings of
the root and its powers, 1.3e-6 for the worst pair and a third of it in L2.
"""
import numpy as np
import pytest
import torch

from openonda_amd import autograd as AG
from openonda_amd import batch as B
from openonda_amd import physics as P
from oracle import vpm_oracle as O

pytestmark = pytest.mark.gpu

ALL = ("vel", "stretch", "pse", "vort", "enstrophy")
TOL = {"f32c": 1e-6, "f64": 1e-12}


def rel(g, r):
    return np.linalg.norm(g - r) / np.linalg.norm(r)


def particles(n, general):
    rng = np.random.default_rng(n)
    x, a = rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1, (n, 3)) / n
    s = rng.uniform(0.9, 1.1, n) if general else np.full(n, 1.0)
    return x, a, s, rng.uniform(1e-4, 1e-3, n)


def dev(x, a, s, nu):
    return P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(), torch.from_numpy(nu).cuda()


@pytest.fixture(scope="module")
def reference():
    kept = {}

    def get(n, general):
        if (n, general) not in kept:
            d = particles(n, general)
            i = np.delete(np.arange(n), n // 2)
            k = [t[i] for t in d]
            sample = np.arange(0, n - 1, 37)
            # a sample of targets: the particles' own pair adds nothing to either sum
            r2 = ((k[0][sample, None] - k[0][None]) ** 2).sum(-1)
            sg = 0.5 * (k[2][sample, None] + k[2][None])
            w = 105.0 * k[3][sample, None] / (4 * np.pi) / sg ** 2 / (r2 / sg ** 2 + 1) ** 4.5
            pse = np.einsum("ij,ijc->ic", w, k[1][None] - k[1][sample, None])
            vort = O.vorticity_field_at(k[0][sample], *k[:3])
            kept[n, general] = i, sample, {"pse": pse, "vort": vort}
        return kept[n, general]
    return get


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("outputs", [("pse",), ("vort",), ("vort", "enstrophy"),
                                     ("vel", "stretch", "pse"),
                                     ("stretch", "vort", "enstrophy"),
                                     ("vel", "stretch", "vort", "enstrophy"), ALL], ids="-".join)
@pytest.mark.parametrize("n,precision", [(300, "f32c"), (9000, "f32c"), (1500, "f64")])
def test_forward(gpu, reference, outputs, general, n, precision):
    i, sample, ref = reference(n, general)
    x, a, s, nu = particles(n, general)
    x[n // 2] = np.inf
    d = dev(x, a, s, nu)
    print(f"[infinity] n={n} {outputs} general={general} {precision}", flush=True)
    got = P.forward(*d, outputs=outputs, precision=precision,
                    sigma_mode="general" if general else "uniform")
    for k in set(outputs) & {"pse", "vort"}:
        assert rel(P.from_soa(got[k])[i][sample], ref[k]) <= TOL[precision], k


@pytest.mark.parametrize("general", [False, True])
def test_gradient_of_the_diffusion(gpu, general):
    n = 6000
    x, a, s, nu = particles(n, general)
    xi = np.random.default_rng(1).normal(size=(n, 3))
    i = np.delete(np.arange(n), n // 2)

    def dalpha(x, a, s, nu, xi, precision):
        dx, da, ds, dn = dev(x, a, s, nu)
        dx.requires_grad_()
        da.requires_grad_()
        out = AG.pair_sums(dx, da, ds, dn, ("pse",), precision, "general" if general else "uniform")
        return P.from_soa(torch.autograd.grad(out, (dx, da), [P.to_soa(xi)])[1])

    ref = dalpha(x[i], a[i], s[i], nu[i], xi[i], "f64")
    x[n // 2] = np.inf
    print(f"[infinity] gradient general={general}", flush=True)
    assert rel(dalpha(x, a, s, nu, xi, "f32c")[i], ref) <= TOL["f32c"]


def test_batch(gpu, reference):
    n = 9000
    i, sample, ref = reference(n, False)
    x, a, s, nu = particles(n, False)
    x[n // 2] = np.inf
    print("[infinity] batch", flush=True)
    bs = B.BatchedSystem([(x, a, s, nu)], dt=0.01, pse=True, les=True)
    bs.evaluate(bs.x, bs.a, bs.stage_mask, True, bs.stream.cuda_stream)
    bs.synchronize()
    for k, v in (("pse", bs.pse_), ("vort", bs.vort)):
        assert rel(P.from_soa(v[:, :n])[i][sample], ref[k]) <= TOL["f32c"], k
