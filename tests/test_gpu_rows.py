"""The FP64 row sums at the edges of their rows, source groups and splits.

Rows are 64 targets, a wave sums whole groups of four sources, and small sets
split their sources among workgroups when the caller gives a workspace.  Bars
are the plain kernels' (a few ulp of the sum): rel-L2 <= 1e-12 for vectors,
1e-11 relative for scalars, against the NumPy oracle.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from openonda_amd import _lib as L
from openonda_amd import physics as P
from openonda_amd import autograd as AG
from openonda_amd import flow_models as FM
from oracle import vpm_oracle as O
from oracle import vpm_torch as T

pytestmark = pytest.mark.gpu

VEC_TOL, SCAL_TOL = 1e-12, 1e-11


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


def particles(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1, (n, 3)) / max(n, 1),
            rng.uniform(0.1, 0.3, n), rng.uniform(1e-4, 1e-2, n))


def strided(a, pad):
    """(N,3) array -> (3,N) device view with component stride N + pad."""
    n = len(a)
    buf = torch.full((3, n + pad), float("nan"), dtype=torch.float64, device="cuda")
    buf[:, :n] = torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    return buf[:, :n]


def dev(x, a, s, nu, pad):
    return (strided(x, pad), strided(a, pad), torch.from_numpy(s).cuda(),
            torch.from_numpy(nu).cuda())


@pytest.mark.parametrize("variant", ["cuda", "cpu"])
@pytest.mark.parametrize("n,pad", [(1, 0), (3, 2), (63, 1), (64, 0), (65, 7), (129, 0), (511, 3),
                                   (1031, 1), (2999, 0)])
def test_self_sums_at_row_edges(gpu, variant, n, pad):
    print(f"[rows] n={n} pad={pad} {variant}", flush=True)
    x, a, s, nu = particles(n, n)
    dx, da, ds, dn = dev(x, a, s, nu, pad)
    for got, ref in [
        (P.selfinduced_velocity(dx, da, ds, variant), O.selfinduced_velocity(x, a, s, variant)),
        (P.strength_gradients(dx, da, ds), O.strength_gradients(x, a, s)),
        (P.strength_gradients_pse(dx, da, ds, dn, variant),
         O.strength_gradients_pse(x, a, s, nu, variant)),
        (P.vorticity_field_at(dx, dx, da, ds, variant), O.vorticity_field_at(x, x, a, s, variant)),
    ]:
        assert rel(P.from_soa(got), ref) <= VEC_TOL
    for got, ref in [
        (P.total_kinetic_energy(dx, da, ds, variant), O.total_kinetic_energy(x, a, s, variant)),
        (P.total_helicity(dx, da, ds, variant), O.total_helicity(x, a, s, variant)),
        (P.total_enstrophy(dx, da, ds, variant), O.total_enstrophy(x, a, s, variant)),
    ]:
        assert abs(got.item() - ref) <= SCAL_TOL * max(abs(ref), 1e-12)


@pytest.mark.parametrize("m,n", [(1, 1000), (65, 3), (64, 0), (700, 5001), (4100, 130)])
def test_sums_at_targets(gpu, m, n):
    print(f"[rows] m={m} n={n}", flush=True)
    x, a, s, nu = particles(n, n + 1)
    y = np.random.default_rng(m).uniform(-1.2, 1.2, (m, 3))
    dx, da, ds, _ = dev(x, a, s, nu, 0)
    dy = strided(y, 5)
    u, w = P.induced_velocity_at(dy, dx, da, ds), P.vorticity_field_at(dy, dx, da, ds)
    if n == 0:
        assert not u.any() and not w.any()
        return
    assert rel(P.from_soa(u), O.induced_velocity_at(y, x, a, s)) <= VEC_TOL
    assert rel(P.from_soa(w), O.vorticity_field_at(y, x, a, s)) <= VEC_TOL


@pytest.mark.parametrize("n", [200, 1031, 5000])
def test_splits_agree_with_the_unsplit_sum(gpu, n):
    """The entry points without a workspace sum the same pairs in one split."""
    x, a, s, nu = particles(n, n)
    dx, da, ds, dn = dev(x, a, s, nu, 0)
    p = P._particles(dx, da, ds, dn)
    st = P._stream(dx)
    out = torch.empty_like(dx)
    L.call("vpm_get_selfinduced_velocity", C.byref(p), 0, out.data_ptr(), n, st)
    assert rel(P.from_soa(P.selfinduced_velocity(dx, da, ds)), P.from_soa(out)) <= 1e-14
    L.call("vpm_get_strength_gradients", C.byref(p), out.data_ptr(), n, st)
    assert rel(P.from_soa(P.strength_gradients(dx, da, ds)), P.from_soa(out)) <= 1e-13
    L.call("vpm_get_strength_gradients_pse", C.byref(p), 0, out.data_ptr(), n, st)
    assert rel(P.from_soa(P.strength_gradients_pse(dx, da, ds, dn)), P.from_soa(out)) <= 1e-13


@pytest.mark.parametrize("m,n", [(1, 1), (3, 65), (5, 64), (700, 63), (130, 2999)])
def test_probe_adjoint_at_row_edges(gpu, m, n):
    """Gradient of the velocity at m points with respect to n particles, one
    point on a particle (masked), against torch autograd of the oracle."""
    print(f"[rows-adjoint] m={m} n={n}", flush=True)
    x, a, s, _ = particles(n, n + 2)
    y = np.random.default_rng(m).uniform(-1.2, 1.2, (m, 3))
    if m > 1:
        y[1] = x[n // 2]
    lam = np.random.default_rng(m + 1).normal(size=(m, 3))
    leaf = [torch.from_numpy(t).cuda().requires_grad_() for t in (x, a)]
    ref = torch.autograd.grad(
        (T.induced_velocity_at(torch.from_numpy(y).cuda(), *leaf, torch.from_numpy(s).cuda())
         * torch.from_numpy(lam).cuda()).sum(), leaf)
    dx, da, ds, _ = dev(x, a, s, s, 3)
    dx.requires_grad_()
    da.requires_grad_()
    got = torch.autograd.grad(AG.probe_velocity(strided(y, 2), dx, da, ds), (dx, da),
                              strided(lam, 0))
    for g, r in zip(got, ref):
        assert rel(P.from_soa(g), r.cpu().numpy()) <= VEC_TOL


def test_stretching_along_a_tube(gpu):
    """Nearly parallel strengths: alpha_i x sum g alpha_j is a small difference."""
    rng = np.random.default_rng(4)
    n = 1500
    x = np.stack([0.05 * rng.standard_normal(n), 0.05 * rng.standard_normal(n),
                  np.linspace(-1, 1, n)], 1)
    a = np.stack([1e-5 * rng.standard_normal(n), 1e-5 * rng.standard_normal(n),
                  1.0 + 0.01 * rng.standard_normal(n)], 1)
    s = np.full(n, 0.05)
    dx, da, ds, _ = dev(x, a, s, s, 0)
    assert rel(P.from_soa(P.strength_gradients(dx, da, ds)), O.strength_gradients(x, a, s)) <= 1e-12


def test_non_finite_inputs_carry_on_as_in_the_reference(gpu):
    """A particle at infinity drops out of PSE and vorticity (weight 1/inf) and
    turns velocity and stretching NaN (inf/inf); NaN strengths spread to the
    others' sums but not to the particle's own; two particles at one point
    make the energy NaN."""
    n = 300
    x, a, s, nu = particles(n, 9)
    far = x.copy()
    far[37] = np.inf
    dx, da, ds, dn = dev(far, a, s, nu, 0)
    others = np.delete(np.arange(n), 37)
    keep = [t[others] for t in (x, a, s, nu)]
    got = P.from_soa(P.strength_gradients_pse(dx, da, ds, dn))[others]
    assert rel(got, O.strength_gradients_pse(*keep)) <= VEC_TOL
    got = P.from_soa(P.vorticity_field_at(strided(keep[0], 0), dx, da, ds))
    assert rel(got, O.vorticity_field_at(keep[0], *keep[:3])) <= VEC_TOL
    assert np.isnan(P.from_soa(P.selfinduced_velocity(dx, da, ds))).all()
    assert np.isnan(P.from_soa(P.strength_gradients(dx, da, ds))).all()

    bad = a.copy()
    bad[5] = np.nan
    dx, da, ds, dn = dev(x, bad, s, nu, 0)
    u = P.from_soa(P.selfinduced_velocity(dx, da, ds))
    assert np.isfinite(u[5]).all() and np.isnan(np.delete(u, 5, 0)).all()

    twin = x.copy()
    twin[7] = twin[250]
    dx, da, ds, dn = dev(twin, a, s, nu, 0)
    assert np.isnan(P.total_kinetic_energy(dx, da, ds).item())
    assert np.isfinite(P.total_enstrophy(dx, da, ds).item())
    assert np.isfinite(P.from_soa(P.selfinduced_velocity(dx, da, ds))).all()


OUTS = [("stretch", "vort", "enstrophy"), ("vel",), ("stretch",), ("vel", "stretch"), ("pse",), ("vort",), ("enstrophy",),
        ("vel", "stretch", "pse"), ("vort", "enstrophy"), ("vel", "stretch", "vort", "enstrophy"),
        ("vel", "pse"), ("vel", "stretch", "pse", "vort", "enstrophy")]


def plain_outputs(d, outputs):
    x, a, s, nu = d
    ref = {"vel": lambda: P.selfinduced_velocity(x, a, s),
           "stretch": lambda: P.strength_gradients(x, a, s),
           "pse": lambda: P.strength_gradients_pse(x, a, s, nu),
           "vort": lambda: P.vorticity_field_at(x, x, a, s),
           "enstrophy": lambda: P.total_enstrophy(x, a, s)}
    return {k: ref[k]() for k in outputs}


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("outputs", OUTS, ids="-".join)
@pytest.mark.parametrize("n", [1, 65, 1031, 8191])
def test_fused_rows(gpu, n, outputs, uniform):
    """The FP64 pass, and the FP32-compensated one up to 8191 particles, are
    the FP64 rows: the plain kernels' values (pinned to the oracle above) to
    1e-12 for every output set, radius mode, split count and input stride."""
    print(f"[rows-forward] n={n} {outputs} uniform={uniform}", flush=True)
    x, a, s, nu = particles(n, n + 3)
    if uniform:
        s[:] = 0.17
    d = dev(x, a, s, nu, 5)
    ref = plain_outputs(d, outputs)
    mode = "uniform" if uniform else "general"
    for kw in ({"precision": "f64"}, {"precision": "f32c"}, {"precision": "f64", "max_splits": 1}):
        got = P.forward(*d, outputs=outputs, sigma_mode=mode, **kw)
        for k in outputs:
            r, g = ref[k].cpu().numpy(), got[k].cpu().numpy()
            assert rel(g, r) <= (SCAL_TOL if k == "enstrophy" else VEC_TOL), (k, kw)


def test_first_size_past_the_rows(gpu):
    """One particle more and the FP32-compensated kernels run: 1e-6, not 1e-12;
    a tile shape asked for by index runs them at any size."""
    for n, kw in ((8192, {}), (8191, {"tile_config": 5})):
        x, a, s, nu = particles(n, n)
        s[:] = 0.17
        d = dev(x, a, s, nu, 0)
        ref = plain_outputs(d, ("vel", "stretch"))
        got = P.forward(*d, outputs=("vel", "stretch"), sigma_mode="uniform", **kw)
        for k in ref:
            e = rel(got[k].cpu().numpy(), ref[k].cpu().numpy())
            assert 1e-10 < e <= 1e-6, (n, k, e)


@pytest.mark.parametrize("layout", ["ring", "cloud"])
@pytest.mark.parametrize("outputs", [("vel", "stretch"), ("vel", "stretch", "pse"),
                                     ("vel", "stretch", "pse", "vort", "enstrophy")])
def test_fp32_kernels_at_small_sizes(gpu, layout, outputs):
    """The FP32-compensated kernels (asked for by tile shape) over near and far
    tiles in one pass and in splits, against the rows; the empty-split and
    ragged edges at sizes the default leaves to the rows."""
    for n in (37, 700, 4096):
        x, a, s, nu = (FM.torus_ring(-(-n // 64), nu=1e-3) if layout == "ring"
                       else FM.random_cloud(n, seed=41))
        x, a, s, nu = x[:n], a[:n], s[:n], np.full(n, 1e-3)
        d = dev(x, a, s, nu, 0)
        ref = P.forward(*d, outputs=outputs, precision="f64", sigma_mode="uniform")
        for splits in (0, 1, 3):
            got = P.forward(*d, outputs=outputs, sigma_mode="uniform", max_splits=splits,
                            tile_config=P.tile_config_default(outputs))
            for k in outputs:
                e = rel(got[k].cpu().numpy(), ref[k].cpu().numpy())
                assert e <= 1e-6, (layout, n, splits, k, e)
