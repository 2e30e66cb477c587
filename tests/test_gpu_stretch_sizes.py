"""Output sets on both sides of the size where the tiled kernels take over from
the row pass (the stretching alone with a uniform radius: 131,072 particles;
PSE with vorticity and per-particle radii: 262,144), and row sets split to fit
the L2, against the FP64 pass.  Bar: rel-L2 <= 1e-6."""
import numpy as np
import pytest
import torch

from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["cloud", "ring"])
@pytest.mark.parametrize("n", [131072, 131073, 164000])
def test_stretching(gpu, layout, n):
    x, a, s, _ = FM.torus_ring(-(-n // 64)) if layout == "ring" else FM.random_cloud(n, seed=n)
    d = P.to_soa(x[:n]), P.to_soa(a[:n]), torch.from_numpy(s[:n].copy()).cuda()
    print(f"[stretch-sizes] {layout} n={n}", flush=True)
    ref = P.forward(*d, outputs=("stretch",), precision="f64", sigma_mode="uniform")["stretch"]
    for kw in ({}, {"presorted": True}) if layout == "ring" else ({},):  # a ring comes in order
        got = P.forward(*d, outputs=("stretch",), precision="f32c", sigma_mode="uniform", **kw)
        assert float((got["stretch"] - ref).norm() / ref.norm()) <= 1e-6, kw


ALL = ("vel", "stretch", "pse", "vort", "enstrophy")


@pytest.mark.parametrize("n,outputs", [(262144, ALL), (262145, ALL), (16385, ("stretch",)),
                                       (65601, ("vel", "stretch", "pse")), (65601, ALL),
                                       (131073, ("stretch", "vort", "enstrophy"))],
                         ids=lambda v: "-".join(v) if isinstance(v, tuple) else str(v))
def test_sets_with_their_own_radii(gpu, n, outputs):
    x, a, s, _ = FM.torus_ring(-(-n // 64))
    s = s[:n] * np.random.default_rng(n).uniform(0.8, 1.25, n)
    d = (P.to_soa(x[:n]), P.to_soa(a[:n]), torch.from_numpy(s).cuda(),
         torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))
    print(f"[stretch-sizes] {outputs} n={n}", flush=True)
    got = P.forward(*d, outputs=outputs, precision="f32c", sigma_mode="general")
    ref = P.forward(*d, outputs=outputs, precision="f64", sigma_mode="general")
    for k in outputs:
        assert float((got[k] - ref[k]).norm() / ref[k].norm()) <= 1e-6, k
