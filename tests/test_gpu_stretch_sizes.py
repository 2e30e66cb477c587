"""The stretching alone with a uniform radius on both sides of the size where
the tiled kernels take over from the row pass (131,072), against the FP64 pass.
Bar: rel-L2 <= 1e-6."""
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
