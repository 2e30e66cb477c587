"""Outputs in the place of the inputs: vpm_forward sums what the arrays held
before the call, in every precision and at every size, bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from openonda_amd import _lib as L
from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu


def particles(n, pad):
    x, a, s, _ = FM.random_cloud(n, seed=n)
    buf = torch.zeros((2, 3, n + pad), dtype=torch.float64, device="cuda")
    buf[0, :, :n], buf[1, :, :n] = P.to_soa(x), P.to_soa(a)
    return (buf[0][:, :n], buf[1][:, :n], torch.from_numpy(s).cuda(),
            torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))


@pytest.mark.parametrize("precision", ["f64", "f32c"])
@pytest.mark.parametrize("n,pad", [(5, 0), (700, 3), (4097, 0), (8192, 5), (30011, 0)])
@pytest.mark.parametrize("outputs,over", [(("vel",), {"vel": 0}), (("stretch",), {"stretch": 1}),
                                          (("vel", "stretch", "pse"), {"vel": 1, "stretch": 0}),
                                          (("stretch", "vort", "enstrophy"), {"vort": 1})],
                         ids=lambda v: "-".join(v))
def test_forward(gpu, outputs, over, n, pad, precision):
    print(f"[in-place] n={n} {outputs} {precision}", flush=True)
    want = P.forward(*particles(n, pad), outputs=outputs, precision=precision,
                     sigma_mode="uniform", out=None if pad == 0 else {
                         k: torch.empty((3, n + pad), dtype=torch.float64, device="cuda")[:, :n]
                         for k in outputs if k != "enstrophy"})
    d = particles(n, pad)
    out = {k: d[q] for k, q in over.items()}
    out.update({k: torch.empty((3, n + pad), dtype=torch.float64, device="cuda")[:, :n]
                for k in outputs if k != "enstrophy" and k not in over})
    got = P.forward(*d, outputs=outputs, precision=precision, sigma_mode="uniform", out=out)
    for k in outputs:
        assert torch.equal(got[k], want[k]), k


def test_partial_overlap_through_the_c_boundary(gpu):
    """The last component of the velocity over the first of the strengths."""
    n = 2001
    x, a, s, nu = particles(n, 0)
    want = P.forward(x, a, s, outputs=("vel",), precision="f64", sigma_mode="uniform")["vel"]
    buf = torch.zeros((8, n), dtype=torch.float64, device="cuda")
    buf[0:3], buf[5:8] = x, a
    p = L.Particles(n, n, buf[0].data_ptr(), buf[5].data_ptr(), s.data_ptr(), None)
    o = L.ForwardOpts(L.OUT_VEL, L.PREC_F64, L.SIGMA_UNIFORM, 0, -1)
    fo = L.ForwardOut(n, buf[3].data_ptr(), None, None, None, None)
    nb = L.load().vpm_forward_workspace_bytes(n, C.byref(o))
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    L.call("vpm_forward", C.byref(p), C.byref(o), C.byref(fo), ws.data_ptr(), nb, P._stream(x))
    assert torch.equal(buf[3:6], want)
