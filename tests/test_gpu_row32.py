"""The FP32-compensated row pass: edges of rows, chunks, waves and splits, against the FP64 pass.

Bar: rel-L2 <= 1e-6 on every output (the pass's documented accuracy).
"""
import ctypes as C

import numpy as np
import pytest
import torch

from openonda_amd import _lib as L
from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

TOL = 1e-6
UNIFORM = [("stretch", "vort", "enstrophy"), ("vel",), ("stretch",), ("pse",), ("vort",), ("enstrophy",), ("vort", "enstrophy"),
           ("vel", "stretch"), ("vel", "stretch", "pse"), ("vel", "stretch", "vort", "enstrophy"),
           ("vel", "stretch", "pse", "vort", "enstrophy")]
GENERAL = UNIFORM


def particles(layout, n, general):
    rng = np.random.default_rng(n)
    if layout == "ring":
        x, a, s, _ = FM.torus_ring(-(-n // 64))
        x, a, s = x[:n], a[:n], s[:n]
    else:
        x, a, s, _ = FM.random_cloud(n, seed=n)
    if general:
        s = s * rng.uniform(0.7, 1.4, n)
    return (P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(),
            torch.from_numpy(rng.uniform(1e-4, 1e-3, n)).cuda())


@pytest.mark.parametrize("layout", ["cloud", "ring"])
@pytest.mark.parametrize("outputs,general", [(o, False) for o in UNIFORM]
                         + [(o, True) for o in GENERAL],
                         ids=lambda v: "-".join(v) if isinstance(v, tuple) else str(v))
def test_sets_at_row_and_split_edges(gpu, layout, outputs, general):
    """Whole and ragged rows and chunks, one split and several, the caller's
    order and the sorted one, a stride above n."""
    mode = "general" if general else "uniform"
    for n in (8192, 8255, 12345):
        d = particles(layout, n, general)
        ref = P.forward(*d, outputs=outputs, precision="f64", sigma_mode=mode)
        wide = [torch.empty((3, n + 3), dtype=torch.float64, device="cuda")[:, :n].copy_(t)
                for t in d[:2]] + list(d[2:])
        for kw in ({}, {"max_splits": 1}, {"presorted": True}, {"d": wide}):
            kw = dict(kw)
            got = P.forward(*kw.pop("d", d), outputs=outputs, precision="f32c", sigma_mode=mode,
                            **kw)
            for k in outputs:
                g, r = got[k].cpu().numpy(), ref[k].cpu().numpy()
                e = np.linalg.norm(g - r) / np.linalg.norm(r)
                assert e <= TOL, (layout, n, kw, k, e)


def test_same_bits_every_time(gpu):
    d = particles("ring", 20011, True)
    one = P.forward(*d, outputs=("stretch",), precision="f32c", sigma_mode="general")["stretch"]
    two = P.forward(*d, outputs=("stretch",), precision="f32c", sigma_mode="general")["stretch"]
    assert torch.equal(one, two)


def test_noalloc_without_room_for_the_records(gpu):
    """1.7 million particles with their own radii fit the static array, their
    records do not: the tiled kernels run, as they always did there."""
    n = 1_700_000
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((3, n), dtype=torch.float64, device="cuda", generator=g)
    a = torch.randn((3, n), dtype=torch.float64, device="cuda", generator=g) / n
    s = 0.01 + 0.005 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    opts = L.ForwardOpts(L.OUT_VEL, L.PREC_F32C, L.SIGMA_GENERAL, 0, -1)
    assert (L.load().vpm_forward_workspace_bytes(n, C.byref(opts))
            > L.load().vpm_forward_noalloc_capacity())
    out = torch.empty_like(x)
    fo = L.ForwardOut(n, out.data_ptr(), None, None, None, None)
    p = P._particles(x, a, s)
    print(f"[row32] noalloc n={n}", flush=True)
    L.call("vpm_forward_noalloc", C.byref(p), C.byref(opts), C.byref(fo), P._stream(x))
    i = torch.arange(0, n, n // 64, device="cuda")[:64]
    d = x[:, i, None] - x[:, None, :]
    sg = 0.5 * (s[i][:, None] + s[None, :])
    r2 = (d * d).sum(0) / (sg * sg)
    q = (r2 + 2.5) / ((r2 + 1.0) ** 2.5 * sg ** 3)
    b = a[:, None, :]
    ref = -torch.stack([(q * (d[1] * b[2] - d[2] * b[1])).sum(1),
                        (q * (d[2] * b[0] - d[0] * b[2])).sum(1),
                        (q * (d[0] * b[1] - d[1] * b[0])).sum(1)]) / (4.0 * np.pi)
    assert float((out[:, i] - ref).norm() / ref.norm()) <= TOL
