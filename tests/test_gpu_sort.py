"""The Morton sort of a pass, at the edges of its 1024-key blocks, with many
equal keys and on both sides of the size above which the radix sort runs:
the pass gives the same bits as over particles that the caller has put in
stable key order.
"""
import numpy as np
import pytest
import torch

from openonda_amd import physics as P

pytestmark = pytest.mark.gpu


def spread(v):
    out = np.zeros_like(v)
    for b in range(10):
        out |= ((v >> b) & 1) << (3 * b)
    return out


def stable_order(x):
    """Stable order of the 30-bit Morton keys on a grid of 1024 per axis."""
    lo, hi = x.min(0), x.max(0)
    ext = np.where(hi > lo, hi - lo, 1.0)
    q = np.clip(((x - lo) / ext * 1023.0).astype(np.int64), 0, 1023)
    key = spread(q[:, 0]) | (spread(q[:, 1]) << 1) | (spread(q[:, 2]) << 2)
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("kind", ["cloud", "cluster", "line"])
@pytest.mark.parametrize("n", [8192, 8193, 9216 + 31, 9216 + 32, 10239, 20011, 65536, 65537])
def test_same_bits_as_in_key_order(gpu, n, kind):
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (n, 3))
    if kind == "cluster":   # some hundred keys in all
        x *= 1e-2
        x[n // 2] = (3.0, 3.0, 3.0)
    elif kind == "line":    # keys already descending; no extent in z
        x = np.stack([np.linspace(1, -1, n), np.linspace(1, -1, n), np.zeros(n)], 1)
    a = rng.normal(0, 1, (n, 3)) / n
    s = rng.uniform(0.01, 0.02, n)
    order = stable_order(x)
    outs = ("vel", "stretch")
    d = (P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda())
    e = (P.to_soa(x[order]), P.to_soa(a[order]), torch.from_numpy(s[order]).cuda())
    got = P.forward(*d, outputs=outs, sigma_mode="general")
    ref = P.forward(*e, outputs=outs, sigma_mode="general", presorted=True)
    pick = torch.from_numpy(order).cuda()
    for k in outs:
        assert torch.equal(got[k][:, pick], ref[k]), k
