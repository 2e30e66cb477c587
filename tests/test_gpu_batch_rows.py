"""The batched row pass: uneven sets at the edges of rows, items and splits,
against the FP64 pass of each set on its own, and its replay in a graph.

Bar: rel-L2 <= 1e-6 per set and output (enstrophy: relative 1e-6).
"""
import numpy as np
import pytest
import torch

from openonda_amd import _lib as L
from openonda_amd import batch as B
from openonda_amd import flow_models as FM
from openonda_amd import physics as P

pytestmark = pytest.mark.gpu

TOL = 1e-6
SMALL = [1, 63, 64, 65, 129, 700, 3000]
MANY = [9000, 2, 64 * 37, 5001, 12345]


def sets_of(sizes):
    out = []
    for i, n in enumerate(sizes):
        x, a, s, _ = FM.torus_ring(-(-n // 64)) if i % 2 else FM.random_cloud(n, seed=100 + i)
        out.append((x[:n], a[:n], s[:n], np.full(n, 1e-3 * (1 + i))))
    return out


@pytest.mark.parametrize("sizes", [SMALL, MANY, MANY * 5], ids=["small", "many", "unsplit"])
@pytest.mark.parametrize("pse,les", [(True, True), (True, False), (False, True), (False, False)])
def test_each_set_matches_its_own_pass(gpu, sizes, pse, les):
    sets = sets_of(sizes)
    bs = B.BatchedSystem(sets, dt=0.01, precision="f32c", pse=pse, les=les)
    assert bs.rows
    names = ["vel", "stretch"] + (["pse"] if pse else []) + (["vort", "enstrophy"] if les else [])
    print(f"[batch-rows] {names} sets={len(sizes)}", flush=True)
    for resort in (True, False):
        bs.evaluate(bs.x, bs.a, bs.stage_mask, resort, bs.stream.cuda_stream)
        bs.synchronize()
        for k, (x, a, s, nu) in enumerate(sets):
            sl = bs.set_slice(k)
            d = (P.to_soa(x), P.to_soa(a), torch.from_numpy(s.copy()).cuda(),
                 torch.from_numpy(nu).cuda())
            ref = P.forward(*d, outputs=names, precision="f64", sigma_mode="uniform")
            got = {"vel": bs.vel[:, sl], "stretch": bs.str_[:, sl], "pse": bs.pse_[:, sl],
                   "vort": bs.vort[:, sl], "enstrophy": bs.enstrophy[k]}
            for q in names:
                assert float((got[q] - ref[q]).norm()) <= TOL * float(ref[q].norm()), (k, q)


def test_replayed_steps_equal_eager_ones(gpu):
    """Six replays, with eager work and synchronisation between them."""
    one = B.BatchedSystem(sets_of(MANY), dt=0.01, pse=True, les=True)
    two = B.BatchedSystem(sets_of(MANY), dt=0.01, pse=True, les=True)
    one.step()
    two.step()
    two.capture()
    for k in range(6):
        one.step()
        two.replay(1)
        two.synchronize()
        torch.cuda.synchronize()
        assert torch.equal(one.x, two.x) and torch.equal(one.a, two.a), k
        assert torch.equal(one.nu_t, two.nu_t), k


def test_bad_item_sizes_are_refused(gpu):
    bs = B.BatchedSystem(sets_of([200]), dt=0.01)
    p = bs._parts(bs.x, bs.a)
    o = L.ForwardOpts(3, L.PREC_F32C, L.SIGMA_UNIFORM, 0, -1)
    fo = L.ForwardOut(bs.n, bs.vel.data_ptr(), bs.str_.data_ptr(), None, None, None)
    for t in (0, 32, 100, 1024):
        with pytest.raises(L.VpmError) as e:
            L.call("vpm_batch_run_rows", p, bs.desc, t, o, fo, bs.ws.data_ptr(), bs.wsb, 0)
        assert e.value.code == L.VPM_ERR_ARG
