"""Workspace sizes of the forward passes: what a query returns covers what the
call writes.

Host part: the row pass writes the same records and chunk boxes for a uniform
radius as for per-particle radii, so both need the same workspace but for
whole source splits; the adjoint's query serves both precisions.  GPU part: every output set, the
adjoint, a batch and the library's autotuner in a workspace of exactly the
queried size, with guard bytes behind it.
"""
import ctypes as C

import numpy as np
import pytest

from openonda_amd import _lib as L

MASKS = [1, 2, 3, 4, 7, 8, 16, 24, 26, 27, 31]


def forward_bytes(n, mask, mode, presorted, tile=-1, precision=L.PREC_F32C):
    o = L.ForwardOpts(mask, precision, mode, presorted, tile)
    return L.load().vpm_forward_workspace_bytes(n, C.byref(o))


@pytest.mark.parametrize("presorted", [0, 1])
@pytest.mark.parametrize("mask", MASKS)
def test_row_pass_workspace_differs_between_radius_modes_by_splits_only(mask, presorted):
    # sorted sets above 65,536 ask the device for the radix sort's scratch
    slots = 3 * bin(mask).count("1") + (3 if mask & L.OUT_STRETCH else 0)
    for n in (8192, 8193, 9000, 16384, 20011, 34914, 65536) + ((100001, 131072) if presorted else ()):
        uniform = forward_bytes(n, mask, L.SIGMA_UNIFORM, presorted)
        general = forward_bytes(n, mask, L.SIGMA_GENERAL, presorted)
        assert uniform > 0
        if n <= 16384 or not mask & L.OUT_STRETCH:
            assert uniform == general, (n, mask)
        assert (general - uniform) % (slots * -(-n // 64) * 64 * 8) == 0, (n, mask)


def test_largest_allocation_free_set():
    """A set without source splits needs 104 bytes per particle, 8 more per 64 of
    them, and 25 KB: 2,577,764 particles in the caller's order fit the
    allocation-free call's 256 MiB."""
    assert L.load().vpm_forward_noalloc_capacity() == 256 << 20
    for mask, precision, tile in ((3, L.PREC_F64, -1), (31, L.PREC_F32C, 1)):
        at = lambda n: forward_bytes(n, mask, L.SIGMA_GENERAL, 1, tile, precision)
        assert at(2577764) <= 256 << 20 < at(2577765)


@pytest.mark.parametrize("n", [1, 5120, 5121, 9000, 20011, 65536])
def test_adjoint_workspace_serves_every_precision(n):
    """One query, with any options or none, covers every call on n particles
    in the caller's order."""
    lib = L.load()
    sizes = [lib.vpm_adjoint_workspace_bytes(n, None)]
    for precision in (L.PREC_F64, L.PREC_F32C):
        o = L.ForwardOpts(3, precision, L.SIGMA_UNIFORM, 0, -1)
        sizes.append(lib.vpm_adjoint_workspace_bytes(n, C.byref(o)))
    assert len(set(sizes)) == 1 and sizes[0] > 0


def test_sets_below_the_split_size_need_no_workspace():
    from openonda_amd import physics as P

    lib = L.load()
    for m in (1, 64, 1000, 1 << 20):
        for n in (0, 1, 255, P.SPLIT_MIN - 1):
            assert lib.vpm_pair_sum_workspace_bytes(m, n) == 0
            assert lib.vpm_induced_velocity_at_adjoint_workspace_bytes(n, m) == 0
    assert lib.vpm_pair_sum_workspace_bytes(64, P.SPLIT_MIN) > 0


GUARD = 1 << 16


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("mask", MASKS)
def test_forward_stays_inside_its_workspace(gpu, mask, general):
    import torch

    from openonda_amd import flow_models as FM
    from openonda_amd import physics as P

    rng = np.random.default_rng(mask)
    for n in (1, 700, 8191, 8192, 9000, 20011, 66001, 132000):
        x, a, s, _ = FM.random_cloud(n, seed=n)
        if general:
            s = s * rng.uniform(0.8, 1.25, n)
        d = (P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(),
             torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))
        p = P._particles(*d)
        mode = L.SIGMA_GENERAL if general else L.SIGMA_UNIFORM
        for precision in (L.PREC_F32C, L.PREC_F64):
            for presorted in (0, 1):
                print(f"[workspace] mask={mask} n={n} general={general} precision={precision} "
                      f"presorted={presorted}", flush=True)
                nb = forward_bytes(n, mask, mode, presorted, precision=precision)
                ws = torch.full((nb + GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
                o = L.ForwardOpts(mask, precision, mode, presorted, -1)
                out = torch.zeros((4, 3, n), dtype=torch.float64, device="cuda")
                ens = torch.zeros(1, dtype=torch.float64, device="cuda")
                fo = L.ForwardOut(n, *[out[q].data_ptr() for q in range(4)], ens.data_ptr())
                L.call("vpm_forward", C.byref(p), C.byref(o), C.byref(fo), ws.data_ptr(), nb,
                       P._stream(d[0]))
                assert bool((ws[nb:] == 0xA5).all()), (n, precision, presorted)


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("mask,n", [(1, 1000), (1, 4096), (3, 4096), (4, 5120), (7, 9001), (8, 1000),
                                    (31, 1000), (27, 20011)])
def test_autotune_accepts_the_workspace_it_asks_for(gpu, mask, n, general):
    import torch

    from openonda_amd import flow_models as FM
    from openonda_amd import physics as P

    x, a, s, _ = FM.random_cloud(n, seed=n)
    d = (P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(),
         torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))
    p = P._particles(*d)
    o = L.ForwardOpts(mask, L.PREC_F32C, L.SIGMA_GENERAL if general else L.SIGMA_UNIFORM, 0, -1)
    print(f"[workspace] autotune mask={mask} n={n} general={general}", flush=True)
    nb = L.load().vpm_autotune_workspace_bytes(n, C.byref(o))
    ws = torch.full((nb + GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
    out = torch.zeros((4, 3, n), dtype=torch.float64, device="cuda")
    ens = torch.zeros(1, dtype=torch.float64, device="cuda")
    fo = L.ForwardOut(n, *[out[q].data_ptr() for q in range(4)], ens.data_ptr())
    best = C.c_int(-1)
    L.call("vpm_autotune", C.byref(p), C.byref(o), C.byref(fo), ws.data_ptr(), nb,
           P._stream(d[0]), 1, C.byref(best), None)
    assert 0 <= best.value < L.load().vpm_tile_config_count()
    assert bool((ws[nb:] == 0xA5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n", [1, 700, 5120, 5121, 9000, 20011, 66001])
def test_adjoint_stays_inside_its_workspace(gpu, n, general):
    import torch

    from openonda_amd import flow_models as FM
    from openonda_amd import physics as P

    x, a, s, _ = FM.random_cloud(n, seed=n)
    d = (P.to_soa(x), P.to_soa(a), torch.from_numpy(s).cuda(),
         torch.full((n,), 1e-3, dtype=torch.float64, device="cuda"))
    p = P._particles(*d)
    cot = torch.ones((3, 3, n), dtype=torch.float64, device="cuda")
    out = torch.zeros((2, 3, n), dtype=torch.float64, device="cuda")
    for precision in (L.PREC_F32C, L.PREC_F64):
        for presorted in (0, 1):
            print(f"[workspace] adjoint n={n} general={general} precision={precision} "
                  f"presorted={presorted}", flush=True)
            o = L.ForwardOpts(3, precision, L.SIGMA_GENERAL if general else L.SIGMA_UNIFORM,
                              presorted, -1)
            nb = L.load().vpm_adjoint_workspace_bytes(n, C.byref(o))
            ws = torch.full((nb + GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
            ci = L.AdjointIn(n, *[cot[q].data_ptr() for q in range(3)])
            co = L.AdjointOut(n, out[0].data_ptr(), out[1].data_ptr())
            L.call("vpm_adjoint", C.byref(p), C.byref(ci), C.byref(o), C.byref(co),
                   ws.data_ptr(), nb, P._stream(d[0]))
            assert bool((ws[nb:] == 0xA5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1], [64, 0, 65, 3], [50] * 40, [9000, 128, 5001], [20011]],
                         ids=str)
def test_batch_stays_inside_its_workspace(gpu, sizes):
    import torch

    from openonda_amd import batch as B
    from openonda_amd import flow_models as FM

    sets = []
    for i, n in enumerate(sizes):
        x, a, s, _ = FM.random_cloud(max(n, 1), seed=i)
        sets.append((x[:n], a[:n], s[:n], np.full(n, 1e-3)))
    for rows in (True, False):
        for les in (True, False):
            print(f"[workspace] batch {sizes[:4]} rows={rows} les={les}", flush=True)
            bs = B.BatchedSystem(sets, dt=0.01, les=les)
            bs.set_launch(bs.tile_config, rows=rows)
            nb = L.load().vpm_batch_workspace_bytes(bs.n, bs.nsets, bs.desc.n_items)
            bs.ws = torch.full((nb + GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
            bs.wsb = nb
            torch.cuda.synchronize()
            bs.evaluate(bs.x, bs.a, bs.stage_mask, True, bs.stream.cuda_stream)
            bs.synchronize()
            assert bool((bs.ws[nb:] == 0xA5).all())
