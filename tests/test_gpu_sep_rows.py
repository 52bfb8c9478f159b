"""The separable 2-D kernels on few coil rows and on one trajectory per batch item, at the
edges of their work split, against the oracle.

Tolerance: both sides sum products of float32 values (36 taps a sample, some hundred
entries a cell) whose rounding errors add up like a random walk, a few eps = 6e-8 times
sqrt(100): 2e-6 in the 2-norm."""
import numpy as np
import pytest
import torch

import inputs as gi
import torchkbnufft_amd as tkbn
from conftest import create_ktraj, rel_l2
from oracle import table_path as tp
from torchkbnufft_amd import _lib
from torchkbnufft_amd._nufft import interp as _interp

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
TOL = 2e-6


def _kernel():
    return _lib.load().tkbn_last_interp_kernel().decode()


def _both(im, grid, J, x, y, om, tabs=None):
    """GPU gather of x and spread of y, and the oracle's."""
    ob = tkbn.KbInterp(im_size=im, grid_size=grid, numpoints=J, dtype=torch.complex64).to(DEV)
    plan = tp.Plan(im, grid, numpoints=J, dtype=torch.complex64)
    tabs = plan.tables if tabs is None else tabs
    args = (ob.n_shift, ob.numpoints, ob.table_oversamp, ob.offsets)
    dt, od = [t.to(DEV) for t in tabs], om.to(DEV)
    kd = _interp.table_interp(x.to(DEV), od, dt, *args, binned=True)
    assert _kernel() == "gather_sep_kernel"
    gr = _interp.table_interp_adjoint(y.to(DEV), od, dt, *args, grid, deterministic=False)
    assert _kernel() == "spread_sep_kernel"
    ns, Jt, L, off = plan.t_n_shift, plan.t_numpoints, plan.t_table_oversamp, plan.offsets
    ref_f = tp.table_interp(x, om, tabs, ns, Jt, L, off)
    ref_a = tp.table_interp_adjoint(y, om, tabs, ns, Jt, L, off, plan.t_grid_size)
    return kd.cpu(), ref_f, gr.cpu(), ref_a


def _traj(M, gen, dense):
    om = create_ktraj(2, M, gen, torch.float32)
    if dense:  # a hot centre: tiles cut into pieces
        om[:, : M // 2] *= 0.04
    return om


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 33])
@pytest.mark.parametrize("im,grid,J,M", [((32, 30), (64, 60), 6, 4000), ((11, 40), (21, 83), (5, 4), 900)])
def test_row_counts_match_oracle(rows, im, grid, J, M):
    print(f"[case] sep rows={rows} grid={grid} J={J}", flush=True)
    gen = torch.Generator().manual_seed(rows)
    om = _traj(M, gen, True)
    kd, rf, gr, ra = _both(im, grid, J, gi.cplx((1, rows) + grid, gen), gi.cplx((1, rows, M), gen), om)
    assert rel_l2(kd, rf) < TOL and rel_l2(gr, ra) < TOL


@pytest.mark.parametrize("B,C,grid,M", [(3, 1, (40, 36), 700), (4, 8, (64, 64), 2500), (2, 20, (48, 50), 1500),
                                        (40, 2, (200, 184), 300)])
def test_trajectory_per_batch_item_matches_oracle(B, C, grid, M):
    print(f"[case] sep frames B={B} C={C} grid={grid}", flush=True)
    gen = torch.Generator().manual_seed(B)
    im = tuple(g // 2 for g in grid)
    om = torch.stack([_traj(M, gen, b % 2 == 0) for b in range(B)])
    kd, rf, gr, ra = _both(im, grid, 6, gi.cplx((B, C) + grid, gen), gi.cplx((B, C, M), gen), om)
    assert rel_l2(kd, rf) < TOL and rel_l2(gr, ra) < TOL


@pytest.mark.parametrize("rows", [1, 4, 8, 12])
def test_tables_of_another_form(rows):
    """Every entry left out of the products (complex weights, more than a wave remembers)."""
    print(f"[case] sep perturbed tables rows={rows}", flush=True)
    gen = torch.Generator().manual_seed(7)
    grid, M = (64, 60), 3000
    tabs = []
    for t in tp.Plan((32, 30), grid, dtype=torch.complex64).tables:
        m = torch.arange(t.numel(), dtype=torch.float64)
        tabs.append((t.to(torch.complex128) * torch.exp(1j * 0.3 * torch.sin(m / 97.0))).to(torch.complex64))
    kd, rf, gr, ra = _both((32, 30), grid, 6, gi.cplx((1, rows) + grid, gen), gi.cplx((1, rows, M), gen),
                           _traj(M, gen, True), tabs)
    assert rel_l2(kd, rf) < TOL and rel_l2(gr, ra) < TOL


@pytest.mark.parametrize("rows", [1, 3, 8, 12, 40])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["data", "trajectory"])
def test_values_that_are_not_finite_stay_on_their_footprint(rows, value, where):
    print(f"[case] sep {value} in {where} rows={rows}", flush=True)
    gen = torch.Generator().manual_seed(11)
    grid, M, J = (64, 60), 500, (6, 5)
    om = _traj(M, gen, False)
    y = gi.cplx((1, rows, M), gen)
    if where == "data":
        y[0, rows // 2, 3] = value
        y[0, 0, 40] = complex(1.0, value)
    else:
        om[1, 17] = value
    x = gi.cplx((1, rows) + grid, gen)
    if where == "data":
        kd, rf, gr, ra = _both((32, 30), grid, J, x, y, om)
    else:  # the oracle takes no such trajectory: the sample-lane kernels (a tile asks for them)
        ob = tkbn.KbInterp(im_size=(32, 30), grid_size=grid, numpoints=J, dtype=torch.complex64).to(DEV)
        args = (om.to(DEV), ob._tables(), ob.n_shift, ob.numpoints, ob.table_oversamp, ob.offsets)
        kd = _interp.table_interp(x.to(DEV), *args, binned=True).cpu()
        gr = _interp.table_interp_adjoint(y.to(DEV), *args, grid, deterministic=False).cpu()
        rf, ra = [], []
        for r in range(0, rows, 16):
            lane = _interp.PlanHolder(tile=(16, 16, 0)), _interp.PlanHolder(tile=(16, 16, 0))
            rf.append(_interp.table_interp(x[:, r : r + 16].to(DEV), *args, binned=True, plan=lane[0]).cpu())
            ra.append(_interp.table_interp_adjoint(y[:, r : r + 16].to(DEV), *args, grid, deterministic=False,
                                                   plan=lane[1]).cpu())
            assert _kernel().startswith("spread_tiles_kernel")
        rf, ra = torch.cat(rf, 1), torch.cat(ra, 1)
    for got, ref in ((kd, rf), (gr, ra)):
        fin = torch.isfinite(torch.view_as_real(ref)).all(-1)
        assert torch.equal(torch.isfinite(torch.view_as_real(got)).all(-1), fin)
        assert rel_l2(got[fin], ref[fin]) < TOL


def test_noalloc_adjoint_takes_the_smaller_plan_where_the_separable_one_does_not_fit():
    import ctypes

    print("[case] noalloc, 1 800 000 samples of one row", flush=True)
    gen = torch.Generator().manual_seed(13)
    grid, M, lib = (128, 128), 1800000, _lib.load()
    ad = tkbn.KbInterpAdjoint(im_size=(64, 64), dtype=torch.complex64).to(DEV)
    om = create_ktraj(2, M, gen, torch.float32).to(DEV)
    y = gi.cplx((1, 1, M), gen).to(DEV)
    tabs = [t.contiguous() for t in ad._tables()]
    desc = _interp.make_desc(y, om, tabs, ad.n_shift, ad.numpoints, ad.table_oversamp, grid, 1, 1)
    assert lib.tkbn_interp_adj_workspace_bytes(ctypes.byref(desc), 0) > lib.tkbn_interp_adj_noalloc_max_bytes()
    out = torch.full((1, 1) + grid, float("nan"), dtype=torch.complex64, device=DEV)
    st = lib.tkbn_interp_adj_noalloc(ctypes.byref(desc), y.data_ptr(), om.data_ptr(), out.data_ptr(), 0,
                                     torch.cuda.current_stream().cuda_stream)
    _lib.check(st, "tkbn_interp_adj_noalloc")
    assert _kernel().startswith("spread_tiles_kernel")
    want = _interp.table_interp_adjoint(y, om, tabs, ad.n_shift, ad.numpoints, ad.table_oversamp, ad.offsets, grid)
    assert _kernel() == "spread_sep_kernel"
    assert rel_l2(out, want) < TOL


def test_tuned_and_plain_problems_in_one_batch():
    """Separable and sample-lane problems (a tile override) side by side."""
    print("[case] batch of both kinds", flush=True)
    gen = torch.Generator().manual_seed(17)
    sizes = [(24, 24), (32, 20), (24, 24)]
    ks = [_traj(m, gen, True) for m in (900, 3000, 65)]
    bt = tkbn.BatchedKbNufft(sizes, ks, coils=6, autotune=False, fused=True)
    bt._fwd_plans[1].set_tuning((16, 16, 0), 256)
    bt._adj_plans[1].set_tuning((16, 16, 0), 256)
    for b in bt.images:
        b.copy_(gi.cplx(b.shape, gen).to(DEV))
    kd = [k.clone() for k in bt.forward()]
    im = [a.clone() for a in bt.adjoint()]
    for p, (s, k) in enumerate(zip(sizes, ks)):
        plan = tp.Plan(s, dtype=torch.complex64)
        rf = tp.kb_table_nufft(plan, bt.images[p].cpu(), k)
        assert rel_l2(kd[p], rf) < TOL, p
        assert rel_l2(im[p], tp.kb_table_nufft_adjoint(plan, kd[p].cpu(), k)) < TOL, p


def test_pair_of_few_rows_under_capture():
    print("[case] sep capture", flush=True)
    gen = torch.Generator().manual_seed(19)
    fw = tkbn.KbNufft(im_size=(40, 40), dtype=torch.complex64).to(DEV)
    ad = tkbn.KbNufftAdjoint(im_size=(40, 40), dtype=torch.complex64).to(DEV)
    om = torch.stack([_traj(2000, gen, True) for _ in range(3)]).to(DEV)
    x = gi.cplx((3, 12, 40, 40), gen).to(DEV)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            ad(fw(x, om), om)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = ad(fw(x, om), om)
    for rep in range(3):
        x.copy_(gi.cplx(x.shape, gen).to(DEV))
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(out, ad(fw(x, om), om)) < TOL, rep
