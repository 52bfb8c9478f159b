"""Many short trajectories, one per batch item, on the separable kernels: their plans share the
tables and cell phases, and the verdict on the tables' form.

Tolerance: as for the separable kernels on other problems, float32 roundings of at most some
hundred terms a cell (2e-6 in the 2-norm)."""
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


@pytest.mark.parametrize("frames,M", [(300, 1), (60, 70), (2, 600)])
@pytest.mark.parametrize("other_form", [False, True])
def test_short_frames(frames, M, other_form):
    print(f"[case] frames={frames} M={M} other_form={other_form}", flush=True)
    gen = torch.Generator().manual_seed(frames)
    im, grid = (20, 17), (40, 34)
    plan = tp.Plan(im, grid, dtype=torch.complex64)
    tabs = plan.tables
    if other_form:
        m = [torch.arange(t.numel(), dtype=torch.float64) for t in tabs]
        tabs = [(t.to(torch.complex128) * torch.exp(1j * 0.3 * torch.sin(k / 97.0))).to(torch.complex64)
                for t, k in zip(tabs, m)]
    ob = tkbn.KbInterp(im_size=im, grid_size=grid, dtype=torch.complex64).to(DEV)
    om = torch.stack([create_ktraj(2, M, gen, torch.float32) for _ in range(frames)])
    x, y = gi.cplx((frames, 2) + grid, gen), gi.cplx((frames, 2, M), gen)
    args = (om.to(DEV), [t.to(DEV) for t in tabs], ob.n_shift, ob.numpoints, ob.table_oversamp, ob.offsets)
    kd = _interp.table_interp(x.to(DEV), *args, binned=True)
    assert _lib.load().tkbn_last_interp_kernel().decode() == "gather_sep_kernel"
    gr = _interp.table_interp_adjoint(y.to(DEV), *args, grid, deterministic=False)
    assert _lib.load().tkbn_last_interp_kernel().decode() == "spread_sep_kernel"
    ref = (om, tabs, plan.t_n_shift, plan.t_numpoints, plan.t_table_oversamp, plan.offsets)
    assert rel_l2(kd, tp.table_interp(x, *ref)) < TOL
    assert rel_l2(gr, tp.table_interp_adjoint(y, *ref, plan.t_grid_size)) < TOL
