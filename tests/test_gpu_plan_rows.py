"""A trajectory's plan serves calls of any number of coil rows below 32, and of any number
from 32 on: a trusted plan (TKBN_PLAN_REUSE) built by one call is taken by the others."""
import pytest
import torch

import inputs as gi
import torchkbnufft_amd as tkbn
from conftest import create_ktraj, rel_l2
from torchkbnufft_amd._nufft import interp as _interp

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


# M: pieces at both ends of their range and between them
@pytest.mark.parametrize("M", [300, 4000, 60000])
@pytest.mark.parametrize("many", [False, True])
def test_plan_serves_other_row_counts(M, many):
    print(f"[case] plan of other rows M={M} many={many}", flush=True)
    gen = torch.Generator().manual_seed(M)
    im, grid = (64, 60), (128, 120)
    ob = tkbn.KbInterp(im_size=im, grid_size=grid, dtype=torch.complex64).to(DEV)
    om = create_ktraj(2, M, gen, torch.float32)
    om[:, : M // 3] *= 0.05
    om = om.to(DEV)
    args = (om, ob._tables(), ob.n_shift, ob.numpoints, ob.table_oversamp, ob.offsets)
    hold_f, hold_a = _interp.PlanHolder(trusted=True), _interp.PlanHolder(trusted=True)
    for rows in (64, 33, 48, 130) if many else (4, 1, 12, 31, 2, 8, 17):
        x, y = gi.cplx((1, rows) + grid, gen).to(DEV), gi.cplx((1, rows, M), gen).to(DEV)
        kd = _interp.table_interp(x, *args, plan=hold_f, binned=True)
        gr = _interp.table_interp_adjoint(y, *args, grid, deterministic=False, plan=hold_a)
        # the same values through a plan of their own; the order of float sums may differ
        assert rel_l2(kd, _interp.table_interp(x, *args, binned=True)) < 1e-6
        assert rel_l2(gr, _interp.table_interp_adjoint(y, *args, grid, deterministic=False)) < 1e-6
