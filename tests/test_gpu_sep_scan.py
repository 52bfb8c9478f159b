"""The work lists of the separable plans at the edges of their scan (rounds of 1024 tiles) and
with every class of tile: empty ones, short ones, and tiles of several pieces.

Tolerance: as for the separable kernels on other problems (2e-6 in the 2-norm); a tile that is
missed or done twice changes the result by its share of the samples."""
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


# tiles: 4, 1023, 1024, 1025, 2 x 1024 + 1 (a last round of one tile), 4096
@pytest.mark.parametrize("nb", [(2, 2), (33, 31), (32, 32), (41, 25), (3, 683), (64, 64)])
@pytest.mark.parametrize("M", [40, 9000])
def test_every_tile_once(nb, M):
    print(f"[case] scan tiles={nb} M={M}", flush=True)
    gen = torch.Generator().manual_seed(nb[0])
    grid = tuple(16 * n - 3 for n in nb)
    im = tuple(g // 2 for g in grid)
    om = create_ktraj(2, M, gen, torch.float32)
    om[:, : M // 2] *= 0.02  # pieces in the middle
    om[:, M // 2 : 2 * M // 3] = 0.03 * om[:, M // 2 : 2 * M // 3] + 1.7  # and off it
    plan = tp.Plan(im, grid, dtype=torch.complex64)
    ob = tkbn.KbInterp(im_size=im, grid_size=grid, dtype=torch.complex64).to(DEV)
    x, y = gi.cplx((1, 2) + grid, gen), gi.cplx((1, 2, M), gen)
    args = (om.to(DEV), [t.to(DEV) for t in plan.tables], ob.n_shift, ob.numpoints, ob.table_oversamp, ob.offsets)
    kd = _interp.table_interp(x.to(DEV), *args, binned=True)
    assert _lib.load().tkbn_last_interp_kernel().decode() == "gather_sep_kernel"
    gr = torch.full((1, 2) + grid, float("nan"), dtype=torch.complex64, device=DEV)
    _interp.table_interp_adjoint(y.to(DEV), *args, grid, deterministic=False, out=gr)
    assert _lib.load().tkbn_last_interp_kernel().decode() == "spread_sep_kernel"
    ref = (om, plan.tables, plan.t_n_shift, plan.t_numpoints, plan.t_table_oversamp, plan.offsets)
    assert rel_l2(kd, tp.table_interp(x, *ref)) < TOL
    assert rel_l2(gr, tp.table_interp_adjoint(y, *ref, plan.t_grid_size)) < TOL
