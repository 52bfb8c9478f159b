"""The sums of the separable spread below 32 coil rows on data of one sign in one dense spot,
cell by cell against 64-bit sums of the same table values.

Every sample sits on a table node within 0.3 cells, so the float32 and the float64 index
arithmetic agree and all terms of a cell have nearly one phase; n_shift = 0 leaves no phase
of the sample to round.  Tolerance per cell: the last rounding of the two components,
2^-24 of the cell, and the roundings of an entry's own factors (about 2^-24 each, 900
independent ones in a cell: a few percent of that): 1.5 * 2^-24."""
import numpy as np
import pytest
import torch

import torchkbnufft_amd as tkbn
from oracle import table_path as tp
from torchkbnufft_amd import _lib
from torchkbnufft_amd._nufft import interp as _interp

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
BOUND = 1.5 * 2.0**-24


@pytest.mark.parametrize("rows", [1, 3, 4, 8, 12, 16, 31])
@pytest.mark.parametrize("frames", [1, 2])
def test_cells_are_rounded_once(rows, frames):
    print(f"[case] one-sign sums rows={rows} frames={frames}", flush=True)
    im, grid, L, dense, M = (32, 30), (64, 60), 1024, 900, 600000 // frames
    rng = np.random.RandomState(rows)
    tm = np.empty((frames, 2, M))
    tm[:, 0], tm[:, 1] = rng.uniform(44, 58, (frames, M)), rng.uniform(44, 53, (frames, M))  # zero data, other tiles
    tm[:, :, :dense] = 20 + rng.randint(0, 300, (frames, 2, dense)) / L
    om = torch.tensor(tm * (2 * np.pi / np.array(grid))[:, None], dtype=torch.float32)
    y = torch.zeros((frames, rows, M), dtype=torch.complex64, device=DEV)
    amp = torch.complex(torch.linspace(1, 2, rows), torch.linspace(0.5, -0.5, rows))
    y[:, :, :dense] = amp[:, None].to(DEV)
    plan = tp.Plan(im, grid, dtype=torch.complex64)
    zero = torch.zeros(2)
    od = om if frames > 1 else om[0]
    ad = tkbn.KbInterpAdjoint(im_size=im, grid_size=grid, dtype=torch.complex64).to(DEV)
    got = _interp.table_interp_adjoint(y, od.to(DEV), [t.to(DEV) for t in plan.tables], zero.to(DEV), ad.numpoints,
                                       ad.table_oversamp, ad.offsets, grid, deterministic=False).cpu()
    assert _lib.load().tkbn_last_interp_kernel().decode() == "spread_sep_kernel"
    want = tp.table_interp_adjoint(y[:, :, :dense].cpu().to(torch.complex128), od[..., :dense].to(torch.float64),
                                   [t.to(torch.complex128) for t in plan.tables], zero.to(torch.float64),
                                   plan.t_numpoints, plan.t_table_oversamp, plan.offsets, plan.t_grid_size)
    big = want.abs() > 0.02 * want.abs().amax((-2, -1), keepdim=True)
    assert int(big.sum()) >= 12 * rows * frames
    err = ((got.to(torch.complex128) - want).abs() / want.abs())[big]
    print(f"[sums] largest error of a cell {float(err.max()):.2e}", flush=True)
    assert float(err.max()) < BOUND
