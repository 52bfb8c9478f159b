"""The separable spread with one wave per piece and with four, in every form, with pieces,
entries left out of the products, and in batches whose launch differs from the problems' own.

Tolerance: as for the separable kernels on other problems, float32 roundings of some hundred
terms a cell (2e-6 in the 2-norm)."""
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
IM, GRID = (100, 92), (200, 184)  # 13 x 12 tiles
# four waves share a piece from 32 entries a tile on (7/4 entries a sample): 2800 samples take
# one wave, 4000 four
ONE, FOUR = 2800, 4000


def _kernel():
    return _lib.load().tkbn_last_interp_kernel().decode()


def _crowded(M, gen, n):
    """Uniform samples, the first n in one tile (more than a piece's entries)."""
    om = create_ktraj(2, M, gen, torch.float32)
    om[:, :n] = 0.3 + 0.05 * om[:, :n]
    return om


def _adjoint(y, om, tabs, plan):
    ob = tkbn.KbInterp(im_size=IM, grid_size=GRID, dtype=torch.complex64).to(DEV)
    got = _interp.table_interp_adjoint(y.to(DEV), om.to(DEV), [t.to(DEV) for t in tabs], ob.n_shift, ob.numpoints,
                                       ob.table_oversamp, ob.offsets, GRID, deterministic=False)
    assert _kernel() == "spread_sep_kernel"
    ref = tp.table_interp_adjoint(y, om, tabs, plan.t_n_shift, plan.t_numpoints, plan.t_table_oversamp, plan.offsets,
                                  plan.t_grid_size)
    return got.cpu(), ref


@pytest.mark.parametrize("M", [ONE, FOUR])
@pytest.mark.parametrize("rows", [1, 2, 4, 8, 12, 17, 40])
@pytest.mark.parametrize("what", ["plain", "other tables", "not finite"])
def test_forms_and_waves(M, rows, what):
    print(f"[case] waves M={M} rows={rows} {what}", flush=True)
    gen = torch.Generator().manual_seed(rows)
    plan = tp.Plan(IM, GRID, dtype=torch.complex64)
    tabs, om, y = plan.tables, _crowded(M, gen, 1200), gi.cplx((1, rows, M), gen)
    if what == "other tables":  # every entry left out, more and fewer than a wave remembers
        m = torch.arange(tabs[0].numel(), dtype=torch.float64)
        tabs = [(t.to(torch.complex128) * torch.exp(1j * 0.3 * torch.sin(m / 97.0))).to(torch.complex64) for t in tabs]
    elif what == "not finite":
        y[0, rows // 2, 3] = float("nan")  # in the split tile
        y[0, 0, 700:760] = complex(1.0, float("inf"))  # more than a wave remembers
        y[0, rows - 1, M - 5 : M - 2] = float("-inf")
    got, ref = _adjoint(y, om, tabs, plan)
    fin = torch.isfinite(torch.view_as_real(ref)).all(-1)
    assert bool(fin.all()) == (what != "not finite")
    assert torch.equal(torch.isfinite(torch.view_as_real(got)).all(-1), fin)
    assert rel_l2(got[fin], ref[fin]) < TOL


@pytest.mark.parametrize("sizes,M", [
    ([(256, 256)] * 5, [21000] * 5),  # four waves each, one in the batch (5 x 1024 tiles)
    ([(100, 92), (100, 92), (32, 32)], [600, 60000, 200]),  # one wave each for two of them, four in the batch
])
@pytest.mark.parametrize("coils", [2, 9])
def test_batches_that_launch_otherwise_than_their_problems(sizes, M, coils):
    print(f"[case] waves batch {sizes[0]} x {len(sizes)} coils={coils}", flush=True)
    gen = torch.Generator().manual_seed(coils)
    ks = [_crowded(m, gen, m // 4) for m in M]
    bt = tkbn.BatchedKbNufft(sizes, ks, coils=coils, autotune=False, fused=True)
    for b in bt.kdata:
        b.copy_(gi.cplx(b.shape, gen).to(DEV))
    im = [a.clone() for a in bt.adjoint()]
    for p in range(len(sizes)):
        ad = tkbn.KbNufftAdjoint(im_size=sizes[p], dtype=torch.complex64).to(DEV)
        assert rel_l2(im[p], ad(bt.kdata[p], ks[p].to(DEV))) < TOL
    plan = tp.Plan(sizes[1], dtype=torch.complex64)
    assert rel_l2(im[1], tp.kb_table_nufft_adjoint(plan, bt.kdata[1].cpu(), ks[1])) < TOL
