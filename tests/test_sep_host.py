"""Sizes and decisions of the separable 2-D plans that the host makes (no GPU work)."""
import ctypes

import pytest
import torch

from torchkbnufft_amd import _lib

ATOMIC = _lib.TKBN_ADJ_ATOMIC


def _desc(batch, coils, klength, grid=(64, 60), numpoints=6, batched=False, tile=0, target=0):
    d = _lib.InterpDesc()
    d.dtype = _lib.dtype_code(torch.zeros(1, dtype=torch.complex64))
    d.ndim = len(grid)
    for i, k in enumerate(grid):
        d.grid_size[i], d.numpoints[i], d.table_oversamp[i], d.n_shift[i] = k, numpoints, 1024, k / 4
        d.tables[i] = 4096  # any non-NULL pointer: nothing reads it here
        d.tile[i] = tile
    d.work_target = target
    d.batch, d.coils, d.klength, d.omega_batched, d.flags = batch, coils, klength, int(batched), 0
    return d


def _bytes(d, direction="adj"):
    lib = _lib.load()
    if direction == "fwd":
        return int(lib.tkbn_interp_fwd_workspace_bytes(ctypes.byref(d)))
    return int(lib.tkbn_interp_adj_workspace_bytes(ctypes.byref(d), ATOMIC))


@pytest.mark.parametrize("batch,coils,batched", [(1, 0, False), (0, 3, False), (2, 0, True), (0, 3, True)])
def test_empty_problems_have_a_workspace_size(batch, coils, batched):
    """No coil rows at all: a size, as for any other problem (the pieces' size was a division
    by the rows of a chunk)."""
    d = _desc(batch, coils, 100, batched=batched)
    assert _bytes(d, "fwd") >= 0 and _bytes(d, "adj") > 0


@pytest.mark.gpu
@pytest.mark.parametrize("batch,coils", [(1, 0), (0, 3)])
def test_calls_without_rows_return_empty_results(batch, coils):
    import torchkbnufft_amd as tkbn

    ad = tkbn.KbInterpAdjoint(im_size=(32, 30), dtype=torch.complex64).cuda()
    om = torch.zeros(2, 100, device="cuda")
    out = ad(torch.zeros(batch, coils, 100, dtype=torch.complex64, device="cuda"), om)
    assert out.shape == (batch, coils, 64, 60)
