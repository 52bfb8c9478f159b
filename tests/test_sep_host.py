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


# grids whose last tiles (16 cells) hold 16, 2 and 2 x 2 cells: up to 4, 6 and 9 tiles a sample
@pytest.mark.parametrize("grid,adj", [((640, 640), 88), ((434, 640), 96), ((434, 434), 108)])
@pytest.mark.parametrize("rows", [1, 8, 9, 12, 16, 31])
def test_plan_bytes_per_sample_below_32_rows(grid, adj, rows):
    fixed = _bytes(_desc(1, rows, 0, grid), "adj")
    M = 2000000
    assert (_bytes(_desc(1, rows, M, grid), "fwd") - _bytes(_desc(1, rows, 0, grid), "fwd")) / M < 72.1
    assert (_bytes(_desc(1, rows, M, grid), "adj") - fixed) / M < adj + 1
    # a batch item's trajectory each: the same bytes a sample
    assert (_bytes(_desc(4, rows, M // 4, grid, batched=True), "adj") - 4 * fixed) / M < adj + 1


@pytest.mark.parametrize("grid", [(640, 640), (434, 434), (18, 640)])
@pytest.mark.parametrize("rows,batch", [(1, 1), (12, 1), (31, 1), (8, 1000)])
def test_separable_workspaces_stay_within_their_limit(grid, rows, batch):
    """Sizes on both sides of the limit: a workspace either holds the separable plan, within
    1 GiB, or the sample-lane plan, as sized for a caller that tunes (a tile)."""
    seen = set()
    for M in range(1000000, 40000000, 1700000):
        d = _desc(batch, rows, M // batch, grid, batched=batch > 1)
        lane = _desc(batch, rows, M // batch, grid, batched=batch > 1, tile=32, target=512)
        for way in ("fwd", "adj"):
            n = _bytes(d, way)
            sep = n > 60 * M
            seen.add(sep)
            assert n <= (1 << 30) if sep else n < 45 * M + (1 << 26)
        assert _bytes(lane, "adj") <= max(_bytes(d, "adj"), 45 * M + (1 << 26))
    assert seen == {True, False}


def test_workspace_holds_the_larger_plan_not_both():
    d = _desc(1, 4, 200000, (512, 512))
    lane = 24 * 200000
    assert _bytes(d) < 88 * 200000 + lane


def test_frames_share_tables_and_phases():
    """Per trajectory a plan holds its samples and tile lists only: the real tables (12290
    floats here) and cell phases are one per workspace."""
    one, many = _desc(1, 1, 128, (128, 128), batched=True), _desc(1001, 1, 128, (128, 128), batched=True)
    for way, per_sample in (("fwd", 72), ("adj", 88)):
        per_frame = (_bytes(many, way) - _bytes(one, way)) / 1000
        assert per_frame < 128 * per_sample + 4 * 10 * (64 + 4)
