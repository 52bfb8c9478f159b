"""Adjoint FFT with coil maps on grids that are not products of 2, 3, 5: the last pass sums the
coils itself wherever the last dimension is no convolution and is short enough, whatever the
others are.

Tolerance: per dimension at most a convolution's rms error, (2 log2(M) + 6) * 2^-24 * 0.6 =
9.3e-7 for M <= 1280 (a planned dimension has less than half); two dimensions, the maps' product
and the sum of the coils stay under 2e-6.
"""
import pytest
import torch

from torchkbnufft_amd._nufft import fft as _fft

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 2e-6

# (image, grid, coils, combined by the last pass): last dimensions of primes 7 to 17, one lone
# radix, a smooth one, the longest line; coils on both sides of a group's lines (16 at most, fewer
# where LDS holds no more), in several rounds where there are 256 lines of the image; a convolution
# before the last dimension, and as the last
CASES = [
    ((9, 13), (18, 26), 3, True),
    ((9, 11), (18, 11), 16, True),
    ((9, 11), (18, 11), 17, False),
    ((128, 24), (143, 48), 40, True),
    ((127, 24), (254, 48), 40, False),
    ((128, 45), (130, 91), 17, True),
    ((31, 13), (62, 26), 5, True),
    ((19, 45), (38, 90), 16, True),
    ((3, 385), (7, 770), 16, True),
    ((3, 400), (7, 800), 11, True),
    ((3, 401), (7, 819), 11, False),
    ((2, 1024), (4, 2002), 4, False),
    ((7,), (14,), 9, True),
    ((5, 6, 7), (11, 12, 14), 6, True),
    ((13, 31), (26, 62), 5, False),
    ((16, 19), (32, 38), 3, False),
]


def _rel(a, b):
    return float(torch.linalg.norm(a.to(torch.complex128) - b) / torch.linalg.norm(b))


@pytest.mark.parametrize("im,gs,coils,combined", CASES)
def test_last_pass_sums_the_coils(im, gs, coils, combined, monkeypatch):
    print("[case]", im, gs, coils, flush=True)
    gen = torch.Generator().manual_seed(sum(gs) + coils)

    def cplx(shape):
        return torch.complex(torch.randn(shape, generator=gen), torch.randn(shape, generator=gen)).to(DEV)

    grid, sm, sc = cplx((2, coils) + gs), cplx((2, coils) + im), cplx(im)
    extra, into = [], _fft._crop_deapod_into
    monkeypatch.setattr(_fft, "_crop_deapod_into", lambda *a: (extra.append(1), into(*a))[1])
    got = _fft.fft_grid_adj(grid, sm, sc, im, 0.5)
    y = torch.fft.ifftn(grid.to(torch.complex128).cpu(), dim=tuple(range(-len(im), 0)), norm="forward")
    for ax, n in enumerate(im):
        y = y.narrow(2 + ax, 0, n)
    want = (y * sc.cpu().conj() * 0.5 * sm.cpu().conj()).sum(1, keepdim=True)
    assert got.shape == want.shape and _rel(got.cpu(), want) < TOL
    assert (not extra) == combined
