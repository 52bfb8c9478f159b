"""Grid sizes that are not products of 2, 3, 5: the convolution passes against 64-bit torch.fft.

Tolerance: a convolution is two float32 transforms of M <= 1280 values and three chirp
products, rms error about (2 log2(M) + 6) * 2^-24 * 0.6 = 9.3e-7 a dimension at most; three
dimensions of it stay under 2e-6 (root sum of squares 1.6e-6).
"""
import pytest
import torch

import torchkbnufft_amd as tkbn
from torchkbnufft_amd._nufft import fft as _fft

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 2e-6

# (image, grid): primes, a smooth dimension beside one that is not, no oversampling, the
# edges of the convolution lengths (im + grid - 1 = 192, 193, 1024, 1025, 1152, 1153, 1280),
# one value, 1-D, 3-D
CASES = [
    ((33, 24), (66, 48)),
    ((217, 181), (434, 362)),
    ((24, 33), (48, 67)),
    ((7,), (7,)),
    ((19,), (19,)),
    ((1, 1), (7, 11)),
    ((97, 13), (97, 13)),
    ((62,), (131,)),
    ((55, 64), (139, 130)),
    ((340, 5), (685, 11)),
    ((6, 342), (14, 684)),
    ((384, 384), (769, 770)),
    ((5, 427), (22, 854)),
    ((9, 14, 11), (19, 28, 22)),
    ((8, 15, 23), (16, 30, 46)),
    ((63, 75), (126, 150)),
    ((17, 13), (34, 26)),
    ((11,), (221,)),
    ((17, 60), (17, 119)),
    ((21, 13, 16), (49, 26, 32)),
]


def _rel(a, b):
    b = b.to(torch.complex128)
    return float(torch.linalg.norm(a.to(torch.complex128) - b) / torch.linalg.norm(b))


def _cplx(shape, gen):
    return torch.complex(torch.randn(shape, generator=gen), torch.randn(shape, generator=gen)).to(DEV)


@pytest.mark.parametrize("im,gs", CASES)
@pytest.mark.parametrize("coils,maps", [(1, False), (5, False), (3, True)])
def test_any_length_matches_64_bit(im, gs, coils, maps):
    print("[case]", im, gs, coils, maps, flush=True)
    gen = torch.Generator().manual_seed(sum(im) + coils)
    d = len(im)
    dims = tuple(range(-d, 0))
    assert not _fft.fused_supported(torch.complex64, im, gs) and _fft.pipeline_supported(torch.complex64, im, gs)
    image, grid = _cplx((2, 1 if maps else coils) + im, gen), _cplx((2, coils) + gs, gen)
    sm = _cplx((2, coils) + im, gen) if maps else None
    sc = _cplx(im, gen)
    got = _fft.fft_grid_fwd(image, sm, sc, im, gs, 0.5)
    x = image.to(torch.complex128) * sc
    x = x * sm if maps else x
    want = torch.fft.fftn(x.cpu(), s=gs, dim=dims) * 0.5
    assert _rel(got.cpu(), want) < TOL
    back = _fft.fft_grid_adj(grid, sm, sc, im, 0.5)
    y = torch.fft.ifftn(grid.to(torch.complex128).cpu(), dim=dims, norm="forward")
    for ax, n in enumerate(im):
        y = y.narrow(2 + ax, 0, n)
    y = y * sc.cpu().conj() * 0.5
    if maps:
        y = (y * sm.cpu().conj()).sum(1, keepdim=True)
    assert back.shape == y.shape and _rel(back.cpu(), y) < TOL


def test_module_route_switch_capture_and_limits():
    """Same results as with torch.fft through the modules, replayed from a graph too; larger
    convolutions, complex128 and the C entry of the planned sizes keep their routes."""
    print("[case] any-length route", flush=True)
    gen = torch.Generator().manual_seed(3)
    im, gs = (33, 24), (66, 48)
    nufft = tkbn.KbNufft(im_size=im, dtype=torch.complex64).to(DEV)
    om = ((torch.rand(2, 500, generator=gen) - 0.5) * 6).to(DEV)
    image, sm = _cplx((2, 1) + im, gen), _cplx((1, 4) + im, gen)
    here = nufft(image, om, smaps=sm)
    _fft.set_fused_fft(False)
    try:
        assert not _fft.pipeline_supported(torch.complex64, im, gs)
        there = nufft(image, om, smaps=sm)
    finally:
        _fft.set_fused_fft(True)
    assert _rel(here, there) < TOL
    sc, out = _cplx(im, gen), torch.empty((2, 4) + gs, dtype=torch.complex64, device=DEV)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        _fft.fft_grid_fwd(image, sm, sc, im, gs, 1.0, out=out)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            _fft.fft_grid_fwd(image, sm, sc, im, gs, 1.0, out=out)
    for k in range(3):
        image.copy_(_cplx((2, 1) + im, gen))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, _fft.fft_grid_fwd(image, sm, sc, im, gs, 1.0)), k
    assert not _fft.pipeline_supported(torch.complex128, im, gs)
    assert not _fft.pipeline_supported(torch.complex64, (430, 8), (862, 16))
