"""Error of the FFT passes whose radices are products of coprime factors (6, 10, 12), against
64-bit values of random data: no larger than that of passes of radices 2 to 5 and 8.

Tolerance: the errors that such passes had on this card (forward, adjoint, filter), plus 3 %:
the 2-norm over 60 000 values and more varies by less than 1 % from draw to draw."""
import pytest
import torch

from torchkbnufft_amd._nufft import fft as _fft

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,before", [
    (100, (1.244e-7, 1.329e-7, 1.877e-7)),
    (216, (1.422e-7, 1.429e-7, 2.192e-7)),
    (1000, (1.629e-7, 1.664e-7, 2.465e-7)),
])
def test_coprime_radices_cost_no_accuracy(n, before):
    print("[case] fft error", n, flush=True)
    gen = torch.Generator().manual_seed(n)
    im, gs, dims = (n // 2, n // 2), (n, n), (-2, -1)

    def cplx(shape):
        return torch.complex(torch.randn(shape, generator=gen), torch.randn(shape, generator=gen)).to(DEV)

    def rel(a, b):
        return float(torch.linalg.norm(a.cpu().to(torch.complex128) - b) / torch.linalg.norm(b))

    one = torch.ones(im, dtype=torch.complex64, device=DEV)
    err = torch.zeros(3, dtype=torch.float64)
    for _ in range(3):
        x, grid, kern = cplx((1, 2) + im), cplx((1, 2) + gs), cplx(gs)
        full = torch.fft.fftn(x.cpu().to(torch.complex128), s=gs, dim=dims)
        back = torch.fft.ifftn(grid.cpu().to(torch.complex128), dim=dims, norm="forward")[..., : im[0], : im[1]]
        filt = torch.fft.ifftn(full * kern.cpu().to(torch.complex128), dim=dims)[..., : im[0], : im[1]]
        err += torch.tensor([
            rel(_fft.fft_grid_fwd(x, None, one, im, gs, 1.0), full),
            rel(_fft.fft_grid_adj(grid, None, one, im, 1.0), back),
            rel(_fft.fft_filter_fused(x, None, kern, False, 1.0, 1.0 / n**2), filt),
        ], dtype=torch.float64) / 3
    print(err.tolist(), flush=True)
    assert all(e < 1.03 * b for e, b in zip(err.tolist(), before))
