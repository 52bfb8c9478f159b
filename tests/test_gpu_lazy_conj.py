"""Tensors with a lazy conjugate (torch sets a bit and leaves the memory) give what their
values give, in each argument a kernel reads and in the gradients autograd hands back.

Tolerance: the same kernels on the same values; only the order of the adjoint's sums may
differ from call to call, a few float32 roundings (1e-6)."""
import pytest
import torch

import inputs as gi
import torchkbnufft_amd as tkbn
from conftest import create_ktraj, rel_l2
from torchkbnufft_amd._nufft import fft as _fft

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
TOL = 1e-6


def _c(shape, gen):
    return gi.cplx(shape, gen).to(DEV)


@pytest.mark.parametrize("im,gs", [((33, 24), (66, 48)), ((32, 24), (64, 48)), ((24, 33), (48, 67))])
@pytest.mark.parametrize("maps", [False, True])
def test_fft_stages(im, gs, maps):
    print("[case] lazy conj fft", im, gs, maps, flush=True)
    gen = torch.Generator().manual_seed(1)
    sc = _c(im, gen)
    x, g = _c((2, 1 if maps else 3) + im, gen).conj(), _c((2, 3) + gs, gen).conj()
    sm = _c((2, 3) + im, gen).conj() if maps else None
    rsm = None if sm is None else sm.resolve_conj()
    assert x.is_conj() and g.is_conj()
    assert rel_l2(_fft.fft_grid_fwd(x, sm, sc, im, gs, 1.0), _fft.fft_grid_fwd(x.resolve_conj(), rsm, sc, im, gs, 1.0)) < TOL
    assert rel_l2(_fft.fft_grid_adj(g, sm, sc, im, 1.0), _fft.fft_grid_adj(g.resolve_conj(), rsm, sc, im, 1.0)) < TOL


def test_module_calls_and_gradients():
    print("[case] lazy conj modules", flush=True)
    gen = torch.Generator().manual_seed(2)
    im = (33, 24)
    fw = tkbn.KbNufft(im_size=im, dtype=torch.complex64).to(DEV)
    ad = tkbn.KbNufftAdjoint(im_size=im, dtype=torch.complex64).to(DEV)
    om = create_ktraj(2, 700, gen, torch.float32).to(DEV)
    x, y = _c((1, 2) + im, gen), _c((1, 2, 700), gen)
    assert rel_l2(fw(x.conj(), om), fw(x.conj().resolve_conj(), om)) < TOL
    assert rel_l2(ad(y.conj(), om), ad(y.conj().resolve_conj(), om)) < TOL
    grads = []
    for lazy in (True, False):
        xr, yr = x.clone().requires_grad_(True), y.clone().requires_grad_(True)
        for out in (fw(xr, om), ad(yr, om)):  # the gradient arrives as a lazy conjugate
            c = out.conj() if lazy else out.conj().resolve_conj()
            c.backward(torch.full_like(c, 1 + 2j))
        grads.append((xr.grad, yr.grad))
    for a, b in zip(*grads):
        assert rel_l2(a, b) < TOL


def test_toeplitz_filter_gradient():
    print("[case] lazy conj filter", flush=True)
    gen = torch.Generator().manual_seed(3)
    x, k = _c((1, 2, 16, 16), gen), _c((32, 32), gen)
    xr = x.clone().requires_grad_(True)
    w = _c((1, 2, 16, 16), gen)
    out = _fft.fft_filter(xr, k, norm="ortho")
    out.backward(w)
    assert rel_l2(xr.grad, _fft.fft_filter(w, k.conj().resolve_conj(), norm="ortho")) < TOL
