"""The staged FFT passes at the edges of their work split, against the float64 transform.

Tolerance: an FFT in float32 is off by a small multiple of eps log2(prod K) in the 2-norm;
4 eps log2(prod K) leaves room for the scaling and coil products."""
import math

import pytest
import torch

import inputs as gi
from conftest import rel_l2
from oracle import table_path as tp
from torchkbnufft_amd._nufft import fft as F

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")

GEOMS = [
    # every radix alone and in pairs, lengths of one value, lone radices, many stages
    ((1,), (1,), 2, 1), ((1, 3), (2, 3), 1, 2), ((2, 5), (4, 5), 1, 2), ((4, 3), (9, 6), 3, 1), ((5, 6), (10, 12), 1, 3),
    ((8, 7), (16, 15), 1, 2), ((13, 40), (27, 81), 1, 2), ((62, 121), (125, 243), 1, 2), ((100, 9), (625, 18), 1, 1),
    # compiled lengths (288, 400, 480, 576, 1024, 128, 160) with N = K/2, less, odd, and more than half
    ((144, 200), (288, 400), 1, 3), ((240, 288), (480, 576), 2, 1), ((512, 64), (1024, 128), 1, 1),
    ((77, 31), (160, 128), 2, 2), ((100, 130), (160, 192), 1, 2), ((320, 256), (320, 256), 1, 1),
    # more coils than lines of a group, ragged last groups of lines and columns, three dimensions
    ((40, 64), (80, 128), 1, 37), ((33, 50), (72, 100), 3, 5), ((3, 320), (6, 640), 1, 17), ((5, 9, 11), (10, 18, 24), 2, 3),
    ((7, 4, 64), (15, 8, 128), 1, 9),
    # longest
    ((2, 1024), (4, 2048), 1, 3), ((1024, 3), (2048, 6), 1, 1),
]


@pytest.mark.parametrize("im,gs,B,C", GEOMS)
def test_stages_match_float64(im, gs, B, C):
    print(f"[case] fft stages {im}->{gs} B={B} C={C}", flush=True)
    assert F.fused_supported(torch.complex64, im, gs)
    gen = torch.Generator().manual_seed(len(im) * 100 + im[0])
    tol = 4 * 2.0**-24 * max(2.0, math.log2(math.prod(gs)))
    plan = tp.Plan(im, gs, dtype=torch.complex64)
    sc = plan.scaling_coef
    dims = list(range(-len(im), 0))
    box = (Ellipsis,) + tuple(slice(0, n) for n in im)
    for smaps in (False, True):
        x = gi.cplx((B, 1 if smaps else C) + im, gen)
        s = gi.cplx((B, C) + im, gen) if smaps else None
        g = gi.cplx((B, C) + gs, gen)
        x64, sc64 = x.to(torch.complex128), sc.to(torch.complex128)
        ref = torch.fft.fftn((x64 * s if smaps else x64) * sc64, s=gs, dim=dims)
        got = F.fft_grid_fwd(x.to(DEV), s.to(DEV) if smaps else None, sc.to(DEV), im, gs, 1.0).cpu()
        assert rel_l2(got.to(torch.complex128), ref) < tol
        ref_a = torch.fft.ifftn(g.to(torch.complex128), dim=dims, norm="forward")[box] * sc64.conj()
        if smaps:
            ref_a = (ref_a * s.conj()).sum(1, keepdim=True)
        got_a = F.fft_grid_adj(g.to(DEV), s.to(DEV) if smaps else None, sc.to(DEV), im, 1.0).cpu()
        assert rel_l2(got_a.to(torch.complex128), ref_a) < tol
        if len(im) > 1:
            kern = gi.cplx(gs, gen)
            ref_f = torch.fft.ifftn(torch.fft.fftn(x64 * s if smaps else x64, s=gs, dim=dims) * kern, dim=dims,
                                    norm="forward")[box]
            if smaps:
                ref_f = (ref_f * s.conj()).sum(1, keepdim=True)
            got_f = F.fft_filter_fused(x.to(DEV), s.to(DEV) if smaps else None, kern.to(DEV), False, 1.0, 1.0).cpu()
            assert rel_l2(got_f.to(torch.complex128), ref_f) < 2 * tol
