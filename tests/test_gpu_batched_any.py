"""Batches whose grids are not products of 2, 3, 5 (convolutions, butterflies of primes 7 to 17)
among others that are: each problem as its own module calls, eager and replayed from a graph.

Tolerance: the same FFT passes either way; the spreads' sums differ in order only (1e-6)."""
import pytest
import torch

import inputs as gi
import torchkbnufft_amd as tkbn
from conftest import create_ktraj, rel_l2

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
SIZES = [(31, 29), (32, 32), (33, 26), (31, 29), (19, 45)]


@pytest.mark.parametrize("coils", [3, 12, 40])
def test_batched_grids_of_any_factors(coils):
    print(f"[case] batched any-length coils={coils}", flush=True)
    gen = torch.Generator().manual_seed(coils)
    ks = [create_ktraj(2, 300 + 170 * p, gen, torch.float32) for p in range(len(SIZES))]
    bt = tkbn.BatchedKbNufft(SIZES, ks, coils=coils, autotune=False)
    mods = [(tkbn.KbNufft(im_size=s, dtype=torch.complex64).to(DEV),
             tkbn.KbNufftAdjoint(im_size=s, dtype=torch.complex64).to(DEV)) for s in SIZES]

    def check(images):
        for p, (fw, ad) in enumerate(mods):
            kd = fw(bt.images[p], ks[p].to(DEV))
            assert rel_l2(bt.kdata[p], kd) < 1e-6, p
            assert rel_l2(images[p], ad(kd, ks[p].to(DEV))) < 1e-6, p

    def draw():
        for b in bt.images:
            b.copy_(gi.cplx(b.shape, gen).to(DEV))

    draw()
    images = bt.pair()
    assert bt.fused == (coils < 32)
    check(images)
    bt.capture()
    for _ in range(3):
        draw()
        bt.replay()
        torch.cuda.synchronize()
        check(bt.adjoint_images)
