"""Workspaces cut from shared blocks: disjoint, per stream, also when several threads ask at
once, and given back with the cache."""
import threading

import pytest
import torch

import inputs as gi
import torchkbnufft_amd as tkbn
from conftest import create_ktraj, rel_l2
from torchkbnufft_amd._nufft import interp as _interp

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def test_workspaces_of_a_block_are_disjoint_and_given_back():
    print("[case] plan blocks", flush=True)
    gen = torch.Generator().manual_seed(5)
    M = 170000  # 12 to 15 MB a plan
    ad = tkbn.KbInterpAdjoint(im_size=(64, 64), dtype=torch.complex64).to(DEV)
    fw = tkbn.KbInterp(im_size=(64, 64), dtype=torch.complex64).to(DEV)
    y, x = gi.cplx((1, 1, M), gen).to(DEV), gi.cplx((1, 1, 128, 128), gen).to(DEV)
    oms = [create_ktraj(2, M, gen, torch.float32).to(DEV) for _ in range(7)]
    tkbn.clear_plan_cache()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    out, side = {}, [torch.cuda.Stream() for _ in range(2)]
    main = torch.cuda.current_stream()

    def work(k, stream):
        stream.wait_stream(main)
        with torch.cuda.stream(stream):
            out[k] = (fw(x, oms[k]), ad(y, oms[k]))

    ts = [threading.Thread(target=work, args=(k, side[k % 2])) for k in range(7)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    spans = sorted((w.data_ptr(), w.data_ptr() + w.numel()) for w in _interp._WORKSPACES.values())
    assert len(spans) == 14 and all(w.data_ptr() % 512 == 0 for w in _interp._WORKSPACES.values())
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    blocks = {w.untyped_storage().data_ptr() for w in _interp._WORKSPACES.values()}
    assert 4 <= len(blocks) <= 8  # two streams, four workspaces a block (a larger one starts a new block)
    tkbn.clear_plan_cache()
    for k in range(7):  # the same plans, one at a time, each in memory of its own
        assert rel_l2(out[k][0], fw(x, oms[k])) < 1e-6 and rel_l2(out[k][1], ad(y, oms[k])) < 1e-6
        tkbn.clear_plan_cache()
    out.clear()
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() <= before
