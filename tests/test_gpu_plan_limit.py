"""The limit of the cached plan workspaces counts the memory that they keep: blocks whole, and
few blocks being cut."""
import pytest
import torch

import torchkbnufft_amd as tkbn
from torchkbnufft_amd._nufft import interp as _interp

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _workspace(x, om, nbytes=12 * MB):
    return _interp._plan_workspace("fwd", om, x, nbytes)


@pytest.fixture(autouse=True)
def _empty():
    tkbn.clear_plan_cache()
    torch.cuda.synchronize()
    yield
    tkbn.clear_plan_cache()


def test_one_workspace_kept_of_each_block(monkeypatch):
    """A quarter of the workspaces stay in use: the others' memory is held with theirs."""
    print("[case] workspaces kept of each block", flush=True)
    monkeypatch.setattr(_interp, "_WORKSPACES_MAX_BYTES", 300 * MB)
    x = torch.zeros(1, device="cuda")
    oms = torch.zeros(160, 2, 4, device="cuda")
    before = torch.cuda.memory_allocated()
    for r in range(40):
        for j in range(4):
            _workspace(x, oms[4 * r + j])
        for q in range(r + 1):
            key = [k for k in _interp._WORKSPACES if k[3] == oms[4 * q].data_ptr()]
            if key:
                _workspace(x, oms[4 * q])
        # the limit, the block being cut, and the allocator's own rounding
        assert torch.cuda.memory_allocated() - before <= (300 + 48 + 4) * MB
    assert len(_interp._WORKSPACES) >= 6


def test_few_blocks_are_kept_open():
    print("[case] open blocks of many streams", flush=True)
    x, om = torch.zeros(1, device="cuda"), torch.zeros(2, 4, device="cuda")
    before = torch.cuda.memory_allocated()
    for _ in range(12):
        with torch.cuda.stream(torch.cuda.Stream()):
            a = _workspace(x, om)
            assert _workspace(x, om) is a and not a[:256].any()
            b = _workspace(x, om, 13 * MB)  # a larger one in its place
            assert b.numel() == 13 * MB and _workspace(x, om) is b
    torch.cuda.synchronize()
    held = {w.untyped_storage().data_ptr(): w.untyped_storage().nbytes() for w in _interp._WORKSPACES.values()}
    assert {k: v[1] for k, v in _interp._HELD.items()} == held
    del a, b
    _interp._WORKSPACES.clear()
    _interp._HELD.clear()
    assert torch.cuda.memory_allocated() - before <= 4 * 54 * MB
