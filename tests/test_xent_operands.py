"""The fused cross-entropy's kernels take w's element type, width and device from x: operands
that differ in one of them are refused before anything is allocated or launched."""
import pytest
import torch

from tritonops_amd import xent


@pytest.fixture(autouse=True)
def nothing_runs(monkeypatch):
    def load():
        raise AssertionError("the library was reached")

    monkeypatch.setattr(xent, "_require_gpu", lambda *ts: None)
    monkeypatch.setattr(xent._lib, "load", load)


# vocabularies on either side of xent._SPLIT_VOCAB, from which on grad_x comes from a kernel of this library
@pytest.mark.parametrize("N", [4096, 8192])
@pytest.mark.parametrize("w,error", [
    (dict(dtype=torch.float32), TypeError), (dict(dtype=torch.float16), TypeError),
    (dict(device="meta"), ValueError), (dict(cols=120), ValueError), (dict(cols=136), ValueError)],
    ids=["fp32", "fp16", "device", "narrow", "wide"])
@pytest.mark.parametrize("kept", [None, object()], ids=["recomputed", "kept"])
def test_backward(N, w, error, kept):
    x, y = torch.zeros((64, 128), dtype=torch.bfloat16), torch.zeros(64, dtype=torch.int64)
    w = torch.zeros((N, w.get("cols", 128)), dtype=w.get("dtype", torch.bfloat16), device=w.get("device", "cpu"))
    lse = go = torch.zeros(64)
    with pytest.raises(error):
        xent._bwd(go, x, w, y, lse, kept, xent.BWD_ROWS)
    with pytest.raises(error):
        xent.cross_entropy_dlogits(x, w, y, lse, go)
    with pytest.raises(error):
        xent.cross_entropy_fused_fwd(x, w, y)


def test_only_16_bit_elements_are_turned():
    assert xent._can_turn(torch.zeros((8, 64), dtype=torch.float16))
    assert not xent._can_turn(torch.zeros((8, 64), dtype=torch.float32))
