"""The block lists of a sparse prefill are built once per call, whichever way the call takes.
(On the CPU, with stand-ins for the device, the native call and the library.)"""
import ctypes as C

import pytest
import torch

from tritonops_amd import _lib, masks, ops


class _OnDevice(torch.Tensor):
    is_cuda = True


class _Native:
    def sparse_fwd(self, *args):
        return None


class _Library:
    def mi_attn_fwd_blocksparse(self, args, stream):
        return 0


def _randn(*shape):
    return torch.randn(shape).to(torch.bfloat16).as_subclass(_OnDevice)


@pytest.mark.parametrize("form", ["packed", "int64_lengths", "slice_of_qkv", "batched", "k_apart"])
def test_built_once(monkeypatch, form):
    built = []
    block_mask_to_csr = masks.block_mask_to_csr
    monkeypatch.setattr(masks, "block_mask_to_csr", lambda *args: built.append(1) or block_mask_to_csr(*args))
    monkeypatch.setattr(_lib, "native", _Native)
    monkeypatch.setattr(_lib, "load", _Library)
    monkeypatch.setattr(ops, "_here", lambda: (0, 0))
    monkeypatch.setattr(ops, "_stream", lambda: C.c_void_p(0))
    monkeypatch.setattr(ops, "_require_gpu", lambda *ts: None)
    q, k, v, cu = _randn(1, 128, 4, 64), _randn(1, 128, 2, 64), _randn(1, 128, 2, 64), torch.tensor([0, 64, 128], dtype=torch.int32)
    if form == "int64_lengths":
        cu = cu.long()
    if form == "slice_of_qkv":
        q = _randn(1, 128, 8, 64)[:, :, :4]
    if form == "k_apart":
        k = _randn(1, 128, 2, 128)[..., ::2]
    if form == "batched":
        q, k, v, cu = q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), None
    o, lse = ops.flash_attn_sparse_triton(q, k, v, cu, block_mask=torch.ones((2, 2), dtype=torch.bool).tril())
    assert len(built) == 1
    assert o.shape == q.shape and lse.shape == q.shape[:3]
