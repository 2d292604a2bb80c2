"""Operands of the fused cross-entropy's gradient products the other way round: the
transposition kernel, the second copy of the dlogits, and the gradients over them."""
import ctypes as C

import pytest
import torch

from oracle import xent_oracle as xo
from tritonops_amd import _lib

pytestmark = pytest.mark.gpu


def _turned(src):
    rows, cols = src.shape
    out = torch.full((cols + 1, -(-rows // 64) * 64), float("nan"), device="cuda", dtype=src.dtype)
    _lib.check(_lib.load().mi_transpose16(C.c_void_p(src.data_ptr()), rows, cols, src.stride(0), C.c_void_p(out.data_ptr()),
                                          out.shape[1], C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return out


@pytest.mark.parametrize("rows,cols,pitch", [(1, 8, 8), (63, 64, 64), (64, 72, 80), (65, 136, 136), (256, 8, 24),
                                             (257, 1000, 1000), (5, 4096, 4096), (3000, 200, 208)])
def test_transposition(rows, cols, pitch):
    src = torch.randn((rows, pitch), device="cuda").to(torch.float16)[:, :cols]
    out = _turned(src)
    assert torch.equal(out[:cols, :rows], src.t())
    assert (out[:cols, rows:] == 0).all()
    assert out[cols].isnan().all()            # nothing behind the last column


def test_transposition_refuses():
    lib = _lib.load()
    def call(src=4096, rows=64, cols=64, ld=64, dst=1 << 20, ld_dst=64):
        rc = lib.mi_transpose16(C.c_void_p(src), rows, cols, ld, C.c_void_p(dst), ld_dst, None)
        return lib.mi_status_name(rc).decode()
    assert call(src=0) == call(dst=0) == "MI_ERR_NULL_POINTER"
    assert call(src=4098) == call(dst=(1 << 20) + 8) == "MI_ERR_ALIGNMENT"
    assert call(cols=60) == call(rows=-1) == call(rows=1 << 30, cols=1 << 10, ld=1 << 10, ld_dst=1 << 30) == "MI_ERR_SHAPE"
    assert call(ld=56) == call(ld=68) == call(rows=65) == call(ld_dst=68) == "MI_ERR_STRIDE"
    assert call(rows=0) == call(cols=0) == "MI_OK"


@pytest.mark.parametrize("T,N", [(1, 8), (31, 129), (64, 256), (65, 257), (96, 300), (257, 1000), (320, 4096 + 37)])
def test_both_copies_of_the_dlogits(T, N):
    from tritonops_amd import xent

    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, 128), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((N, 128), device="cuda", generator=g) * 0.2).to(torch.bfloat16)
    y = torch.randint(0, N, (T,), device="cuda", generator=g)
    go = torch.rand((T,), device="cuda", generator=g)
    _, lse, kept = xent._fwd(x, w, y, True)
    want = xent._kept_dlogits(kept, 0, y, lse, go, N, xent._dlogits_rows(T, N, x))
    dl_t = torch.full((N + 1, -(-T // 64) * 64), float("nan"), device="cuda", dtype=x.dtype)
    got = xent._kept_dlogits(kept, 0, y, lse, go, N, xent._dlogits_rows(T, N, x), dl_t)
    assert torch.equal(got, want) and torch.equal(dl_t[:N, :T], want.t())
    assert (dl_t[:N, T:] == 0).all() and dl_t[N].isnan().all()


# rows, columns and tiles on either side of each rule (xent._turns_x, _turns_w), an odd vocabulary, blocks of rows
@pytest.mark.parametrize("T,D,N,block", [(300, 1536, 1000, None), (300, 1528, 1000, None), (255, 1536, 1003, None),
                                         (2100, 1024, 515, None), (4100, 2048, 203, None), (700, 1536, 600, 512)])
def test_gradients(monkeypatch, T, D, N, block):
    import tritonops_amd as ta
    from tritonops_amd import xent

    if block:
        monkeypatch.setattr(xent, "BWD_ROWS", block)
    g = torch.Generator().manual_seed(T)
    x = torch.randn((T, D), generator=g).to(torch.bfloat16)
    w = (torch.randn((N, D), generator=g) * 3 * D ** -0.5).to(torch.bfloat16)
    y = torch.randint(0, N, (T,), generator=g)
    go = torch.rand(T, generator=g) + 0.5
    got = []
    for keep in (True, False):
        xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
        loss = ta.CrossEntropyFusedFunction.apply(xg, wg, y.cuda(), keep)
        got.append(torch.autograd.grad(loss, (xg, wg), go.cuda()))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    # dlogits rounded to bf16 once (2^-9 relative each, independent) and the result once: 2^-8 of the norm with room
    for a, want in zip(got[0], xo.linear_cross_entropy_backward(go, x, w, y)):
        assert (a.cpu().double() - want).norm() <= 2.0 ** -8 * want.norm()
