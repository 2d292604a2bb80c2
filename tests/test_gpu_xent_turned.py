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


def _split_product(dl, w, n_split):
    lib = _lib.load()
    gx = torch.full((dl.shape[0] + 1, w.shape[1]), float("nan"), device="cuda", dtype=dl.dtype)
    a = _lib.XentGradXArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = 0 if dl.dtype == torch.bfloat16 else 1
    a.tokens, a.dim, a.vocab = dl.shape[0], w.shape[1], w.shape[0]
    a.n_split = n_split or lib.mi_xent_grad_x_splits(a.tokens, a.dim, a.vocab, 256)
    a.dlogits, a.w, a.grad_x = (C.c_void_p(t.data_ptr()) for t in (dl, w, gx))
    a.ld, a.w_stride, a.grad_x_stride = dl.stride(0), w.stride(0), gx.stride(0)
    a.workspace_bytes = lib.mi_xent_grad_x_workspace_bytes(a.tokens, a.dim, a.n_split)
    ws = torch.full((a.workspace_bytes // 4 + 4,), float("nan"), device="cuda")
    a.workspace = C.c_void_p(ws.data_ptr())
    _lib.check(lib.mi_xent_grad_x(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert ws[a.workspace_bytes // 4:].isnan().all() and gx[a.tokens:].isnan().all()
    return gx[:a.tokens]


# tokens and columns on either side of a tile, vocabularies on either side of a step of 64, of a pair of them and of a
# piece of 8; what lies behind a row of dlogits holds NaN
@pytest.mark.parametrize("n_split", [0, 1, 2, 3])
@pytest.mark.parametrize("T,D,N", [(1, 8, 64), (3, 64, 65), (31, 200, 127), (256, 256, 128), (257, 264, 129), (300, 520, 192),
                                   (255, 1024, 1000), (513, 128, 5003), (40, 256, 8200)])
def test_grad_x_over_vocabulary_ranges(T, D, N, n_split):
    pairs = (-(-N // 64) + 1) // 2
    if n_split > pairs:
        pytest.skip("more ranges than pairs of steps")
    dt = torch.bfloat16 if T % 2 else torch.float16
    g = torch.Generator(device="cuda").manual_seed(T + N)
    ld = N if N % 8 == 0 else -(-N // 64) * 64
    buf = torch.full((T, ld), float("nan"), device="cuda", dtype=dt)
    buf[:, :N] = torch.randn((T, N), device="cuda", generator=g) * 0.1
    w = torch.randn((N, D + 8), device="cuda", generator=g).to(dt)[:, :D]
    got = _split_product(buf[:, :N], w, n_split)
    want = buf[:, :N].double() @ w.double()
    # one rounding to the storage type, half a unit in the last of its 8 (11) bits: 2^-8 (2^-11) of each value at most,
    # and fp32 sums of N terms, 2^-24 each of their magnitude, which is N^0.5 times the result's
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    assert ((got.double() - want).norm() <= (eps + N ** 0.5 * 2.0 ** -24) * want.norm()).item()
    assert torch.equal(got, _split_product(buf[:, :N], w, n_split))


def test_grad_x_with_values_that_are_not_finite():
    dl, w = torch.ones((4, 200), device="cuda").bfloat16(), torch.ones((200, 16), device="cuda").bfloat16()
    dl[1, 199], dl[2, 3], w[199, 5] = float("inf"), float("nan"), float("inf")
    got, want = _split_product(dl, w, 2), (dl.float() @ w.float()).bfloat16()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


def test_grad_x_refuses():
    lib = _lib.load()
    def call(**kw):
        a = _lib.XentGradXArgs()
        a.struct_size = C.sizeof(a)
        a.tokens, a.dim, a.vocab, a.n_split, a.ld, a.w_stride, a.grad_x_stride = 300, 1024, 1000, 4, 1000, 1024, 1024
        a.dlogits = a.w = a.grad_x = a.workspace = 1 << 20
        a.workspace_bytes = lib.mi_xent_grad_x_workspace_bytes(300, 1024, 4)
        for k, v in kw.items():
            setattr(a, k, v)
        return lib.mi_status_name(lib.mi_xent_grad_x(C.byref(a), None)).decode()
    assert call(tokens=0) == "MI_OK"
    assert call(struct_size=8) == "MI_ERR_STRUCT_SIZE" and call(dtype=2) == "MI_ERR_DTYPE"
    assert {call(dim=1020), call(vocab=63), call(tokens=-1), call(n_split=0), call(n_split=9)} == {"MI_ERR_SHAPE"}
    assert {call(w=None), call(grad_x=None), call(workspace=None)} == {"MI_ERR_NULL_POINTER"}
    assert call(w=(1 << 20) + 8) == "MI_ERR_ALIGNMENT"
    assert {call(ld=992), call(ld=1004), call(w_stride=1 << 23), call(grad_x_stride=1016)} == {"MI_ERR_STRIDE"}
    assert call(workspace_bytes=1000) == "MI_ERR_WORKSPACE"


# rows, columns and tiles on either side of each rule (xent._turns_x, _turns_w, _splits_vocab), an odd vocabulary, blocks of rows
@pytest.mark.parametrize("T,D,N,block", [(300, 1536, 1000, None), (300, 1528, 1000, None), (255, 1536, 1003, None),
                                         (2100, 1024, 515, None), (4100, 2048, 203, None), (700, 1536, 600, 512),
                                         (100, 1024, 9001, None), (90, 136, 8192, None), (600, 1024, 8200, 512)])
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


# several rounds of workgroups of the divided grad_x, whose rule wants more tiles than a third of the CUs and a large
# vocabulary; from 4096 rows on w would otherwise be turned
@pytest.mark.parametrize("T,D,N", [(1292, 4096, 50257), (2876, 2048, 50257), (4100, 2560, 40003)])
def test_gradients_with_uneven_rounds(monkeypatch, T, D, N):
    import tritonops_amd as ta
    from tritonops_amd import xent

    lib = _lib.load()
    n_split = lib.mi_xent_grad_x_uneven_splits(T, D, N, lib.mi_device_cu_count())
    assert n_split > 1
    divided, turned = [], []
    grad_x, turn = xent._grad_x, xent._turn
    monkeypatch.setattr(xent, "_grad_x", lambda dl, w, out, n: divided.append(n) or grad_x(dl, w, out, n))
    monkeypatch.setattr(xent, "_turn", lambda t, out: turned.append(t.shape[0]) or turn(t, out))
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, D), generator=g, device="cuda").bfloat16()
    w = (torch.randn((N, D), generator=g, device="cuda") * 3 * D ** -0.5).bfloat16()
    y = torch.randint(0, N, (T,), generator=g, device="cuda")
    go = torch.rand(T, generator=g, device="cuda") + 0.5
    got = []
    for keep in (True, False):
        xg, wg = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
        loss = ta.CrossEntropyFusedFunction.apply(xg, wg, y, keep)
        got.append(torch.autograd.grad(loss, (xg, wg), go))
    assert divided == [n_split] * 2 and N not in turned
    for a, b in zip(*got):
        assert torch.equal(a, b)
    some = torch.randperm(T, generator=g, device="cuda")[:300].sort().values   # rows; the last tile is in part behind them
    some[-1] = T - 1
    p = torch.softmax(x[some].double() @ w.double().t(), 1)
    p[torch.arange(len(some), device="cuda"), y[some]] -= 1
    want = (p * go[some, None]) @ w.double()
    # as in test_gradients: the dlogits are rounded to bf16 once and so is the result
    assert ((got[0][0][some].double() - want).norm() <= 2.0 ** -8 * want.norm()).item()
    worst = (got[0][0][some].double() - want).norm(dim=1) / want.norm(dim=1)
    assert (worst <= 2.0 ** -7).all().item()   # (of a single row: its few large dlogits carry their rounding whole)
