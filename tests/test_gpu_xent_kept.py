"""The fused cross-entropy whose forward keeps its logits for the backward:
the same values as computing them again, bit for bit, and the oracle's."""
import ctypes as C
import math

import pytest
import torch

from oracle import xent_oracle as xo


def _inputs(T, D, N, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((T, D), generator=g).to(dtype)
    w = (torch.randn((N, D), generator=g) * 3.0 / math.sqrt(D)).to(dtype)
    y = torch.randint(0, N, (T,), generator=g)
    return x, w, y, torch.rand(T, generator=g) + 0.5


def _both(x, w, y, go):
    import tritonops_amd as ta

    res = []
    for keep in (False, True):
        xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
        loss = ta.CrossEntropyFusedFunction.apply(xg, wg, y.cuda(), keep)
        assert len(loss.grad_fn.saved_tensors) == (5 if keep else 4)
        res.append((loss.detach(),) + torch.autograd.grad(loss, (xg, wg), go.cuda()))
    return res


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,D,N", [
    (1, 128, 1),             # one token, one class
    (31, 128, 129),          # one token short of a unit; one row in a tile's second half
    (33, 200, 128),          # padded hidden size; the tile's second half empty
    (256, 128, 256),         # exactly one tile
    (257, 128, 264),         # a token tile of one token; rows that end on a 16-byte piece
    (320, 256, 4096 + 37),   # several ranges; rows that no 16-byte piece fits
])
def test_kept_logits_give_the_recomputed_gradients(dtype, T, D, N):
    x, w, y, go = _inputs(T, D, N, dtype)
    if T > 30:
        y[3], y[4] = -100, N + 5  # labels outside the vocabulary
    again, kept = _both(x, w, y, go)
    for a, b in zip(again, kept):
        assert torch.equal(a, b)
    if T > 30:
        return
    dx, dw = xo.linear_cross_entropy_backward(go, x, w, y)
    # dlogits are rounded to the storage type once and the sums over them again: two roundings of at most 2^-8
    # (bf16) relative to terms no larger than the sum of magnitudes, here one row
    assert (kept[1].cpu().double() - dx).abs().max() <= 2e-2 * max(1.0, dx.abs().max().item())
    assert (kept[2].cpu().double() - dw).abs().max() <= 2e-2 * max(1.0, dw.abs().max().item())


@pytest.mark.gpu
def test_infinite_and_nan_inputs_like_recomputed():
    x, w, y, go = _inputs(64, 128, 300, torch.bfloat16)
    x[2, 5], x[3, 7], w[17, 3] = float("inf"), float("nan"), 1e30
    again, kept = _both(x, w, y, go)
    for a, b in zip(again, kept):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.gpu
def test_rows_in_blocks_and_a_second_backward(monkeypatch):
    import tritonops_amd as ta
    from tritonops_amd import xent

    x, w, y, go = _inputs(1200, 128, 700, torch.bfloat16)
    monkeypatch.setattr(xent, "BWD_ROWS", 512)
    again, kept = _both(x, w, y.to(torch.int32), go)
    for a, b in zip(again, kept):
        assert torch.equal(a, b)
    xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    loss = ta.CrossEntropyFusedFunction.apply(xg, wg, y.cuda(), True)
    first = torch.autograd.grad(loss, (xg, wg), go.cuda(), retain_graph=True)
    second = torch.autograd.grad(loss, (xg, wg), go.cuda())
    for a, b in zip(first, second):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows", [1, 255, 256, 257, 1000, 1024, 16384])
def test_row_blocks_of_kept_logits_start_on_whole_tiles(monkeypatch, rows):
    """Whatever number of rows the backward takes at a time.  (On the CPU: only where
    the blocks lie, with a stand-in for the kernel.)"""
    from tritonops_amd import xent

    blocks = []

    def kept_dlogits(kept, first, y, lse, dloss, N, dl):
        blocks.append((first, dl.shape[0]))
        return dl.zero_()

    monkeypatch.setattr(xent, "_require_gpu", lambda *ts: None)
    monkeypatch.setattr(xent, "_kept_dlogits", kept_dlogits)
    x, w, y, go = _inputs(1001, 16, 8, torch.float32)
    xent._bwd(go, x, w, y, torch.zeros(1001), object(), rows)
    assert all(first % 256 == 0 for first, _ in blocks)
    assert blocks[0][0] == 0 and sum(n for _, n in blocks) == 1001
    assert all(a + n == b for (a, n), (b, _) in zip(blocks, blocks[1:]))
    assert max(n for _, n in blocks) <= max(rows, 256)


def test_kept_rows_that_start_inside_a_tile_are_refused():
    from tritonops_amd import xent

    with pytest.raises(ValueError):
        xent._kept_dlogits(torch.zeros(1), 1000, None, None, None, 8, None)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [100, 1000])
def test_rows_in_blocks_that_are_no_whole_tiles(monkeypatch, rows):
    from tritonops_amd import xent

    x, w, y, go = _inputs(1001, 128, 700, torch.bfloat16)
    monkeypatch.setattr(xent, "BWD_ROWS", rows)
    again, kept = _both(x, w, y, go)
    assert torch.equal(again[0], kept[0])
    # both divide the rows in other blocks: dx is rounded once to bf16 (2^-8 of a value that the order of its fp32
    # sum has moved across a rounding point), dw once per block of rows, eleven of them at 100
    dx, dw = xo.linear_cross_entropy_backward(go, x, w, y)
    for got, want, tol in ((kept[1], dx, 2e-2), (kept[2], dw, 4e-2)):
        assert (got.cpu().double() - want).abs().max() <= tol * max(1.0, want.abs().max().item())


@pytest.mark.gpu
def test_when_the_logits_are_kept(monkeypatch):
    import tritonops_amd as ta
    from tritonops_amd import xent

    x, w, y, _ = _inputs(40, 1024, 300, torch.bfloat16)
    x, w, y = x.cuda(), w.cuda(), y.cuda()

    def saved(xx, ww):
        loss = ta.cross_entropy_fused_triton(xx, ww, y)
        return len(loss.grad_fn.saved_tensors)

    wg = w.clone().requires_grad_(True)
    assert saved(x, wg) == 5
    assert saved(x[:, :1016], wg[:, :1016]) == 4        # rows too short to pay
    with torch.autograd.graph.save_on_cpu():             # hooks on saved tensors
        assert not xent._keeps_logits(x, wg)
    with torch.no_grad():
        assert not xent._keeps_logits(x, wg)
    assert not xent._keeps_logits(x, w)
    monkeypatch.setattr(xent, "KEEP_BYTES", 2 * 256 * 256 * 4 - 1)
    assert saved(x, wg) == 4
    monkeypatch.setattr(xent, "KEEP_BYTES", 2 * 256 * 256 * 4)
    assert saved(x, wg) == 5


@pytest.mark.parametrize("getter,want", [
    (lambda ignore: None, True), (lambda ignore: ("pack", "unpack"), False), (lambda: None, True),
    (lambda: ("pack", "unpack"), False), (lambda a, b: None, False), (None, False)],
    ids=["none", "hooks", "none_no_argument", "hooks_no_argument", "other_signature", "no_getter"])
def test_the_getter_of_saved_tensor_hooks_may_differ(monkeypatch, getter, want):
    """torch's getter is private: without it, or with a signature that is not known, nothing is kept."""
    from tritonops_amd import xent

    monkeypatch.setattr(xent, "_saved_hooks", getter)
    x, w = torch.zeros((4, 1024)), torch.zeros((8, 1024), requires_grad=True)
    assert xent._keeps_logits(x, w) is want


def test_the_getter_of_this_torch():
    from tritonops_amd import xent

    x, w = torch.zeros((4, 1024)), torch.zeros((8, 1024), requires_grad=True)
    assert xent._keeps_logits(x, w) is True
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert xent._keeps_logits(x, w) is False


@pytest.mark.gpu
def test_all_live_graphs_share_one_budget(monkeypatch):
    import tritonops_amd as ta
    from tritonops_amd import xent

    x, w, y, _ = _inputs(40, 1024, 300, torch.bfloat16)
    x, w, y = x.cuda(), w.cuda().requires_grad_(True), y.cuda()
    one = 2 * 256 * 256 * 4
    assert not xent._kept_live
    monkeypatch.setattr(xent, "KEEP_BYTES", 3 * one - 1)

    def call(**kw):
        return ta.cross_entropy_fused_triton(x, w, y, **kw)

    def saved(loss):  # (a call in its argument holds the graph until this returns)
        return len(loss.grad_fn.saved_tensors)

    losses = [call(), call(), call()]
    assert [saved(a) for a in losses] == [5, 5, 4]
    losses[0].sum().backward(retain_graph=True)          # still held
    assert saved(call()) == 4
    losses[0].sum().backward()                           # given back by the backward pass ...
    again = call()
    assert saved(again) == 5 and saved(call()) == 4
    del losses[1]                                        # ... and with a graph that has none
    assert saved(call()) == 5
    forced = call(keep_logits=True)                      # the caller's own choice, which counts as well
    assert saved(forced) == 5 and saved(call(keep_logits=True)) == 5 and saved(call()) == 4
    del again, forced, losses
    assert not xent._kept_live and saved(call()) == 5
    assert saved(call(keep_logits=False)) == 4


@pytest.mark.gpu
def test_little_free_memory_means_no_kept_logits(monkeypatch):
    import tritonops_amd as ta
    from tritonops_amd import xent

    x, w, y, _ = _inputs(40, 1024, 300, torch.bfloat16)
    x, w, y = x.cuda(), w.cuda().requires_grad_(True), y.cuda()
    need = 4 * (2 * 256 * 256 * 4 + 40 * 300 * 2)

    def saved(**kw):
        loss = ta.cross_entropy_fused_triton(x, w, y, **kw)
        return len(loss.grad_fn.saved_tensors)

    assert xent._free_bytes(x.device) > need
    monkeypatch.setattr(xent, "_free_bytes", lambda device: need - 1)
    assert saved() == 5                                  # a few hundred KiB are not asked about
    monkeypatch.setattr(xent, "KEEP_UNASKED", 0)
    assert saved() == 4 and saved(keep_logits=True) == 5
    monkeypatch.setattr(xent, "_free_bytes", lambda device: need)
    assert saved() == 5
    out_of_memory = torch.OutOfMemoryError("no memory")

    def empty(*size, **kw):
        if size == (2 * 256 * 256,):
            raise out_of_memory
        return torch_empty(*size, **kw)

    torch_empty = torch.empty
    monkeypatch.setattr(xent.torch, "empty", empty)
    assert saved() == 4 and saved(keep_logits=True) == 4 and not xent._kept_live


@pytest.mark.gpu
def test_replays_of_a_captured_step():
    import tritonops_amd as ta

    x, w, y, go = _inputs(300, 1024, 1000, torch.bfloat16)
    xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    y, go = y.cuda(), go.cuda()

    def step():
        loss = ta.cross_entropy_fused_triton(xg, wg, y)
        return (loss.detach(),) + torch.autograd.grad(loss, (xg, wg), go)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for i in range(3):
        with torch.no_grad():
            xg.copy_(torch.roll(xg, 1, 0))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, step()):
            assert torch.equal(a, b), i


def test_kept_entry_points_validate():
    from tritonops_amd import _lib

    lib = _lib.load()

    def name(rc):
        return lib.mi_status_name(rc).decode()

    assert lib.mi_xent_kept_bytes(0, 10) == lib.mi_xent_kept_bytes(10, 0) == 0
    assert lib.mi_xent_kept_bytes(257, 256) == 2 * 256 * 256 * 4
    a = _lib.XentArgs()
    a.struct_size, a.dtype, a.tokens, a.dim, a.vocab = C.sizeof(a), _lib.MI_DTYPE_BF16, 4, 128, 16
    assert name(lib.mi_xent_fwd_keep(None, C.c_void_p(16), None)) == "MI_ERR_NULL_POINTER"
    assert name(lib.mi_xent_fwd_keep(C.byref(a), None, None)) == "MI_ERR_NULL_POINTER"
    assert name(lib.mi_xent_fwd_keep(C.byref(a), C.c_void_p(24), None)) == "MI_ERR_ALIGNMENT"
    a.tokens = 0
    assert lib.mi_xent_fwd_keep(C.byref(a), None, None) == 0
    b = _lib.XentBwdArgs()
    b.struct_size, b.dtype, b.tokens, b.vocab, b.ld = C.sizeof(b), _lib.MI_DTYPE_BF16, 4, 16, 16
    some = C.c_void_p(64)
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), some, None)) == "MI_ERR_NULL_POINTER"
    b.y = b.lse = b.dloss = b.dlogits = 64
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), None, None)) == "MI_ERR_NULL_POINTER"
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), C.c_void_p(72), None)) == "MI_ERR_ALIGNMENT"
    b.ld = 15
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), some, None)) == "MI_ERR_STRIDE"
    b.ld = b.vocab = 2 ** 31 - 1
    b.tokens = 65
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), some, None)) == "MI_ERR_SHAPE"
    b.dtype = _lib.MI_DTYPE_F32
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), some, None)) == "MI_ERR_DTYPE"
    b.struct_size = 1
    assert name(lib.mi_xent_kept_dlogits(C.byref(b), some, None)) == "MI_ERR_STRUCT_SIZE"
    assert name(lib.mi_xent_kept_dlogits(None, some, None)) == "MI_ERR_NULL_POINTER"
