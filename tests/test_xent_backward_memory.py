"""What the backward of the fused cross-entropy holds on the device, with stand-ins on the CPU
for the kernels it launches: the operations are the real ones, the memory is counted."""
import weakref

import pytest
import torch

from oracle import xent_oracle as xo
from tritonops_amd import xent


@pytest.fixture
def on_cpu(monkeypatch):
    def dlogits(x, w, y, lse, g, dl):
        p = torch.exp(x.double() @ w.double().t() - lse[:, None].double())
        p[torch.arange(x.shape[0]), y] -= 1
        return dl.copy_(p * g[:, None].double())

    def turn(t, out):
        out.zero_()
        out[:t.shape[1], :t.shape[0]] = t.t()
        return out

    monkeypatch.setattr(xent, "_require_gpu", lambda *ts: None)
    monkeypatch.setattr(xent, "_dlogits", dlogits)
    monkeypatch.setattr(xent, "_turn", turn)
    monkeypatch.setattr(xent, "_splits_vocab", lambda rows, w: 0)


def _problem(T, D, N):
    g = torch.Generator().manual_seed(T + D + N)
    x = torch.randn((T, D), generator=g).to(torch.bfloat16)
    w = (torch.randn((N, D), generator=g) * 3 * D ** -0.5).to(torch.bfloat16)
    y = torch.randint(0, N, (T,), generator=g)
    go = torch.rand(T, generator=g) + 0.5
    return go, x, w, y, torch.logsumexp(x.double() @ w.double().t(), 1).float()


def _check(grads, go, x, w, y):
    # dlogits rounded to bf16 once (2^-9 relative each, independent) and the result once per block of rows,
    # two of them at most: 2^-8 of the norm with room
    for got, want in zip(grads, xo.linear_cross_entropy_backward(go, x, w, y)):
        assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("D", [1536, 1528], ids=["turned", "as_they_are"])
def test_a_block_is_freed_before_the_next(on_cpu, monkeypatch, D):
    go, x, w, y, lse = _problem(600, D, 72)
    alive = []

    def tracked(make):
        def call(*args):
            t = make(*args)
            alive.append(weakref.ref(t.untyped_storage()))
            return t
        return call

    rows = xent._dlogits_rows

    def first_of_a_block(*args):
        assert all(r() is None for r in alive)
        return rows(*args)

    monkeypatch.setattr(xent, "_dlogits_rows", tracked(first_of_a_block))
    monkeypatch.setattr(xent, "_room_turned", tracked(xent._room_turned))
    grads = xent._bwd(go, x, w, y, lse, None, 300)
    assert len(alive) == (6 if D == 1536 else 2)   # dlogits, x and dlogits turned, twice; or dlogits alone
    _check(grads, go, x, w, y)


# the copies of the weights, of x and of the dlogits, and grad_w, which is allocated while they are held
@pytest.mark.parametrize("fails", ["w", "x", "dlogits", "grad_w"])
@pytest.mark.parametrize("step", [300, 600], ids=["blocks", "one_block"])
def test_without_memory_for_the_copies_the_products_run_as_they_are(on_cpu, monkeypatch, fails, step):
    go, x, w, y, lse = _problem(600, 1536, 72)
    monkeypatch.setattr(xent, "_TURN_W_ROWS", 256)
    monkeypatch.setattr(xent, "_TURN_W_TILES", 1)
    room, mm, held = xent._room_turned, torch.mm, []

    def out_of_memory():
        raise torch.OutOfMemoryError("no memory")

    def empty(t):
        if tuple(t.shape) == {"w": (72, 1536), "x": (step, 1536), "dlogits": (step, 72)}.get(fails):
            out_of_memory()
        t = room(t)
        held.append(weakref.ref(t.untyped_storage()))
        return t

    def product(a, b, out=None):
        if fails == "grad_w" and out is None and any(r() is not None for r in held):
            out_of_memory()
        return mm(a, b) if out is None else mm(a, b, out=out)

    monkeypatch.setattr(xent, "_room_turned", empty)
    monkeypatch.setattr(xent.torch, "mm", product)
    grads = xent._bwd(go, x, w, y, lse, None, step)
    assert held or fails == "w"
    _check(grads, go, x, w, y)
    assert all(r() is None for r in held)


def test_copies_take_a_quarter_of_the_free_memory(on_cpu, monkeypatch):
    go, x, w, y, lse = _problem(600, 1536, 72)
    made = []
    room = xent._room_turned
    monkeypatch.setattr(xent, "_room_turned", lambda t: made.append(t.shape) or room(t))
    monkeypatch.setattr(xent.torch.cuda, "is_current_stream_capturing", lambda: False)
    need = 4 * 600 * (1536 + 72) * 2

    def kept_dlogits(kept, first, y, lse, g, N, dl, dl_t=None):
        xent._dlogits(x, w, y, lse, g, dl)
        if dl_t is not None:
            xent._turn(dl, dl_t)

    def run(free, kept=None):
        made.clear()
        monkeypatch.setattr(xent, "_free_bytes", lambda device: free)
        _check(xent._bwd(go, x, w, y, lse, kept, 768), go, x, w, y)
        return len(made)

    monkeypatch.setattr(xent, "_kept_dlogits", kept_dlogits)

    assert run(0) == 2                                   # a few MB are not asked about
    monkeypatch.setattr(xent, "KEEP_UNASKED", need // 4 - 1)
    assert run(need) == 2 and run(need - 1) == 0
    assert run(0, object()) == 2                         # the forward asked for them along with the logits it kept
    monkeypatch.setattr(xent.torch.cuda, "is_current_stream_capturing", lambda: True)
    assert run(0) == 2                                   # (its program has run the same before)


def test_the_bytes_asked_for_cover_what_is_allocated(monkeypatch):
    """Dlogits, copies and the partial sums of a divided vocabulary (fp32 tiles of 256 x 256)."""
    monkeypatch.setattr(xent, "_num_cus", lambda lib: 256)

    def asked(T, D, N):
        return xent._bwd_bytes(torch.empty((T, D), dtype=torch.bfloat16), torch.empty((N, D), dtype=torch.bfloat16))

    assert asked(40, 1024, 300) == 40 * 300 * 2                    # a small vocabulary is not divided
    n_split = xent._lib.load().mi_xent_grad_x_splits(300, 1536, 8192, 256)
    assert n_split > 1
    assert asked(300, 1536, 8192) == 300 * 8192 * 2 + 300 * (1536 + 8192) * 2 + 2 * 6 * n_split * 65536 * 4


@pytest.mark.parametrize("layout", ["rows", "columns", "padded_rows"])
def test_weights_are_turned_where_the_layout_of_grad_x_keeps_the_vocabulary_whole(on_cpu, monkeypatch, layout):
    """The divided product writes whole rows of grad_x, which has x's strides: where it cannot, w is turned as the
    rules say, and its copy is in what the memory is asked for."""
    go, x, w, y, lse = _problem(600, 1536, 72)
    x = {"rows": x, "columns": x.t().contiguous().t(), "padded_rows": torch.cat((x, x), 1)[:, :1536]}[layout]
    whole = layout == "columns"
    assert torch.empty_like(x).is_contiguous() is not whole
    monkeypatch.setattr(xent, "_TURN_W_ROWS", 256)
    monkeypatch.setattr(xent, "_TURN_W_TILES", 1)
    monkeypatch.setattr(xent, "_splits_vocab", lambda rows, w: 2)
    divided, made = [], []
    room = xent._room_turned
    monkeypatch.setattr(xent, "_room_turned", lambda t: made.append(tuple(t.shape)) or room(t))
    monkeypatch.setattr(xent, "_grad_x", lambda dl, w, out, n: divided.append(n) or out.copy_(dl.double() @ w.double()) is out)
    _check(xent._bwd(go, x, w, y, lse, None, 600), go, x, w, y)
    assert (made, divided) == (([(72, 1536)], []) if whole else ([(600, 1536), (600, 72)], [2]))
    assert xent._copy_bytes(600, x, w) == 2 * sum(a * b for a, b in made)
    split = 0 if whole else xent._lib.load().mi_xent_grad_x_workspace_bytes(600, 1536, 2)
    assert xent._bwd_bytes(x, w) == 2 * 600 * 72 + xent._copy_bytes(600, x, w) + split


def test_without_memory_for_the_partial_sums_the_library_multiplies(on_cpu, monkeypatch):
    go, x, w, y, lse = _problem(90, 136, 200)
    asked = []

    def empty(*size, dtype=None, **kw):
        if dtype == torch.uint8:
            asked.append(size)
            raise torch.OutOfMemoryError("no memory")
        return torch_empty(*size, dtype=dtype, **kw)

    torch_empty = torch.empty
    monkeypatch.setattr(xent.torch, "empty", empty)
    monkeypatch.setattr(xent, "_splits_vocab", lambda rows, w: 2)
    grads = xent._bwd(go, x, w, y, lse, None, 90)
    assert asked == [(xent._lib.load().mi_xent_grad_x_workspace_bytes(90, 136, 2),)]
    _check(grads, go, x, w, y)
