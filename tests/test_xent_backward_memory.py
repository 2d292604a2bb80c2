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
