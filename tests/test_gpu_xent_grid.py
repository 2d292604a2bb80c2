"""Counts of token tiles that are no multiple of a panel's eight, and of vocabulary
ranges that are no multiple of anything: every (tile, range) has its workgroup."""
import pytest
import torch

from tests.util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [200, 769, 5 * 256, 21000])
@pytest.mark.parametrize("T", [1, 257, 700, 2049, 2304, 2876, 4200])
def test_every_tile_and_range(T, N):
    import tritonops_amd as ta

    D = 128
    x, w = randn((T, D), T).cuda(), (randn((N, D), N + 1) * D ** -0.5).cuda()
    y = torch.arange(T, device="cuda") * 7919 % N
    loss, lse = ta.cross_entropy_fused_fwd(x, w, y)
    logits = x.float() @ w.float().t()
    want = torch.logsumexp(logits, 1)
    # fp32 sums of 128 products of 16-bit values, and of up to 21000 exponentials: 1e-5 of values up to 20
    assert (lse - want).abs().max() <= 2e-4
    assert (loss - (want - logits.gather(1, y[:, None])[:, 0])).abs().max() <= 2e-4
    g = torch.full((T,), 0.5, device="cuda")
    dl = ta.cross_entropy_dlogits(x, w, y, lse, g)
    p = 0.5 * (torch.exp(logits - want[:, None]) - torch.nn.functional.one_hot(y, N))
    assert (dl.float() - p).abs().max() <= 3e-3   # one rounding to bf16 of values up to 0.5


@pytest.mark.parametrize("T", [95, 96, 97, 255])
def test_gradients_on_either_side_of_the_turned_operands(T):
    """From 96 rows on grad_w reads transposed copies of both its operands, padded to 64 rows."""
    import tritonops_amd as ta

    D, N = 1536, 1003
    x, w = randn((T, D), T).cuda().requires_grad_(True), (randn((N, D), 5) * D ** -0.5).cuda().requires_grad_(True)
    y = torch.arange(T, device="cuda") * 31 % N
    gx, gw = torch.autograd.grad(ta.cross_entropy_fused_triton(x, w, y).mean(), (x, w))
    xr, wr = x.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
    want = torch.autograd.grad(torch.nn.functional.cross_entropy(xr @ wr.t(), y), (xr, wr))
    for got, ref in zip((gx, gw), want):
        # dlogits and the result are rounded to bf16: 2^-8 of a value at most each
        assert ((got.double() - ref).norm() <= 2 * 2.0 ** -8 * ref.norm()).item()
