"""The step pipeline of the fused cross-entropy forward (xent.hip): the loads of a
step are sent a step and a half ahead, across the ends of vocabulary tiles, so the
numbers of steps of a tile and of tiles of a workgroup are where it can go wrong."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# steps of 64 elements to a tile (2, 4, 6, 14) x 256-row tiles to a workgroup (1, 2, many)
@pytest.mark.parametrize("D", [128, 256, 384, 896])
@pytest.mark.parametrize("T,N", [(256, 256), (3, 200), (257, 257), (20000, 1100), (33, 66000)])
def test_log_sum_exp_over_steps_and_tiles(T, N, D):
    from tritonops_amd import xent

    g = torch.Generator(device="cuda").manual_seed(T + N + D)
    x = torch.randn((T, D), generator=g, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn((N, D), generator=g, device="cuda") * D ** -0.5).to(torch.bfloat16)
    y = torch.randint(0, N, (T,), generator=g, device="cuda")
    loss, lse, _ = xent._fwd(x, w, y, False)
    loss_k, lse_k, kept = xent._fwd(x, w, y, True)
    assert kept is not None and torch.equal(loss, loss_k) and torch.equal(lse, lse_k)
    logits = x.float() @ w.float().t()     # exact products of 16-bit values, fp32 sums
    # fp32 sums of D terms of size one and a log-sum-exp over them: D 2^-24 of |x| |w| (about D^0.5) on either side,
    # and 2^-20 of a value of about 12
    tol = 2 * D ** 1.5 * 2.0 ** -24 + 12 * 2.0 ** -20
    assert (lse - torch.logsumexp(logits, 1)).abs().max().item() <= tol
    target = logits.gather(1, y[:, None])[:, 0]
    assert (loss - (torch.logsumexp(logits, 1) - target)).abs().max().item() <= 2 * tol
