"""Work items numbered by level (csrc/item_order.h): more items than workgroups, so
that every workgroup walks several.  A sequence's rows meet the same keys in the same
order wherever its items are dealt, so a packed batch must give the bits of the same
sequences called one by one (a single round each, in the order the other tests check
against the oracle)."""
import random

import pytest
import torch

from tests.util import cu_from, randn

pytestmark = pytest.mark.gpu

# 64 sequences is the largest batch the order holds, 65 falls back to the other one
CASES = [
    ([0, 1, 255, 256, 257, 0, 2049, 127, 129, 1023, 1500, 0, 640], 24, 3, 128, torch.bfloat16),
    ([random.Random(64).choice([0, 1, 64, 128, 200, 257, 513, 700]) for _ in range(63)] + [300], 16, 2, 64, torch.float16),
    ([200] * 64 + [900], 8, 8, 96, torch.bfloat16),
    ([3000], 32, 32, 128, torch.bfloat16),
]


@pytest.mark.parametrize("lens,Hq,Hkv,D,dt", CASES)
def test_ragged_batch_equals_its_sequences(lens, Hq, Hkv, D, dt):
    import tritonops_amd as ta

    T = sum(lens)
    q, k, v, do = (randn((1, T, h, D), 1 + i, dt).cuda() for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    cu = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda()
    sm = D ** -0.5 * ta.LOG2E
    for form in ("256", "128"):
        with ta.dense_form(form):
            o, lse = ta.flash_attn_triton_fwd(q, k, v, cu, sm)
        at = 0
        for n in lens:
            if n:
                s = slice(at, at + n)
                one = cu_from(torch.tensor([n], dtype=torch.int32)).cuda()
                with ta.dense_form(form):
                    for h in range(0, Hq, Hq // Hkv):      # one kv-head at a time keeps the call to one round
                        hs, kh = slice(h, h + Hq // Hkv), slice(h * Hkv // Hq, h * Hkv // Hq + 1)
                        o1, lse1 = ta.flash_attn_triton_fwd(q[:, s, hs], k[:, s, kh], v[:, s, kh], one, sm)
                        assert torch.equal(o[:, s, hs], o1) and torch.equal(lse[:, s, hs], lse1), (form, n, h)
            at += n
    grads = ta.flash_attn_triton_bwd(q, k, v, o, do, lse, cu, sm)
    at = 0
    for n in lens:
        if n:
            s = slice(at, at + n)
            one = cu_from(torch.tensor([n], dtype=torch.int32)).cuda()
            want = ta.flash_attn_triton_bwd(q[:, s], k[:, s], v[:, s], o[:, s], do[:, s], lse[:, s], one, sm)
            for a, b in zip(grads, want):
                assert torch.equal(a[:, s], b), n
        at += n


@pytest.mark.parametrize("B,H,S,D", [(2, 20, 2600, 128), (1, 40, 3000, 64)])
def test_batched_call_of_a_few_rounds(B, H, S, D):
    import tritonops_amd as ta

    q, k, v, do = (randn((B, H, S, D), 1 + i, torch.bfloat16).cuda().requires_grad_(i < 3) for i in range(4))
    o = ta.flash_attention(q, k, v)
    grads = torch.autograd.grad(o, (q, k, v), do)
    for h in range(0, H, 10):
        part = [t.detach()[:1, h:h + 5].requires_grad_(True) for t in (q, k, v)]
        o1 = ta.flash_attention(*part)
        assert torch.equal(o[:1, h:h + 5], o1), h
        for a, b in zip(grads, torch.autograd.grad(o1, part, do[:1, h:h + 5])):
            assert torch.equal(a[:1, h:h + 5], b), h


def _gpu_randn(shape, seed, dt=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=dt)


# A workgroup holds the items of 64 rounds (one per lane); beyond that a launch has several generations of
# workgroups.  256 compute units hold one workgroup of the 256-row forms and two of the 128-row form.
@pytest.mark.parametrize("B,H,S,D", [(1100, 32, 16, 128), (130, 40, 1100, 64)])
def test_more_rounds_than_a_wavefront_has_lanes(B, H, S, D):
    """Batched (unit order): the bits of calls on parts of the batch."""
    import tritonops_amd as ta

    q, k, v, do = (_gpu_randn((B, H, S, D), i) for i in range(4))
    sm = D ** -0.5 * ta.LOG2E
    for form in ("256", "128"):
        with ta.dense_form(form):
            o, lse = ta.flash_attn_triton_fwd(q, k, v, None, sm)
            for b in range(0, B, 50):
                e = min(b + 50, B)
                o1, lse1 = ta.flash_attn_triton_fwd(q[b:e], k[b:e], v[b:e], None, sm)
                assert torch.equal(o[b:e], o1) and torch.equal(lse[b:e], lse1), (form, b)
    grads = ta.flash_attn_triton_bwd(q, k, v, o, do, lse, None, sm)
    for b in range(0, B, 50):
        e = min(b + 50, B)
        want = ta.flash_attn_triton_bwd(q[b:e], k[b:e], v[b:e], o[b:e], do[b:e], lse[b:e], None, sm)
        for a, w in zip(grads, want):
            assert torch.equal(a[b:e], w), b


def test_more_rounds_by_level():
    """Packed, with more heads than models have: the bits of calls on parts of the heads."""
    import tritonops_amd as ta

    lens, H, D = [1300, 1, 700, 256, 0, 900, 257, 128], 1100, 64
    q, k, v, do = (_gpu_randn((1, sum(lens), H, D), i) for i in range(4))
    cu = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda()
    sm = D ** -0.5 * ta.LOG2E
    parts = [slice(h, min(h + 100, H)) for h in range(0, H, 100)]
    for form in ("256", "128"):
        with ta.dense_form(form):
            o, lse = ta.flash_attn_triton_fwd(q, k, v, cu, sm)
            for p in parts:
                o1, lse1 = ta.flash_attn_triton_fwd(q[:, :, p], k[:, :, p], v[:, :, p], cu, sm)
                assert torch.equal(o[:, :, p], o1) and torch.equal(lse[:, :, p], lse1), (form, p)
    grads = ta.flash_attn_triton_bwd(q, k, v, o, do, lse, cu, sm)
    for p in parts:
        want = ta.flash_attn_triton_bwd(q[:, :, p], k[:, :, p], v[:, :, p], o[:, :, p], do[:, :, p], lse[:, :, p], cu, sm)
        for a, w in zip(grads, want):
            assert torch.equal(a[:, :, p], w), p


@pytest.mark.parametrize("lens,H,D", [
    ([random.Random(i).randint(490, 700) for i in range(48)], 16, 128),   # nine rounds and more, nearly even: unit order
    ([8192, 5900, 7000], 16, 128),                                        # few and uneven: level order
    ([8192, 8101, 8192, 8040], 8, 64),
], ids=["many", "few", "alike"])
def test_rounds_enough_for_either_order(lens, H, D):
    """From six rounds up the kernels choose the order from the lengths: the bits of calls on one head."""
    import tritonops_amd as ta

    q, k, v, do = (_gpu_randn((1, sum(lens), H, D), i) for i in range(4))
    cu = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda()
    sm = D ** -0.5 * ta.LOG2E
    for form in ("256", "128"):
        with ta.dense_form(form):
            o, lse = ta.flash_attn_triton_fwd(q, k, v, cu, sm)
            for h in range(H):
                p = slice(h, h + 1)
                o1, lse1 = ta.flash_attn_triton_fwd(q[:, :, p], k[:, :, p], v[:, :, p], cu, sm)
                assert torch.equal(o[:, :, p], o1) and torch.equal(lse[:, :, p], lse1), (form, h)
    grads = ta.flash_attn_triton_bwd(q, k, v, o, do, lse, cu, sm)
    for h in range(H):
        p = slice(h, h + 1)
        want = ta.flash_attn_triton_bwd(q[:, :, p], k[:, :, p], v[:, :, p], o[:, :, p], do[:, :, p], lse[:, :, p], cu, sm)
        for a, w in zip(grads, want):
            assert torch.equal(a[:, :, p], w), h
