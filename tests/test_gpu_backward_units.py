"""The dK + dV kernel with its units dealt out at run time, whole items and halves of
64 keys (a workspace with room for the queues), against the same kernel in its fixed
order of whole items (a workspace without): a key's tiles are met in the same order
in all of them, so the bits are the same."""
import random

import pytest
import torch

from tests.util import cu_from, randn

pytestmark = pytest.mark.gpu

R = random.Random(5)
CASES = [
    # lengths (None: batched, S x B), Hq, Hkv, D, dtype, causal
    ([1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 0, 2], 6, 2, 64, torch.bfloat16, True),     # edges of tiles and halves
    ([2731, 517, 1024, 3400, 520], 32, 8, 128, torch.bfloat16, True),                              # wholes and halves
    ([4096], 32, 8, 128, torch.float16, True),                                                     # one item per workgroup
    ([8500], 16, 8, 96, torch.bfloat16, True),                                                     # more levels than lanes
    ([R.choice([0, 1, 64, 130, 257, 700]) for _ in range(64)], 4, 4, 96, torch.float16, True),     # as many sequences as lanes
    ([100] * 65, 4, 2, 64, torch.bfloat16, True),                                                  # one more: fixed order
    ([300, 77, 128, 0, 1000], 12, 3, 128, torch.bfloat16, False),                                  # no mask: all halves
    ((2, 333), 5, 5, 128, torch.bfloat16, True),
    ((1, 2000), 40, 5, 64, torch.bfloat16, True),
    ((3, 150), 3, 1, 96, torch.float16, False),
    ((8, 1000), 64, 64, 64, torch.bfloat16, False),                                                # no mask, many items: fixed order
    ([66000], 1, 1, 64, torch.bfloat16, True),                                                     # more levels than the plan holds
]


@pytest.mark.parametrize("lens,Hq,Hkv,D,dt,causal", CASES)
def test_dealt_units_equal_fixed_order(lens, Hq, Hkv, D, dt, causal, monkeypatch):
    import tritonops_amd as ta
    from tritonops_amd import _lib, ops

    if isinstance(lens, tuple):
        cu, shape = None, lens
    else:
        cu, shape = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda(), (1, sum(lens))
    q, k, v, do = (randn((*shape, h, D), 1 + i, dt).cuda() for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    sm = D ** -0.5 * ta.LOG2E
    o, lse = ops._general_fwd(q, k, v, cu, sm, causal, None, True, False)
    dealt = ops._general_bwd(q, k, v, o, do, lse, cu, sm, causal, None)
    again = ops._general_bwd(q, k, v, o, do, lse, cu, sm, causal, None)
    monkeypatch.setattr(_lib, "MI_ATTN_BWD_QUEUE_BYTES", 0)
    fixed = ops._general_bwd(q, k, v, o, do, lse, cu, sm, causal, None)
    for name, a, b, c in zip(("dq", "dk", "dv"), dealt, again, fixed):
        assert torch.isfinite(c).all(), name
        assert torch.equal(a, c) and torch.equal(b, c), name


@pytest.mark.parametrize("lens,H,D,dt,causal", [
    ([127, 128, 129, 255, 256, 257, 383, 1, 0, 65], 40, 128, torch.bfloat16, True),
    ([2100], 64, 96, torch.float16, True),
    ([500, 300], 70, 64, torch.bfloat16, False),
])
def test_query_items_of_128_rows_equal_those_of_256(lens, H, D, dt, causal):
    """Many heads at once have the long items, one head at a time the short ones."""
    import tritonops_amd as ta
    from tritonops_amd import ops

    cu, T = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda(), sum(lens)
    q, k, v, do = (randn((1, T, H, D), 1 + i, dt).cuda() for i in range(4))
    sm = D ** -0.5 * ta.LOG2E
    o, lse = ops._general_fwd(q, k, v, cu, sm, causal, None, True, False)
    grads = ops._general_bwd(q, k, v, o, do, lse, cu, sm, causal, None)
    for h in range(0, H, 7):
        p = slice(h, h + 1)
        want = ops._general_bwd(q[:, :, p], k[:, :, p], v[:, :, p], o[:, :, p], do[:, :, p], lse[:, :, p], cu, sm, causal, None)
        for name, a, b in zip(("dq", "dk", "dv"), grads, want):
            assert torch.equal(a[:, :, p], b), (name, h)
