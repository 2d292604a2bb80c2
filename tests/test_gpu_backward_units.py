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
    ([8192] + [100] * 63, 8, 8, 64, torch.bfloat16, True),                                         # ids for two generations of workgroups
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


@pytest.mark.parametrize("lens,Hq,Hkv,causal", [(c[0], c[1], c[2], c[5]) for c in CASES] + [
    ([60] * 64, 2, 2, True), ([128] * 32, 4, 4, True), ([512] * 8, 8, 8, True), ([1024] * 2, 16, 16, True),  # halves gain too little
    ([65] * 3, 8, 1, True), ([64] * 3, 8, 1, True), ([512] * 4, 8, 8, True), ([512] * 8, 16, 16, True),
    ([300, 700, 20], 6, 6, True), ((2, 500), 8, 8, True), ((1, 4096), 8, 2, False), ([3000] * 43, 4, 1, True),
    ([R.randint(0, 900) for _ in range(37)], 12, 6, True), ([R.randint(0, 5000) for _ in range(6)], 4, 2, True),
    ([4096] + [100] * 63, 16, 16, True),   # two generations by the ids, four rounds of one by the items that exist
])
def test_units_taken_at_run_time(lens, Hq, Hkv, causal, monkeypatch):
    """The counters after a call: a workgroup takes another unit for each that it works on, so their sum is the
    number of units of the plan (which levels are halved with it), and zero in the fixed order."""
    import tritonops_amd as ta
    from tests.key_units import MAX_BATCH, MAX_LEVELS, Plan
    from tritonops_amd import _lib, ops

    if isinstance(lens, tuple):
        cu, shape, lens = None, lens, [lens[1]] * lens[0]
    else:
        cu, shape = cu_from(torch.tensor(lens, dtype=torch.int32)).cuda(), (1, sum(lens))
    q, k, v, do = (randn((*shape, h, 64), 1 + i, torch.bfloat16).cuda() for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    o, lse = ops._general_fwd(q, k, v, cu, 0.125 * ta.LOG2E, causal, None, True, False)
    made = []
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: made.append(empty(*a, **kw)) or made[-1])
    ops._general_bwd(q, k, v, o, do, lse, cu, 0.125 * ta.LOG2E, causal, None)
    torch.cuda.synchronize()
    ws = [t for t in made if t.dtype == torch.uint8]
    assert len(ws) == 1 and ws[0].data_ptr() % 128 == 0
    delta = -(-4 * len(lens) * Hq * max(lens) // 128) * 128
    assert ws[0].numel() >= delta + 512
    taken = ws[0][delta:delta + 512].view(torch.int32)[::16].cpu()
    cus = _lib.load().mi_device_cu_count()
    if len(lens) > MAX_BATCH or -(-max(lens) // 128) > MAX_LEVELS:
        want = 0
    else:
        # (a launch of few items has two workgroups to each)
        items = -(-max(lens) // 128) * len(lens) * Hkv
        p = Plan(lens, Hq, Hkv, causal, min(-(-2 * items // 8) * 8, cus) if items <= cus else cus)
        want = p.units() if p.dealt else 0
    assert int(taken.sum()) == want, taken


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
