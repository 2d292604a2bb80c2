"""The paired form of the dense forward (prefill.hip, dense_pair_kernel): launches of at
most one 128-row item per CU left to the library's choice, against the pinned forms of
the kernel bit for bit, and against the oracle."""
import pytest
import torch

from oracle import attention_oracle as orc
from tests.util import TOL, assert_close

pytestmark = pytest.mark.gpu


def _forms(call):
    import tritonops_amd as ta

    out = call()
    for form in ("128", "256"):
        with ta.dense_form(form):
            for a, b in zip(out, call()):
                assert torch.equal(a.nan_to_num(), b.nan_to_num()) and torch.equal(a.isnan(), b.isnan()), form
    return out


def _qkv(shape_q, shape_kv, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(s, device="cuda", generator=g).to(dtype) for s in (shape_q, shape_kv, shape_kv)]


# lengths on either side of tiles of 32 keys, of the ring of eight of them and of items of 128 rows
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (96, torch.float16), (128, torch.bfloat16), (128, torch.float16)])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 96, 127, 128, 129, 160, 161, 192, 224, 225, 255, 256, 257, 288, 300, 511, 1000, 2049])
def test_lengths(n, D, dtype, causal):
    import tritonops_amd as ta

    q, k, v = _qkv((1, 4, n, D), (1, 2, n, D), dtype, n)
    o, lse = _forms(lambda: ta.flash_attention(q, k, v, causal=causal, return_lse=True))
    ref = orc.causal_attention if causal else orc.full_attention
    kr, vr = (t.repeat_interleave(2, 1).float().cpu() for t in (k, v))
    assert_close(o, ref(q.float().cpu(), kr, vr), TOL)


@pytest.mark.parametrize("lens", [[0, 5, 0, 300, 1, 128], [500, 40, 3], [33] * 20, [0, 0], [1000]])
def test_packed_batches(lens):
    import tritonops_amd as ta

    cu = torch.tensor([0] + lens, device="cuda", dtype=torch.int32).cumsum(0).to(torch.int32)
    T = max(int(cu[-1]), 1)
    q, k, v = _qkv((1, T, 6, 128), (1, T, 3, 128), torch.bfloat16, len(lens))
    wide = _qkv((1, T, 12, 128), (1, T, 6, 128), torch.bfloat16, 1)
    for causal in (True, False):
        _forms(lambda: ta.flash_attention(q, k, v, cu, causal=causal, return_lse=True))
        _forms(lambda: ta.flash_attention(wide[0][:, :, ::2], wide[1][:, :, ::2], wide[2][:, :, ::2], cu, causal=causal, return_lse=True))
        _forms(lambda: ta.flash_attention(q, k, v, cu, causal=causal, return_lse=True, max_seq_len=64))


@pytest.mark.parametrize("slope", [0.05, 2.0, 16.0, -16.0])
@pytest.mark.parametrize("causal", [True, False])
def test_moved_reference_points(slope, causal):
    """Scores that grow along the keys: the score wavefront moves the rows' reference point at some tiles or at all,
    and the output wavefront follows."""
    import tritonops_amd as ta

    n, D = 700, 128
    q, k, v = _qkv((1, 2, n, D), (1, 2, n, D), torch.bfloat16, 3)
    k[..., 0] = torch.arange(n, device="cuda") * slope
    q[..., 0] = 1.0
    _forms(lambda: ta.flash_attention(q, k, v, causal=causal, return_lse=True, softmax_scale=1.0))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38])
@pytest.mark.parametrize("where", ["q", "k", "v"])
def test_values_that_are_not_finite(value, where):
    import tritonops_amd as ta

    q, k, v = _qkv((1, 2, 300, 64), (1, 2, 300, 64), torch.bfloat16, 3)
    {"q": q, "k": k, "v": v}[where][0, 1, 100, 7] = value
    for causal in (True, False):
        _forms(lambda: ta.flash_attention(q, k, v, causal=causal, return_lse=True))


# one sequence of more items than CUs (256 of them: up to one and a half rounds), several of up to three items per CU
@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("B,H,S", [(1, 32, 1100), (1, 32, 1536), (1, 17, 2600), (3, 16, 900), (2, 24, 2047)])
def test_more_items_than_cus(B, H, S, D):
    import tritonops_amd as ta

    q, k, v = _qkv((B, H, S, D), (B, H if H == 17 else 8, S, D), torch.bfloat16, S)
    for causal in (True, False):
        _forms(lambda: ta.flash_attention(q, k, v, causal=causal, return_lse=True))
