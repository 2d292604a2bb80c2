"""The merge of decode chunks in its three forms (up to 64 slots, up to 256, any number):
a row's bits are those of the same chunks merged among more slots, and the result is
that of plain softmax attention in fp32."""
import pytest
import torch

from tests.util import assert_close, randn

pytestmark = pytest.mark.gpu

LENS = [0, 1, 64, 65, 31 * 64 + 5, 32 * 64, 32 * 64 + 1, 63 * 64 + 9, 64 * 64, 64 * 64 + 1, 96 * 64 + 3, 255 * 64, 256 * 64, 256 * 64 + 1, 300 * 64]


@pytest.mark.parametrize("D,dt", [(64, torch.float16), (96, torch.bfloat16), (128, torch.bfloat16)])
def test_slots_at_the_edges_of_the_forms(D, dt):
    import tritonops_amd as ta

    room = 300 * 64
    q, k, v = randn((1, 6, D), 1, dt).cuda(), randn((1, room, 2, D), 2, dt).cuda(), randn((1, room, 2, D), 3, dt).cuda()
    for n in LENS:
        sl = torch.tensor([n], dtype=torch.int32, device="cuda")
        want = None
        for slots in (1, 2, 32, 33, 64, 65, 256, 257, 300):
            if slots * 64 < n:
                continue
            got = ta.flash_attention_decoding(q, k[:, :slots * 64], v[:, :slots * 64], None, seq_lens=sl, split_tokens=64, return_lse=True)
            if want is None:
                want = got
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (n, slots)
        if n == 0:
            assert (want[0] == 0).all() and (want[1] == float("-inf")).all()
            continue
        qf, kf, vf = q[0].float(), k[0, :n].float().repeat_interleave(3, 1), v[0, :n].float().repeat_interleave(3, 1)
        s = torch.einsum("hd,nhd->hn", qf, kf) * D ** -0.5
        # chunks are accurate to the rounding of their probabilities, the result is rounded once more
        assert_close(want[0][0].cpu(), torch.einsum("hn,nhd->hd", torch.softmax(s, 1), vf).cpu(), 1e-2 if dt == torch.bfloat16 else 2e-3)


@pytest.mark.parametrize("layout", ["batched", "packed", "paged"])
def test_more_sequences_than_lanes(layout):
    """Lengths, first rows and pages of sequences behind the 64th: the bits of the same rows alone."""
    import tritonops_amd as ta

    lens = [(37 * i) % 200 for i in range(70)]
    B, room, H, Hkv, D = 70, 256, 4, 2, 128
    q, k, v = randn((B, H, D), 1).cuda(), randn((B, room, Hkv, D), 2).cuda(), randn((B, room, Hkv, D), 3).cuda()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    want = torch.cat([ta.flash_attention_decoding(q[i:i + 1], k[i:i + 1], v[i:i + 1], None, seq_lens=sl[i:i + 1], split_tokens=64)
                      for i in range(B)])
    cu = torch.cat([sl.new_zeros(1), sl.cumsum(0).to(torch.int32)])
    if layout == "batched":
        got = ta.flash_attention_decoding(q, k, v, cu, split_tokens=64)
    elif layout == "packed":
        kp, vp = (torch.cat([t[i, :n] for i, n in enumerate(lens)])[None].contiguous() for t in (k, v))
        got = ta.flash_attention_decoding(q, kp, vp, cu, kv_layout="packed", max_seq_len=room, split_tokens=64)
    else:
        order = torch.randperm(B * 4, generator=torch.Generator().manual_seed(1)).cuda()
        kp, vp = torch.empty_like(k).view(B * 4, 64, Hkv, D), torch.empty_like(v).view(B * 4, 64, Hkv, D)
        kp[order], vp[order] = k.view(B * 4, 64, Hkv, D), v.view(B * 4, 64, Hkv, D)
        got = ta.flash_attention_decoding(q, kp, vp, cu, kv_layout="paged", page_table=order.view(B, 4).to(torch.int32), split_tokens=64)
    assert torch.equal(got, want)
