"""How a decoding launch divides its work (csrc/decode.hip): chunks of split_tokens
tokens or split_blocks blocks, one, two or four wavefronts to a chunk, and slots of
the workspace that stay empty.  The workspace comes out of memory that held NaN, so
a slot that is used without having been written shows."""
import pytest
import torch

from oracle import attention_oracle as orc
from tests.util import assert_close, randn

pytestmark = pytest.mark.gpu
TOL = 2e-2

LONG = [3000, 0, 1, 31, 32, 33, 4095, 2048, 0, 700]
CASES = [
    # lens, Hq, Hkv, D, split_tokens, max_seq_len
    (LONG, 32, 8, 128, 64, None),         # many slots of two tiles
    (LONG * 6, 32, 8, 128, 2048, None),   # two slots to a sequence
    (LONG * 6, 64, 32, 96, 512, None),    # several rounds of chunks
    (LONG * 13, 16, 16, 64, 256, None),   # 130 sequences: the search steps over the batch
    (LONG, 8, 8, 64, 4096, None),         # one slot: whole sequences
    ([5000], 4, 1, 128, 64, None),        # one sequence, two wavefronts to a chunk of two tiles
    ([8192], 80, 2, 128, 1024, None),     # two slices of query heads
    ([1, 2], 8, 2, 96, None, 4096),       # one tile each under a large bound
    ([0, 0, 0], 8, 2, 64, None, 512),     # nothing at all
    ([2500, 40], 48, 6, 128, 128, 2048),  # longer than the bound: cut at its slots
]


@pytest.mark.parametrize("i", range(len(CASES)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_every_partition_meets_the_oracle(i, dtype):
    import tritonops_amd as ta

    lens, Hq, Hkv, D, split, bound = CASES[i]
    lens = torch.tensor(lens, dtype=torch.int32)
    B, L = len(lens), max(int(lens.max()), bound or 1)
    q, k, v = randn((B, Hq, D), 1, dtype), randn((B, L, Hkv, D), 2, dtype), randn((B, L, Hkv, D), 3, dtype)
    seen = lens if bound is None or split is None else lens.clamp(max=-(-bound // split) * split)
    want = orc.flash_attn_decoding_torch(q, k, v, seen, faithful=False)
    qd, kd, vd, ld = q.cuda(), k.cuda(), v.cuda(), lens.cuda()
    n = -(-(bound or L) // 64) * B * Hq * (D + 1)
    poison = torch.full((n,), float("nan"), device="cuda")
    del poison
    got, lse = ta.flash_attention_decoding(qd, kd, vd, None, seq_lens=ld, split_tokens=split, max_seq_len=bound,
                                           return_lse=True)
    assert_close(got, want, TOL, "o")
    assert torch.equal(torch.isfinite(lse), (ld > 0)[:, None].expand(B, Hq))
    again = ta.flash_attention_decoding(qd, kd, vd, None, seq_lens=ld, split_tokens=split, max_seq_len=bound)
    assert torch.equal(got, again)


@pytest.mark.parametrize("lens,split", [([3000, 700], 64), ([5000], 64), (LONG[:1] * 8, 512), (LONG * 6, 2048)],
                         ids=["chunks", "wavefronts", "one_wavefront", "ranges"])
def test_nan_in_a_key_makes_its_heads_nan(lens, split):
    """One key row that holds NaN: the query heads of its kv-head are NaN however many
    chunks were merged, and nothing else is touched."""
    import tritonops_amd as ta

    B, L = len(lens), max(lens)
    q, k, v = randn((B, 8, 128), 1).cuda(), randn((B, L, 2, 128), 2).cuda(), randn((B, L, 2, 128), 3).cuda()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    want = ta.flash_attention_decoding(q, k, v, None, seq_lens=sl, split_tokens=split)
    k[0, 1777, 1, 5] = float("nan")
    got, lse = ta.flash_attention_decoding(q, k, v, None, seq_lens=sl, split_tokens=split, return_lse=True)
    assert got[0, 4:].isnan().all() and lse[0, 4:].isnan().all()
    got[0, 4:] = want[0, 4:]
    assert torch.equal(got, want)


@pytest.mark.parametrize("split_blocks", [1, 2, 5])
@pytest.mark.parametrize("D", [64, 96, 128])
def test_lists_of_few_chunks(D, split_blocks):
    """Chunks of a block list shared by several wavefronts, some of them without a tile."""
    import tritonops_amd as ta

    lens = torch.tensor([640, 65, 1], dtype=torch.int32)
    q, k, v = randn((3, 8, D), 1), randn((3, 640, 2, D), 2), randn((3, 640, 2, D), 3)
    idx = torch.tensor([[[0, 2, 5, 9, 7], [1, 9, 0, 0, 0]], [[0, 1, 0, 0, 0], [1, 0, 0, 0, 0]], [[0] * 5] * 2],
                       dtype=torch.int32)
    cnt = torch.tensor([[5, 2], [2, 1], [1, 0]], dtype=torch.int32)
    want = orc.block_sparse_decoding(q, k, v, lens, idx, cnt, include_last_block=True, faithful=False)
    got = ta.flash_attention_sparse_decoding(q.cuda(), k.cuda(), v.cuda(), None, seq_lens=lens.cuda(),
                                             block_indices=idx.cuda(), block_counts=cnt.cuda(),
                                             split_blocks=split_blocks)
    assert_close(got, want, TOL)


def _rows(lens, Hq, Hkv, D, room):
    B = len(lens)
    return (randn((B, Hq, D), 5).cuda(), randn((B, room, Hkv, D), 6).cuda(), randn((B, room, Hkv, D), 7).cuda(),
            torch.tensor(lens, dtype=torch.int32, device="cuda"))


@pytest.mark.parametrize("split", [None, 64, 512, 4096])
def test_a_row_does_not_depend_on_the_lengths_of_its_neighbours(split):
    """The same bits for a row whatever the other sequences of the batch hold, and (where
    the caller says how long a chunk is) alone."""
    import tritonops_amd as ta

    lens = [3000, 4095, 1, 700, 2049, 32]
    q, k, v, sl = _rows(lens, 32, 8, 128, 4096)
    o, lse = ta.flash_attention_decoding(q, k, v, None, seq_lens=sl, split_tokens=split, return_lse=True)
    for i in range(len(lens)):
        for others in (4096, 5, 0):
            ln = torch.full_like(sl, others)
            ln[i] = lens[i]
            o2, lse2 = ta.flash_attention_decoding(q, k, v, None, seq_lens=ln, split_tokens=split, return_lse=True)
            assert torch.equal(o2[i], o[i]) and torch.equal(lse2[i], lse[i]), (i, others)
        if split:
            one = slice(i, i + 1)
            o1, lse1 = ta.flash_attention_decoding(q[one], k[one], v[one], None, seq_lens=sl[one], split_tokens=split,
                                                   return_lse=True)
            assert torch.equal(o1[0], o[i]) and torch.equal(lse1[0], lse[i]), i


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("length", [4096, 3937, 33])
def test_bits_do_not_depend_on_the_number_of_wavefronts(D, length):
    """A launch of few chunks puts four wavefronts to a chunk, one of many chunks two or one
    (up to 2048 wavefronts are resident): chunks of 256 tokens and of four blocks, 8 kv-heads."""
    import tritonops_amd as ta

    q, k, v, sl = _rows([length], 32, 8, D, 4096)
    blocks = torch.arange(0, (length + 63) // 64, 2, dtype=torch.int32, device="cuda").expand(1, 8, -1)

    def dense(B):
        r = lambda t: t.expand(B, *t.shape[1:])
        return ta.flash_attention_decoding(r(q), r(k), r(v), None, seq_lens=r(sl).contiguous(), split_tokens=256,
                                           return_lse=True)

    def listed(B):
        r = lambda t: t.expand(B, *t.shape[1:])
        return ta.flash_attention_sparse_decoding(r(q), r(k), r(v), None, seq_lens=r(sl).contiguous(),
                                                  block_indices=r(blocks), split_blocks=4, return_lse=True)

    for call in (dense, listed):
        want = call(1)
        for B in (3, 8, 40):
            for got, w in zip(call(B), want):
                assert torch.equal(got, w.expand_as(got)), (call.__name__, B)


@pytest.mark.parametrize("split", [64, 256, 2048])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_values_that_are_not_finite_reach_the_result(value, split):
    """A value that is infinite or NaN under a key whose probability underflows is
    0 * inf = NaN, whether its chunk holds keys of weight too or is all underflow."""
    import tritonops_amd as ta

    q, k, v, sl = _rows([2000], 8, 2, 128, 2048)
    q.fill_(4.0)
    k.fill_(-4.0)
    k[0, 700:1000] = 4.0  # 522 binades above the others
    want = ta.flash_attention_decoding(q, k, v, None, seq_lens=sl, split_tokens=split)
    v[0, 10, 1, 5] = value
    got = ta.flash_attention_decoding(q, k, v, None, seq_lens=sl, split_tokens=split)
    assert got[0, 4:, 5].isnan().all()
    got[0, 4:, 5] = want[0, 4:, 5]
    assert torch.equal(got, want)
