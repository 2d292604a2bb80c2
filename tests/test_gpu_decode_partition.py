"""How a decoding launch divides its work: chunks of one sequence, tile ranges that
run across sequences (csrc/decode.hip, decode_splitkv_kernel), one, two or four
wavefronts to a chunk, and slots of the workspace that stay empty.  The workspace
comes out of memory that held NaN, so a slot that is used without having been
written shows."""
import pytest
import torch

from oracle import attention_oracle as orc
from tests.util import assert_close, randn

pytestmark = pytest.mark.gpu
TOL = 2e-2

LONG = [3000, 0, 1, 31, 32, 33, 4095, 2048, 0, 700]
CASES = [
    # lens, Hq, Hkv, D, split_tokens, max_seq_len
    (LONG, 32, 8, 128, 64, None),         # many slots: equal chunks of four tiles and more
    (LONG * 6, 32, 8, 128, 2048, None),   # two slots to a sequence: ranges, bounded by the slots
    (LONG * 6, 64, 32, 96, 512, None),    # ranges, several rounds' worth of sequences
    (LONG * 13, 16, 16, 64, 256, None),   # 130 sequences: the search steps over the batch
    (LONG, 8, 8, 64, 4096, None),         # one slot: whole sequences
    ([5000], 4, 1, 128, 64, None),        # one sequence, 4 wavefronts to a chunk
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
