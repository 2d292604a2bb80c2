"""Where grad_x of many tiles is divided over the vocabulary: the rule's edges."""

import pytest

from tritonops_amd import _lib


@pytest.mark.parametrize("tokens,dim,vocab,used", [
    (2876, 4096, 128256, True),
    (4100, 2560, 50257, True),
    (2876, 4096, 32000, False),     # small vocabulary
    (3072, 4096, 128256, False),    # a multiple of 512
    (3001, 4096, 128256, False),    # fills one up
    (6200, 2560, 128256, False),    # 250 of 256 places
    (1800, 4096, 128256, False),    # 256 narrow tiles
    (3900, 3072, 50257, False), (3851, 3072, 50257, False), (5959, 2048, 44032, False), (4646, 2560, 40000, False),  # one round of tiles of 192
    (3353, 3072, 50257, False), (4900, 2048, 50257, False),                                          # of 160
    (2898, 2048, 44032, False), (1929, 3072, 64000, False),                                          # of 192 x 128
    (2574, 3072, 40000, False), (3200, 2560, 48000, False), (6430, 2560, 40000, False),              # of 128 x 256, and two of them
    (6448, 2048, 42000, True), (1292, 4096, 50257, True), (2876, 2048, 50257, True), (1585, 4096, 42000, True),
    (0, 4096, 128256, False),
    (2876, 0, 128256, False),
])
def test_which_results_are_divided(tokens, dim, vocab, used):
    lib = _lib.load()
    s = lib.mi_xent_grad_x_uneven_splits(tokens, dim, vocab, 256)
    assert (s > 0) == used
    if used:  # the partial sums are no larger than the 16-bit dlogits
        assert s * tokens * dim * 4 <= tokens * vocab * 2
        assert lib.mi_xent_grad_x_workspace_bytes(tokens, dim, s) > 0


def test_partial_sums_are_no_larger_than_the_dlogits():
    """As the workspace holds them, in whole tiles of 256 x 256: token counts and columns a little past a tile among
    them (1548 x 3136 x 50257 had 8 ranges, 1.23 times the dlogits)."""
    lib = _lib.load()
    some = 0
    for tokens in (1292, 1548, 1793, 2049, 2876, 4100, 5121, 7777):
        for dim in (1032, 2048, 2312, 2568, 3136, 4096, 5128):
            for vocab in (40000, 50257, 128256):
                s = lib.mi_xent_grad_x_uneven_splits(tokens, dim, vocab, 256)
                some += s > 1
                assert lib.mi_xent_grad_x_workspace_bytes(tokens, dim, s) <= 2 * tokens * vocab, (tokens, dim, vocab, s)
    assert some > 20
