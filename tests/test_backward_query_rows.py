"""How many queries an item of the backward's dQ launch has: the rule's edges, and launches of
which it was measured that the other form is slower."""

import pytest

from tritonops_amd import _lib


@pytest.mark.parametrize("max_seqlen,batch,heads,causal,rows", [
    (1000, 1, 16, 1, 128), (129, 1, 1, 1, 128), (512, 8, 8, 0, 128),     # one round
    (4096, 1, 8, 1, 128), (4096, 1, 8, 0, 128),                          # one round exactly
    (4096, 1, 9, 0, 256),                                                # no mask: no second round
    (128, 8, 4, 1, 256), (60, 64, 2, 1, 256), (100, 64, 4, 1, 256), (1, 1, 1, 1, 256),   # items of 256 rows are no longer
    (2048, 1, 32, 1, 128), (4096, 1, 16, 1, 128), (8192, 1, 8, 1, 128), (2400, 1, 16, 1, 128), (1354, 3, 8, 1, 128),  # long chains
    (256, 64, 4, 1, 256), (256, 16, 16, 1, 256), (384, 24, 4, 1, 256), (130, 6, 32, 1, 256),                     # short ones
    (700, 40, 2, 1, 256), (926, 64, 1, 1, 256), (1342, 40, 1, 1, 128), (1384, 10, 4, 1, 128), (855, 4, 16, 1, 128),     # many sequences
    (512, 8, 16, 1, 256), (810, 32, 2, 1, 256), (954, 2, 32, 1, 256),
    (4096, 1, 17, 1, 256), (2731, 5, 32, 1, 256),                        # more than two rounds
    (0, 1, 1, 1, 256),
])
def test_rows(max_seqlen, batch, heads, causal, rows):
    lib = _lib.load()
    assert lib.mi_attn_bwd_query_rows(max_seqlen, batch, heads, causal, 256) == rows
