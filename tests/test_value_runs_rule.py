"""Which steps write values a value block at a time: points where both ways were timed, on either side of every line of the rule."""

from __future__ import annotations

import pytest

from cwm_amd.ops import build


# tokens, sequences, query heads, key and value heads, head; (us, narrow writes and whole blocks)
@pytest.mark.parametrize("tokens,seqs,n_q,n_kv,head_dim,takes", [
    (2048, 1, 16, 4, 128, True),  # (13.4 / 12.3)
    (2048, 32, 32, 8, 128, True),  # (23.5 / 20.4)
    (2048, 2048, 32, 8, 128, False),  # a token a sequence (26.9 / 29.5)
    (2048, 186, 16, 4, 128, False),  # eleven in a row (14.1 / 15.5)
    (512, 1, 8, 8, 64, True),  # (6.0 / 5.5)
    (511, 1, 8, 8, 64, False),  # several blocks a token
    (64, 1, 2, 1, 64, False),  # few heads, one block a token at any number of tokens (4.3 / 4.5)
    (8192, 1, 8, 2, 128, False),  # (25.1 / 27.0)
    (8192, 1, 40, 8, 128, True),  # (69.7 / 59.2)
    (8192, 1, 28, 4, 128, False),  # (44.1 / 45.0)
])
def test_where_whole_blocks_are_written(tokens, seqs, n_q, n_kv, head_dim, takes):
    assert bool(build.load("rope_kv").cwm_value_runs_pay(tokens, seqs, n_q, n_kv, head_dim)) is takes
