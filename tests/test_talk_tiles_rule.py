"""Which portions of a prompt make no table of scores: sizes on both sides of every line, each as it was timed."""

from __future__ import annotations

import pytest

from cwm_amd.ops import mixing

HEADS = {  # query heads, key/value heads, head size, blocks of the tiles' kernels for 32 rows
    "8 on 8": (8, 8, 128, 8), "16 on 8": (16, 8, 128, 8), "16 on 4": (16, 4, 128, 4), "8 on 1": (8, 1, 128, 2), "24 on 3": (24, 3, 128, 6),
    "32 on 8": (32, 8, 128, 8), "8 on 4 of 64": (8, 4, 64, 4), "1 on 1": (1, 1, 128, 1), "20 on 4": (20, 4, 128, 8),
}


@pytest.mark.parametrize("heads", HEADS)
def test_blocks_of_a_tile(heads):
    n_q, n_kv, hd, groups = HEADS[heads]
    assert mixing._talk_tile_groups(n_q, n_kv, hd) == groups


@pytest.mark.parametrize(
    "heads,tokens,keys,tiles",
    [
        ("16 on 8", 15, 2000, False), ("16 on 8", 16, 16, True), ("16 on 8", 16, 30016, True), ("16 on 8", 1500, 1500, True), ("16 on 8", 128, 8192, True),
        ("16 on 8", 128, 8193, False), ("16 on 8", 1024, 31024, False), ("8 on 8", 128, 4096, True), ("8 on 8", 128, 6128, False), ("8 on 8", 512, 6512, True),
        ("32 on 8", 1024, 13024, True), ("32 on 8", 1024, 31024, False), ("20 on 4", 1024, 31024, False),
        ("24 on 3", 16, 4016, False), ("24 on 3", 22, 4022, True), ("24 on 3", 1024, 13024, False),
        ("16 on 4", 16, 4016, False), ("16 on 4", 63, 1063, False), ("16 on 4", 64, 1064, True), ("16 on 4", 64, 64, False), ("16 on 4", 128, 4128, False),
        ("16 on 4", 512, 4512, True), ("8 on 4 of 64", 128, 4128, True), ("8 on 4 of 64", 128, 12128, False),
        ("8 on 1", 32, 4032, False), ("8 on 1", 64, 4064, True), ("8 on 1", 128, 128, False), ("8 on 1", 512, 512, False), ("8 on 1", 2048, 3048, True),
        ("1 on 1", 64, 4064, False), ("1 on 1", 2048, 2048, False),
    ],
)
def test_portions_without_a_table(heads, tokens, keys, tiles):
    n_q, n_kv, hd, groups = HEADS[heads]
    assert mixing.talk_tiles_take(tokens, keys, groups, n_q, n_kv, hd) == tiles


def test_heads_without_kernels():
    for n_q, n_kv, hd in [(33, 3, 64), (36, 4, 128), (18, 9, 128), (16, 8, 96), (12, 5, 128)]:
        assert mixing._talk_tile_groups(n_q, n_kv, hd) == 0
        assert not mixing.talk_tiles_take(1500, 1500, 0, n_q, n_kv, hd)
