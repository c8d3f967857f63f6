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


@pytest.mark.parametrize(
    "tokens,context,n_q,window,steps",
    [
        (1500, 0, 16, None, 6), (2048, 0, 16, None, 13), (1800, 0, 16, None, 9), (1024, 1000, 16, None, 8), (64, 0, 16, None, 2), (1500, 0, 8, None, 3), (2048, 0, 8, None, 7),
        (300, 2000, 8, None, 4), (2979, 0, 4, 128, 3), (4096, 0, 16, 128, 5), (2048, 0, 24, None, 11), (16, 4000, 8, None, 2), (4096, 28000, 16, None, 26),
    ],
)
def test_steps_of_a_block(tokens, context, n_q, window, steps):
    """Where the rounds of blocks take least, counted by hand for a few: 2,048 tokens of 16 heads in blocks of 11 steps are 221, nine in
    the fullest of 32 lots, so two rounds."""
    from cwm_amd.ops import build

    assert build.load("attention_talk_tile").cwm_talking_tile_steps(tokens, context, n_q, -1 if window is None else window - 1) == steps


def test_steps_against_a_plain_count():
    from cwm_amd.ops import build

    lib = build.load("attention_talk_tile")

    def plain(n, pos0, n_q, left):
        rows, room, best = 32 if n_q <= 16 else 16, 2 if n_q <= 8 else 1, None
        tiles = []
        for r0 in range(0, n, rows):
            first, last = pos0 + r0, pos0 + min(r0 + rows, n) - 1
            tiles.append(last // 32 - (max(first - left, 0) if left >= 0 else 0) // 32 + 1)
        for steps in range(2, 33):
            cuts = [-(-t // steps) for t in reversed(tiles)]
            blocks, lots = sum(cuts), [0] * 32
            for b, c in enumerate(cuts):
                for r in range(c):
                    lots[(r * len(tiles) + b) % 32] += 1
            fullest = max(lots) if blocks <= 896 * room else 0
            rounds = max(-(-blocks // (224 * room)), -(-fullest // (8 * room)))
            us = rounds * (7 + 3.7 * steps) * (1.0 if room == 1 or (blocks <= 192 and fullest <= 8) else 1.6)
            if best is None or us < best[0] * (1 - 1e-6):  # float32 in the library: what is level keeps the fewer steps
                best = (us, steps)
        return best[1]

    for n in (16, 33, 130, 500, 1023, 2048, 4096):
        for pos0 in (0, 77, 5000):
            for n_q in (8, 16, 24):
                for left in (-1, 0, 127, 1000):
                    assert lib.cwm_talking_tile_steps(n, pos0, n_q, left) == plain(n, pos0, n_q, left), (n, pos0, n_q, left)
