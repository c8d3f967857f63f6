"""Tokens of a block of the token input's matrix kernel: its rows fit the LDS at every width, and the lines lie where they were timed."""

from __future__ import annotations

import pytest

from cwm_amd.ops import build

LDS = 160 * 1024 - 64  # what a kernel with its own 64 bytes beside may ask for


@pytest.mark.parametrize("n_tokens", [256, 1024, 1025, 2048, 2049, 4096, 4097, 6144, 6145, 100000])
@pytest.mark.parametrize("side", [32, 64, 96, 128])
def test_rows_fit(n_tokens, side):
    lib = build.load("token_side")
    for dim in range(64, 4097, 64):
        tok = lib.cwm_token_side_tile_tokens(n_tokens, dim, side)
        assert tok in (4, 8, 16) and 0 < lib.cwm_token_side_tile_lds(tok, dim) <= LDS, (dim, tok)


@pytest.mark.parametrize(
    "n_tokens,dim,side,tok",
    [(256, 2048, 64, 8), (2048, 4096, 64, 8), (2049, 64, 64, 16), (4096, 4096, 128, 16), (300, 3520, 64, 4), (1024, 4096, 64, 4), (1025, 4096, 64, 8),
     (300, 3456, 64, 8), (4097, 2048, 32, 8), (6144, 2048, 32, 8), (6145, 2048, 32, 16), (4096, 2048, 32, 16), (5000, 1024, 32, 16), (5000, 2048, 64, 16)],
)
def test_lines(n_tokens, dim, side, tok):
    assert build.load("token_side").cwm_token_side_tile_tokens(n_tokens, dim, side) == tok
