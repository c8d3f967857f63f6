"""Which bfloat16 rows the matrix memory's blocks take on the bfloat16 instruction: those of whole pieces of 16 bytes."""

from __future__ import annotations

import ctypes

import pytest

from cwm_amd.ops import build


@pytest.mark.parametrize("heads,d,e,extra,tiles", [
    (16, 128, 128, 0, True), (2, 8, 8, 0, True), (3, 32, 24, 0, True), (6, 100, 60, 0, False), (4, 64, 60, 0, False), (4, 100, 64, 0, False),
    (2, 6, 33, 0, False), (16, 128, 128, 4, False), (16, 128, 128, 8, True), (2, 4, 4, 0, False),
])
def test_whole_pieces(heads, d, e, extra, tiles):
    width = heads * (2 * d + 2 * e) + extra
    took = build.load("matrix_memory").cwm_matrix_memory_tiles(ctypes.c_long(width), 0, heads * d, 2 * heads * d, d, e)
    assert bool(took) == tiles
