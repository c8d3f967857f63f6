"""The rows that the persistent blocks of the routed experts' products read lie inside the list, whether its tiles in use are counted
or not (index arithmetic on the host; the kernel uses the same functions)."""

from __future__ import annotations

import ctypes

import pytest

from cwm_amd.ops import build


@pytest.mark.parametrize("n_tiles", range(8, 41))
@pytest.mark.parametrize("col_blocks", [1, 3])
@pytest.mark.parametrize("quarters", [0, 1])
def test_every_row_lies_in_the_list(n_tiles, col_blocks, quarters):
    lib, first = build.load("routed"), ctypes.c_int()
    tiles, rows = -(-n_tiles // 8) * col_blocks * (4 if quarters else 1), 64 if quarters else 128
    read = set()
    for tile in range(tiles):
        for row in range(rows):
            past = lib.cwm_grouped_loop_rows(n_tiles, col_blocks, tile, quarters, row, ctypes.byref(first))
            assert 0 <= past < rows and first.value + past < 16 * n_tiles, (tile, row, first.value, past)
            read.add(first.value + past)
    assert read == set(range(16 * n_tiles))
