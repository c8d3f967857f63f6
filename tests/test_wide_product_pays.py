"""Which products of many rows are given to the wide kernel, on either side of the lines of its rule."""

from __future__ import annotations

import pytest

from cwm_amd.ops import build


# rows, columns, K, with the gated epilogue; (us, the library and the wide kernel)
@pytest.mark.parametrize("m,n,k,glu,takes", [
    (1040, 4096, 4096, 0, True),  # the library's large tiles leave a quarter of the chip idle (46 / 39)
    (2296, 2048, 2048, 0, True),  # (27.5 / 21.7)
    (1040, 28672, 4096, 1, True),  # the costs of both kernels' tiles (249 / 227)
    (2048, 28672, 4096, 1, False),  # (382 / 395)
    (4096, 8192, 6144, 0, False),  # two full rounds of the library's largest tile (284 / 338)
    (130, 512, 3072, 0, True),  # a few hundredths of the chip: a K that is short enough (24 / 19)
    (130, 512, 6144, 0, False),  # and one that the library cuts (25 / 35)
    (2048, 16, 2048, 0, False),  # fewer columns than a tile (11.5 / 12.2)
    (2048, 2056, 2048, 0, False),  # sizes that the kernel does not take
    (2048, 2048, 2080, 0, False),
])
def test_what_it_takes(m, n, k, glu, takes):
    assert bool(build.load("gemm_bf16_wide").cwm_gemm_bf16_wide_pays(m, n, k, 256, glu)) is takes
