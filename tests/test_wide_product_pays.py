"""Which products of many rows are given to the wide kernel: points where both were timed, on either side of every line of the rule."""

from __future__ import annotations

import pytest

from cwm_amd.ops import build


# rows, columns, K, with the gated epilogue; (us, the library and the wide kernel)
@pytest.mark.parametrize("m,n,k,glu,takes", [
    (1040, 4096, 4096, 0, True),  # (46 / 39)
    (2296, 2048, 2048, 0, True),  # (27.5 / 21.7)
    (4096, 8192, 6144, 0, False),  # two full rounds of the library's largest tile (284 / 338)
    (384, 128, 1536, 0, False),  # small results, where the library cuts K (7.0 / 10.6)
    (450, 512, 3072, 0, False),  # (9.5 / 18.0)
    (600, 1024, 3072, 0, False),  # (16 / 20)
    (384, 128, 512, 0, True),  # and a K too short to cut
    (600, 512, 3072, 1, False),  # (16.6 / 18.7)
    (3000, 512, 14336, 0, False),  # a quarter of the chip idle and a long K (73 / 85)
    (2652, 512, 14336, 1, False),  # (73 / 82)
    (600, 4128, 14336, 1, False),  # (103 / 124)
    (512, 6144, 14336, 0, False),  # (115 / 134)
    (512, 5120, 21504, 0, True),  # cuts that cost more than they give (234 / 148)
    (300, 6144, 21504, 0, True),  # (178 / 136)
    (2048, 3072, 28672, 0, False),  # (276 / 362)
    (3538, 10304, 14336, 0, False),  # many full rounds (807 / 931)
    (3538, 10304, 8192, 0, False),  # (457 / 505)
    (1040, 4096, 14336, 0, True),  # too many small tiles to cut K, and large ones that fill little (148 / 135)
    (1040, 28672, 4096, 1, True),  # (255 / 238)
    (900, 5120, 21504, 1, True),  # (283 / 213)
    (8192, 10304, 512, 1, True),  # a short K (194 / 115)
    (2048, 16, 2048, 0, False),  # fewer columns than a tile (11.5 / 12.2)
])
def test_what_it_takes(m, n, k, glu, takes):
    assert bool(build.load("gemm_bf16_wide").cwm_gemm_bf16_wide_pays(m, n, k, 256, glu)) is takes
