"""Which kernel a product of few rows goes to: the rule and the kernel agree on where K is split (host arithmetic only)."""

from __future__ import annotations

import pytest
import torch

from cwm_amd import ops


def matrices(m, n, k):
    """Operands that nothing reads, and a stand-in for the streaming copy."""
    return torch.empty((m, k), dtype=torch.bfloat16), torch.empty((n, k), dtype=torch.bfloat16), torch.empty(0)


@pytest.mark.parametrize("m", [9, 16, 17, 24, 32])
@pytest.mark.parametrize("k", [2048, 2112, 3072, 3136, 6144, 6208])
def test_the_limit_is_that_of_a_split_k(m, k):
    """2^25 entries for products that split K, 2^27 for those that do not: the plain product of 17 to 32 rows splits from a K
    of 2,048, with an epilogue from 3,072, of up to 16 rows both from 6,144."""
    x, w, copy = matrices(m, (1 << 25) // k + 16 & -16, k)
    for fused, most in ((False, 6144 if m <= 16 else 2048), (True, 6144 if m <= 16 else 3072)):
        assert ops.stream_unsplit_k(m, fused) == most
        assert ops._prefers_tile(x, w, None, copy, fused) == (k > most)
    x, w, copy = matrices(m, (1 << 27) // k + 16 & -16, k)
    assert ops._prefers_tile(x, w, None, copy, False) and ops._prefers_tile(x, w, None, copy, True)


def test_a_head_of_24_rows_is_one_launch_of_whole_tiles():
    x, w, copy = matrices(24, 32768, 3072)
    assert ops._prefers_tile(x, w, None, copy)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("m", [9, 16, 17, 32])
def test_a_copy_decides_only_for_larger_matrices(m, fused):
    """Below 2^22 entries (2^24 up to 8 rows) the kernel, and with it the order of the sums, is the same with a copy and without."""
    for n, k in ((208, 128), (2048, 64), (256, 512), (512, 64), (2032, 2048), (512, 8128), (32768, 64), (16384, 192), (65520, 64), (16, 8192)):
        x, w, copy = matrices(m, n, k)
        assert n * k < 1 << 22
        assert ops._prefers_tile(x, w, None, copy, fused) == ops._prefers_tile(x, w, None, None, fused) == (n * k < 1 << 15 or n >= 20480), (n, k)
        x, w, copy = matrices(8, 8 * n, k)
        assert not ops._prefers_tile(x, w, None, copy, fused) and ops._prefers_tile(x, w, None, None, fused) == (8 * n * k >= 1 << 24), (n, k)
    x, w, copy = matrices(m, 2048, 2048)
    assert not ops._prefers_tile(x, w, None, copy, fused) and ops._prefers_tile(x, w, None, None, fused)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("m,n,k,tiled", [
    (9, 32768, 512, True), (32, 32768, 512, True), (16, 128256, 512, True), (17, 20480, 960, True), (9, 20464, 960, False), (9, 16384, 256, False),
    (16, 32768, 1024, True), (17, 32768, 1024, False), (16, 32752, 1024, False), (16, 32768, 1088, False), (8, 32768, 512, False), (9, 20480, 1024, False),
])
def test_wide_results_of_a_short_k_are_tiled(m, n, k, tiled, fused):
    x, w, copy = matrices(m, n, k)
    assert ops._prefers_tile(x, w, None, copy, fused) == tiled
