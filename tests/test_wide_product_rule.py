"""Which products of many rows the wide kernel takes: what it refuses goes to the library, as any operand did before there was such a kernel."""

from __future__ import annotations

import pytest
import torch

from cwm_amd import ops

M, N, K = 300, 1024, 512


def _operands(device):
    gen = torch.Generator().manual_seed(1)
    x, w = torch.randn(M, K + 8, generator=gen).bfloat16().to(device), (torch.randn(N, K + 8, generator=gen) * K**-0.5).bfloat16().to(device)
    return x, w


def _overlapping(x, w):
    """Pairs with rows that repeat or overlap: one row for all, and windows that move on by eight elements."""
    flat_x, flat_w = x.reshape(-1), w.reshape(-1)
    yield x[:1, :K].expand(M, K), w[:, :K]
    yield x[:, :K], w[:1, :K].expand(N, K)
    yield flat_x.as_strided((M, K), (8, 1)), w[:, :K]
    yield x[:, :K], flat_w.as_strided((N, K), (K - 8, 1))


def test_rows_that_overlap_are_not_taken():
    x, w = _operands("cpu")
    assert ops._wide_takes(x[:, :K], w[:, :K])
    assert ops._wide_takes(x[:1, :K], w[:, :K])  # of a lone row the stride says nothing
    assert not any(ops._wide_takes(*pair) for pair in _overlapping(x, w))


@pytest.mark.gpu
def test_rows_that_overlap_go_to_the_library():
    x, w = _operands("cuda:0")
    assert ops._prefers_wide(x[:, :K], w[:, :K])
    for a, b in _overlapping(x, w):
        assert torch.equal(ops.gemm_bf16(a, b), torch.mm(a, b.t()))
        assert torch.equal(ops.gate_up_silu(a, b, None, True), ops.silu_mul(torch.mm(a, b.t()), grouped=True))


def test_rows_that_overlap_stay_with_the_tiled_kernels_check():
    """Up to its number of rows the tiled kernel has always been asked first, and refuses such operands."""
    x, w = _operands("cpu")
    assert all(ops._tile_takes(a[:100], b) for a, b in _overlapping(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [40, 100, 200])
def test_few_rows_that_overlap_are_refused(rows):
    x, w = _operands("cuda:0")
    for a, b in _overlapping(x, w):
        with pytest.raises(ops.KernelError):
            ops.gemm_bf16(a[:rows], b)


def test_float32_results_of_a_long_k_are_not_the_wide_kernels():
    assert ops._wide_keeps_sums(1500, 4096, 1024) and ops._wide_keeps_sums(1500, 4096, 2048)
    for m, n, k in ((130, 512, 2048), (2652, 28672, 2048), (1500, 4096, 2112), (600, 1024, 21504)):
        assert not ops._wide_keeps_sums(m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(900, 4096, 21504), (777, 4096, 6144), (1040, 2048, 512)])
def test_float32_results_are_as_near_as_the_librarys(m, n, k):
    gen = torch.Generator().manual_seed(m)
    x, w = torch.randn(m, k, generator=gen).bfloat16().to("cuda:0"), (torch.randn(n, k, generator=gen) * k**-0.5).bfloat16().to("cuda:0")
    assert ops._prefers_wide(x, w)
    exact = x.double() @ w.double().t()
    off = lambda y: ((y.double() - exact).norm() / exact.norm()).item()  # noqa: E731
    # the same sums, or the library's own; a different order of terms of equal length would differ by about a fiftieth
    assert off(ops.gemm_bf16(x, w, out_dtype=torch.float32)) <= 1.02 * off(torch.mm(x, w.t(), out_dtype=torch.float32))
