"""The bfloat16 product of many rows whose tiles pass through LDS (csrc/gemm_bf16_wide.hip), against float64."""

import pytest
import torch

from cwm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = 9  # of the kernel's list; the last three have no gated epilogue


def _operands(m, n, k, pad):
    gen = torch.Generator().manual_seed(m * 7919 + n * 31 + k)
    x = torch.randn(m, k + pad, generator=gen).bfloat16().to(DEV)[:, :k]
    w = (torch.randn(n, k + pad, generator=gen) * k**-0.5).bfloat16().to(DEV)[:, :k]
    return x, w


# one step of K, fewer steps than buffers, many; a lone row and column group, edges of the 64- to 256-high tiles, ragged ones; fewer
# blocks than XCDs, blocks that walk several tiles (their loads run on across tiles), a block a tile
@pytest.mark.parametrize("units", [1, 3, 11, 256])
@pytest.mark.parametrize("m,n,k,pad", [(1, 16, 64, 0), (64, 128, 128, 8), (130, 208, 192, 0), (257, 528, 320, 64), (513, 1040, 1024, 0)])
def test_every_tile_against_float64(m, n, k, pad, units):
    x, w = _operands(m, n, k, pad)
    exact = x.double() @ w.double().t()
    most = x.double().abs() @ w.double().abs().t()  # a float32 sum of K products is off by at most K * 2^-24 of this
    bound = k * 2.0**-24 * most
    first = ops.gemm_bf16_wide(x, w, torch.float32, units=units)
    assert ((first.double() - exact).abs() <= bound).all()
    gated = ops.silu_mul(ops.gemm_bf16_wide(x, w, units=units), grouped=True)
    for tile in range(TILES):
        got = ops.gemm_bf16_wide(x, w, torch.float32, units=units, tile=tile)
        assert torch.equal(got, first)  # a sum's order does not depend on the tile
        assert torch.equal(ops.gemm_bf16_wide(x, w, units=units, tile=tile), first.bfloat16())
        if tile < TILES - 3:
            assert torch.equal(ops.gemm_bf16_wide(x, w, glu=True, units=units, tile=tile), gated)


@pytest.mark.parametrize("m,n,k", [(300, 1024, 512), (1040, 4096, 512), (777, 6144, 1024)])
def test_the_products_that_go_there(m, n, k):
    """The entry point's result where the rule picks this kernel, beside the library's."""
    x, w = _operands(m, n, k, 0)
    assert ops._prefers_wide(x, w)
    got = ops.gemm_bf16(x, w)
    assert torch.equal(got, ops.gemm_bf16_wide(x, w))
    exact = x.double() @ w.double().t()
    # the float32 sum's error, and the rounding to bfloat16's eight significant bits: 2^-8 of the sum
    bound = (1 + 2.0**-8) * k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 2.0**-8 * exact.abs()
    assert ((got.double() - exact).abs() <= bound).all()
    assert ((torch.mm(x, w.t()).double() - exact).abs() <= bound).all()
    # a row's bits are its own
    assert torch.equal(ops.gemm_bf16_wide(x[5:200].contiguous(), w), got[5:200])


def test_what_it_refuses():
    x, w = _operands(130, 208, 192, 0)
    for bad in ((x[:, :100], w[:, :100]), (x, w[:100]), (x.float(), w.float())):
        with pytest.raises(ops.KernelError):
            ops.gemm_bf16_wide(*bad)
        assert not ops._wide_takes(*bad)
    with pytest.raises(ops.KernelError):
        ops.gemm_bf16_wide(x, w, tile=TILES)
    with pytest.raises(ops.KernelError):
        ops.gemm_bf16_wide(x, w, glu=True, tile=TILES - 1)


# thousands of rows: several bands of row tiles, blocks that walk several tiles each, with and without ragged ends
@pytest.mark.parametrize("m,n,k", [(2296, 2048, 2048), (2652, 10304, 576), (8193, 2064, 192)])
def test_thousands_of_rows(m, n, k):
    x, w = _operands(m, n, k, 0)
    got = ops.gemm_bf16_wide(x, w, torch.float32)
    assert torch.equal(ops.gemm_bf16_wide(x, w), got.bfloat16())
    assert torch.equal(ops.gemm_bf16_wide(x, w, glu=True), ops.silu_mul(got.bfloat16(), grouped=True))
    for lo in range(0, m, 1024):
        exact = x[lo : lo + 1024].double() @ w.double().t()
        # a float32 sum of K products is off by at most K * 2^-24 of the sum of their sizes
        bound = k * 2.0**-24 * (x[lo : lo + 1024].double().abs() @ w.double().abs().t())
        assert ((got[lo : lo + 1024].double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("tile", range(TILES))
def test_infinities_and_nan(tile):
    """A row or column of W with one gives what float64 gives there, and the bits of all others stay."""
    m, n, k = 300, 288, 192
    x, w = _operands(m, n, k, 0)
    clean = ops.gemm_bf16_wide(x, w, torch.float32, tile=tile)
    x[3, 7], x[130, 0], x[299, k - 1], w[40, 5], w[287, 100] = float("inf"), float("nan"), -float("inf"), float("inf"), float("nan")
    got = ops.gemm_bf16_wide(x, w, torch.float32, tile=tile)
    exact = x.double() @ w.double().t()
    rows, columns = torch.ones(m, dtype=torch.bool, device=DEV), torch.ones(n, dtype=torch.bool, device=DEV)
    rows[[3, 130, 299]], columns[[40, 287]] = False, False
    assert torch.equal(got[rows][:, columns], clean[rows][:, columns])
    rest = ~(rows[:, None] & columns[None, :])
    assert not exact[rest].isfinite().any()
    assert torch.equal(got[rest].double().nan_to_num(2.0, 1.0, -1.0), exact[rest].nan_to_num(2.0, 1.0, -1.0))
    if tile < TILES - 3:
        gate, up = (got.bfloat16().float().view(m, n // 16, 2, 8)[:, :, i].reshape(m, n // 2).double() for i in range(2))
        want = gate / (1.0 + torch.exp(-gate)) * up
        gated = ops.gemm_bf16_wide(x, w, glu=True, tile=tile).double()
        finite = want.isfinite()
        assert torch.equal(gated[~finite].nan_to_num(2.0, 1.0, -1.0), want[~finite].nan_to_num(2.0, 1.0, -1.0))
        # expf, the quotient and the product in float32 are off by far less than the rounding to bfloat16, 2^-9 of the value
        assert ((gated[finite] - want[finite]).abs() <= 2.0**-8 * want[finite].abs() + 1e-30).all()
