"""The blocks of the float32 product in parts (csrc/gemm_f32.hip): every one gives the same bits, whatever its height and width."""

import pytest
import torch

from cwm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BLOCKS = 7  # of the kernel's list


# a lone step of K and fewer than the buffers hold, a turn of the sums' sign and more; rows and columns at the edges of 32 to 256 and
# of 64 and 128; results whose rows end off a 16-byte boundary; operands whose rows lie apart
@pytest.mark.parametrize("m,n,k,pad", [(1, 1, 32, 0), (33, 64, 96, 4), (64, 130, 160, 0), (257, 129, 288, 8), (300, 520, 1056, 0)])
def test_every_block_gives_the_same_bits(m, n, k, pad):
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k + pad, generator=gen).to(DEV)[:, :k]
    w = torch.randn(n, k + pad, generator=gen).to(DEV)[:, :k]
    b = torch.randn(n, generator=gen).to(DEV)
    # the rows and columns of a value beyond the parts are left to float32 operands, and no other
    far_x, far_w = x.clone(), w.clone()
    far_x[m // 2, 3], far_w[n // 3, 7] = 1e20, -3e15
    exact = x.double() @ w.double().t() + b.double()
    # as for the kernel as a whole: a product is off by less than 2^-23 of itself, each of the 6 k / 32 sums by 2^-24 of the running one
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0**-23 + (0.2 * k + 2) * 2.0**-24 * (k**0.5 + 4)
    first = ops.gemm_f32_parts(x, w, b)
    far = ops.gemm_f32_parts(far_x, far_w, b)
    assert ((first.double() - exact).abs() <= bound).all()
    for block in range(BLOCKS):
        assert torch.equal(ops.gemm_f32_parts(x, w, b, block=block), first)
        assert torch.equal(ops.gemm_f32_parts(x, w, b, torch.bfloat16, block=block), first.bfloat16())
        assert torch.equal(ops.gemm_f32_parts(far_x, far_w, b, block=block), far)
    kept = torch.ones(m, n, dtype=torch.bool, device=DEV)
    kept[m // 2], kept[:, n // 3] = False, False
    assert torch.equal(far[kept], first[kept])
    assert torch.allclose(far.double(), far_x.double() @ far_w.double().t() + b.double(), rtol=1e-5, atol=0.01)


def test_what_it_refuses():
    x, w = torch.randn(40, 64, device=DEV), torch.randn(50, 64, device=DEV)
    for bad in ((x[:, :40], w[:, :40]), (x.bfloat16(), w), (x.t(), w[:, :40])):
        with pytest.raises(ops.KernelError):
            ops.gemm_f32_parts(*bad)
    with pytest.raises(ops.KernelError):
        ops.gemm_f32_parts(x, w, block=BLOCKS)


@pytest.mark.parametrize("rows", [1, 5])
def test_weights_whose_rows_lie_far_apart(rows):
    """Rows 32 MB apart and more are no other product: the bits of the same rows side by side."""
    apart = 1 << 23
    x, far = torch.randn(40, 96, device=DEV), torch.empty((rows - 1) * apart + 96, device=DEV).as_strided((rows, 96), (apart, 1))
    far.copy_(torch.randn(rows, 96, device=DEV))
    assert ops._f32_parts_takes(x, far)
    assert torch.equal(ops.gemm_f32(x, far), ops.gemm_f32(x, far.contiguous()))


# one to eight steps of K, of which half fit the shorter of two forms; rows at the edges of the 32 of a block and of a tile of 16, columns at the edges of 64; operands whose rows lie apart
@pytest.mark.parametrize("m", [1, 15, 17, 32, 33, 100])
@pytest.mark.parametrize("n,k,pad", [(1, 32, 0), (64, 64, 4), (70, 96, 0), (200, 128, 8), (64, 160, 0), (130, 256, 4)])
def test_one_launch_gives_the_same_bits(m, n, k, pad):
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k + pad, generator=gen).to(DEV)[:, :k]
    w = torch.randn(n, k + pad, generator=gen).to(DEV)[:, :k]
    b = torch.randn(n, generator=gen).to(DEV)
    assert torch.equal(ops.gemm_f32_parts(x, w, b, block=-2), ops.gemm_f32_parts(x, w, b))
    assert torch.equal(ops.gemm_f32_parts(x, w, None, torch.bfloat16, block=-2), ops.gemm_f32_parts(x, w, None, torch.bfloat16))
    # values beyond the parts, in rows and steps that different wavefronts take apart; a NaN, which stays in its row and column
    for row, column, value in ((m - 1, k - 1, 1e20), (m // 2, 3, float("inf")), (0, k // 2, float("nan"))):
        far_x, far_w = x.clone(), w.clone()
        far_x[row, column] = far_w[n // 3, k - 1 - column] = value
        got, want = (ops.gemm_f32_parts(far_x, far_w, b, block=block) for block in (-2, 0))
        assert torch.equal(got.nan_to_num(3.0), want.nan_to_num(3.0)) and torch.equal(got.isnan(), want.isnan())


def test_what_one_launch_refuses():
    x, w = torch.randn(40, 288, device=DEV), torch.randn(50, 288, device=DEV)
    for block in (-2, -3, -4):
        with pytest.raises(ops.KernelError):
            ops.gemm_f32_parts(x, w, block=block)
