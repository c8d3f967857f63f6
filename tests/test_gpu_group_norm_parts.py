"""The norm of parts of rows: parts of less than one lane's eight elements, of a team, a wavefront and several, beyond a block's
8,192, rows that start off a 16-byte boundary, sources of one and several partial sums."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("part,groups", [(1, 3), (5, 8), (8, 9), (64, 33), (264, 4), (512, 2), (520, 3), (2048, 1), (8192, 2), (8200, 1), (16391, 1)])
@pytest.mark.parametrize("n_rows,offset,dtype", [(1, 0, torch.float32), (3, 0, torch.bfloat16), (9, 1, torch.bfloat16), (9, 4, torch.float32)])
def test_against_float64(part, groups, n_rows, offset, dtype):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(part + n_rows)
    dim = part * groups
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = normal(n_rows, dim + 8).to(dtype)[:, offset : offset + dim]
    gate, h, weight = normal(n_rows, dim).bfloat16(), normal(n_rows, dim), normal(dim).to(dtype)
    partials = normal(3, n_rows, dim)

    def norm(v):
        v = v.reshape(n_rows, groups, part)
        return (v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-5)).reshape(n_rows, dim) * weight.double()

    # float32 sums of `part` squares, one value's silu and the residual's sum: a few units of 2^-24 for each of the logarithmic
    # and eight serial additions, relative to the value; bfloat16 results round once more (half a unit, 2^-9 of the binade's top)
    def close(got, want, terms):
        unit = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
        assert bool(((got.double() - want).abs() <= (unit + 2.0 ** -18) * terms + 1e-7).all())

    plain = norm(x.double())
    close(ops.group_rmsnorm(x, weight, groups, 1e-5, torch.float32), plain, plain.abs())
    gated = norm(x.double() * torch.nn.functional.silu(gate.double()))
    close(ops.group_rmsnorm(x, weight, groups, 1e-5, torch.bfloat16, gate=gate), gated, gated.abs())
    # the sum of partials may cancel: the error is of their size
    total = norm(partials.double().sum(0))
    scale = weight.double().abs() * (partials.double().abs().sum(0)).reshape(n_rows, groups, part).mul(
        torch.rsqrt(partials.double().sum(0).reshape(n_rows, groups, part).square().mean(-1, keepdim=True) + 1e-5)).reshape(n_rows, dim)
    copy, got = torch.empty(n_rows, dim, device=DEV, dtype=torch.bfloat16), h.clone()
    ops.group_rmsnorm(partials, weight, groups, 1e-5, torch.float32, out=got, accumulate=True, copy=copy)
    close(got, h.double() + total, h.double().abs() + scale)
    assert torch.equal(copy, got.bfloat16())
    inplace = x.clone()
    ops.group_rmsnorm(inplace, weight, groups, 1e-5, dtype, out=inplace)
    close(inplace, plain, plain.abs())


def test_a_row_alone_and_off_its_boundary_gives_the_same_bits():
    from cwm_amd import ops

    x = torch.randn(7, 4096 + 8, device=DEV)
    weight = torch.rand(4096, device=DEV)
    whole = ops.group_rmsnorm(x[:, :4096], weight, 4, 1e-5, torch.float32)
    moved = torch.empty(7, 4096 + 9, device=DEV)[:, 3 : 3 + 4096]
    moved.copy_(x[:, :4096])
    assert torch.equal(ops.group_rmsnorm(moved, weight, 4, 1e-5, torch.float32), whole)
    assert torch.equal(ops.group_rmsnorm(x[2:3, :4096], weight, 4, 1e-5, torch.float32), whole[2:3])
