"""Experts' weights in operand tiles: the bits of the row-major form, for every kernel that a number of rows an expert goes to,
last blocks of one to eight row tiles, and sizes that leave a block's columns or a wavefront's without work."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tokens,experts,top", [(1, 4, 1), (3, 16, 4), (40, 16, 4), (100, 3, 2), (300, 4, 2), (520, 2, 1), (1030, 5, 3)])
@pytest.mark.parametrize("dim,hidden", [(64, 64), (192, 320), (1024, 128)])
def test_both_forms_give_the_same_bits(tokens, experts, top, dim, hidden):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(tokens + dim)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV).bfloat16()  # noqa: E731
    x, gate, up, down = normal(tokens, dim), normal(experts, hidden, dim), normal(experts, hidden, dim), normal(experts, dim, hidden)
    chosen = (torch.rand((tokens, experts), generator=g, device=DEV) + torch.arange(experts, device=DEV) / experts).argsort(-1)[:, :top].int().contiguous()
    groups = ops.group_by_expert(chosen, experts)
    pairs = groups.pair_row.long()
    rows = ops.grouped_gate_up(x, groups, gate, up)
    tiled = ops.grouped_gate_up(x, groups, ops.expert_tiles(gate), ops.expert_tiles(up))
    assert torch.equal(rows[pairs], tiled[pairs])
    off = torch.empty(tokens * dim + 8, dtype=torch.bfloat16, device=DEV)[1 : 1 + tokens * dim].view(tokens, dim)
    off.copy_(x)
    assert torch.equal(ops.grouped_gate_up(off, groups, ops.expert_tiles(gate), ops.expert_tiles(up))[pairs], tiled[pairs])
    want, got = ops.grouped_linear(rows, groups, down)[pairs], ops.grouped_linear(rows, groups, ops.expert_tiles(down))[pairs]
    assert torch.equal(want, got)
    # every pair's row against float64: sums of `hidden` products of float32, a few units of 2^-24 of their size
    picked, expert = rows[pairs].double(), chosen.flatten().long()
    exact = torch.stack([down[e].double() @ row for e, row in zip(expert[:64].tolist(), picked[:64])])
    size = torch.stack([down[e].double().abs() @ row.abs() for e, row in zip(expert[:64].tolist(), picked[:64])])
    assert bool(((got[:64].double() - exact).abs() <= 2.0 ** -18 * size + 1e-30).all())


def test_what_has_no_operand_tiles():
    from cwm_amd import ops

    for shape, dtype in (((2, 24, 64), torch.bfloat16), ((2, 32, 96), torch.bfloat16), ((2, 32, 64), torch.float32)):
        with pytest.raises(ops.KernelError, match="operand tiles"):
            ops.expert_tiles(torch.zeros(shape, dtype=dtype, device=DEV))
