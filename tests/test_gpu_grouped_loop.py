"""Routed experts' products of many rows with weights in operand tiles (persistent blocks) beside the row-major ones: the same bits."""

import dataclasses

import pytest
import torch

from cwm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# fewer tiles of 128 rows and 256 columns than half a round of 256 blocks (quarters alone), more than half of one (one round), rounds with a
# rest in quarters and with one more round; a lone step of K and columns that end inside a tile; experts without rows, or with nearly all of them
@pytest.mark.parametrize("n_tokens,n_experts,top", [(200, 4, 2), (1500, 8, 4), (3000, 8, 4), (2100, 32, 4)])
@pytest.mark.parametrize("dim,hidden", [(64, 1088), (192, 272), (1024, 64)])
@pytest.mark.parametrize("crowded", [False, True])
def test_the_same_bits(n_tokens, n_experts, top, dim, hidden, crowded, monkeypatch):
    monkeypatch.setattr("cwm_amd.ops.routed._loop_pays", lambda *sizes: True)
    g = torch.Generator(device=DEV).manual_seed(n_tokens + dim + hidden)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = normal(n_tokens, dim).bfloat16()
    gate, up = (normal(n_experts, hidden, dim).mul(dim**-0.5).bfloat16() for _ in range(2))
    down = normal(n_experts, dim, hidden).mul(hidden**-0.5).bfloat16()
    scores = normal(n_tokens, n_experts)
    if crowded:
        scores[:, -top:] += 5.0
        scores[:, 0] -= 30.0
    groups = ops.group_by_expert(scores.topk(top).indices.int().contiguous(), n_experts)
    assert groups.tiles_a_block == 8
    mine = groups.pair_row.long()
    for activation in (None, ops.GatedActivation("clamped_swish", 1.7, 2.0)):
        want = ops.grouped_gate_up(x, groups, gate, up, activation)
        got = ops.grouped_gate_up(x, groups, ops.expert_tiles(gate), ops.expert_tiles(up), activation)
        assert torch.equal(got[mine], want[mine])
    if hidden % 64 == 0:
        assert torch.equal(ops.grouped_linear(want, groups, ops.expert_tiles(down))[mine], ops.grouped_linear(want, groups, down)[mine])


# lists of one to eight tiles past a whole block, which end in each of a block's tiles
@pytest.mark.parametrize("past", range(1, 9))
def test_lists_whose_tiles_are_not_counted(past, monkeypatch):
    """Without the number of tiles in use the blocks walk the whole list, whose last one may end inside its rows."""
    monkeypatch.setattr("cwm_amd.ops.routed._loop_pays", lambda *sizes: True)
    n_experts, top, dim, hidden = 4, 2, 192, 320
    n_tokens = 8 * (64 + past) - 3
    g = torch.Generator(device=DEV).manual_seed(past)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x, gate, up = normal(n_tokens, dim).bfloat16(), *(normal(n_experts, hidden, dim).mul(dim**-0.5).bfloat16() for _ in range(2))
    down = normal(n_experts, dim, hidden).mul(hidden**-0.5).bfloat16()
    groups = ops.group_by_expert(normal(n_tokens, n_experts).topk(top).indices.int().contiguous(), n_experts)
    assert groups.tiles_a_block == 8 and groups.n_tiles % 8 == past % 8
    mine = groups.pair_row.long()
    want = ops.grouped_gate_up(x, groups, gate, up)
    lists = dataclasses.replace(groups, used=None)
    assert torch.equal(ops.grouped_gate_up(x, lists, ops.expert_tiles(gate), ops.expert_tiles(up))[mine], want[mine])
    assert torch.equal(ops.grouped_linear(want, lists, ops.expert_tiles(down))[mine], ops.grouped_linear(want, groups, down)[mine])


# the blocks of four wavefronts that the rule leaves other products to: two and four column tiles a wavefront (fewer than 500 blocks of four, and more)
@pytest.mark.parametrize("n_tokens,n_experts,hidden", [(1500, 16, 256), (1500, 16, 1088)])
@pytest.mark.parametrize("loop", [False, True])
def test_both_kernels_against_float64(n_tokens, n_experts, hidden, loop, monkeypatch):
    monkeypatch.setattr("cwm_amd.ops.routed._loop_pays", lambda *sizes: loop)
    top, dim = 4, 192
    g = torch.Generator(device=DEV).manual_seed(hidden)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = normal(n_tokens, dim).bfloat16()
    gate, up = (normal(n_experts, hidden, dim).mul(dim**-0.5).bfloat16() for _ in range(2))
    down = normal(n_experts, 16 * 128 if hidden > 256 else 64, hidden).mul(hidden**-0.5).bfloat16()
    chosen = normal(n_tokens, n_experts).topk(top).indices.int().contiguous()
    groups = ops.group_by_expert(chosen, n_experts)
    assert groups.tiles_a_block == 8
    mine, expert, token = groups.pair_row.long(), chosen.flatten().long(), torch.arange(n_tokens, device=DEV).repeat_interleave(top)
    h = ops.grouped_gate_up(x, groups, ops.expert_tiles(gate), ops.expert_tiles(up))
    assert torch.equal(h[mine], ops.grouped_gate_up(x, groups, gate, up)[mine])
    y = ops.grouped_linear(h, groups, ops.expert_tiles(down))
    assert torch.equal(y[mine], ops.grouped_linear(h, groups, down)[mine])
    for e in range(0, n_experts, 5):
        rows = expert == e
        a, b = x[token[rows]].double(), h[mine[rows]].double()
        # a float32 sum of K products is off by at most K * 2^-24 of the sum of their sizes
        want, most = b @ down[e].double().t(), b.abs() @ down[e].double().abs().t()
        assert ((y[mine[rows]].double() - want).abs() <= hidden * 2.0**-24 * most).all()
        # the gate's and up's sums are off by as much each, silu's slope is below 1.1, and one rounding to bfloat16 is 2^-9 of the value
        gs, us = a @ gate[e].double().t(), a @ up[e].double().t()
        off = dim * 2.0**-24
        gm, um = a.abs() @ gate[e].double().abs().t(), a.abs() @ up[e].double().abs().t()
        want = torch.nn.functional.silu(gs) * us
        bound = 2.0**-8 * want.abs() + 2 * off * (1.1 * gm * us.abs() + gs.abs() * um + 1.1 * off * gm * um) + 1e-6
        assert ((b - want).abs() <= bound).all()
