"""The grouped product whose rows go through LDS: every shape of block (2, 4 and 8 row tiles, 2 and 4 weight tiles a
wavefront), results' columns that no block divides, experts without tokens and one with most of them."""

from __future__ import annotations

import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows an expert: 2 and 3 (the split of K, then two row tiles), 15 and 16 (two, four), 47 and 48 (four, eight), 300;
# 640 columns of 128 make four weight tiles a wavefront pay at 900 tokens and 32 experts
@pytest.mark.parametrize("n_tokens,n_experts,top", [(1, 4, 1), (11, 4, 1), (12, 4, 1), (30, 8, 4), (32, 8, 4), (94, 8, 4), (96, 8, 4), (600, 8, 4), (900, 32, 4)])
@pytest.mark.parametrize("dim,hidden", [(64, 64), (192, 320), (320, 192), (640, 648)])
@pytest.mark.parametrize("crowded", [False, True])
def test_rows_of_experts(n_tokens, n_experts, top, dim, hidden, crowded):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n_tokens * dim + hidden)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = normal(n_tokens, dim).bfloat16()
    gate, up, down = (normal(n_experts, a, b).mul(b ** -0.5).bfloat16() for a, b in ((hidden, dim), (hidden, dim), (dim, hidden)))
    scores = normal(n_tokens, n_experts)
    if crowded:  # nearly everything to the last experts, nothing to the first
        scores[:, -top:] += 6.0
        scores[:, 0] -= 30.0 if n_experts > top else 0.0
    chosen = scores.topk(top).indices.int().contiguous()
    groups = ops.group_by_expert(chosen, n_experts)
    lists = groups.pair_row.long()
    assert len(set(lists.tolist())) == n_tokens * top
    assert torch.equal(groups.row_token[lists].long(), torch.arange(n_tokens * top, device=DEV) // top)
    assert torch.equal(groups.tile_expert[lists // 16], chosen.reshape(-1))
    rows = ops.grouped_gate_up(x, groups, gate, up)
    out = ops.grouped_linear(rows, groups, down)
    token, expert = torch.arange(n_tokens, device=DEV).repeat_interleave(top), chosen.reshape(-1).long()
    # what is stored has bfloat16's 8 bits: half a unit of the last is at most 2^-8 of the value; the sums before it, float32
    # over K <= 648 products of order K^-0.5, are off by some K^0.5 2^-24 < 2e-6, here and through the activation below 2e-5
    for e in range(n_experts):
        mine = torch.nonzero(expert == e)[:, 0]
        if not mine.numel():
            continue
        a = x[token[mine]].double()
        want = torch.nn.functional.silu(a @ gate[e].double().T) * (a @ up[e].double().T)
        got = rows[lists[mine]].double()
        assert bool(((got - want).abs() <= want.abs() * 2.0 ** -8 + 2e-5).all()), f"expert {e}: gate and up"
        want = got @ down[e].double().T
        assert bool(((out[lists[mine]].double() - want).abs() <= 1e-5 * want.abs() + 1e-5).all()), f"expert {e}: down"


@pytest.mark.parametrize("n_tokens", [1, 15, 16, 17, 48, 129, 700])
@pytest.mark.parametrize("heads,lead,d,n", [(3, 64, 128, 192), (5, 0, 64, 64), (2, 16, 64, 72)])
def test_rows_of_heads(n_tokens, heads, lead, d, n):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n_tokens + n)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    rest = normal(n_tokens, heads, lead + d).bfloat16()[..., lead:]
    weight = normal(heads, n, d).mul(d ** -0.5).bfloat16()
    ask = normal(n_tokens, heads, lead + n).bfloat16()
    before = ask.clone()
    ops.absorb_queries(rest, ask, lead, weight)
    assert torch.equal(ask[..., :lead], before[..., :lead])
    want = torch.einsum("thd,hnd->thn", rest.double().cpu(), weight.double().cpu()).to(DEV)
    assert bool(((ask[..., lead:].double() - want).abs() <= want.abs() * 2.0 ** -8 + 2e-5).all())


@pytest.mark.parametrize("n_tokens", [30, 96, 600])
def test_lists_that_lie_elsewhere(n_tokens):
    """Copies of a step's lists, and lists without the number of tiles in use: what is read lies inside what is handed over."""
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n_tokens)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x, (gate, up) = normal(n_tokens, 128).bfloat16(), (normal(8, 192, 128).bfloat16() for _ in range(2))
    groups = ops.group_by_expert(normal(n_tokens, 8).topk(4).indices.int().contiguous(), 8)
    want = ops.grouped_gate_up(x, groups, gate, up)[groups.pair_row.long()]
    copies = dataclasses.replace(groups, row_token=groups.row_token.clone(), tile_expert=groups.tile_expert.clone(), used=groups.used.clone())
    for lists in (copies, dataclasses.replace(copies, used=None)):
        assert lists.tile_expert.numel() == lists.n_tiles
        assert torch.equal(ops.grouped_gate_up(x, lists, gate, up)[groups.pair_row.long()], want)
    with pytest.raises(ops.KernelError):
        ops.grouped_gate_up(x, dataclasses.replace(groups, tile_expert=groups.tile_expert[:-1]), gate, up)


@pytest.mark.parametrize("dtype,n_tokens", [(torch.bfloat16, 8), (torch.bfloat16, 96), (torch.float32, 8)])
def test_a_captured_product_reads_nothing_that_other_sizes_replace(dtype, n_tokens):
    """Lists of many other sizes come between a capture and its replays, as prompts do between decode steps."""
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n_tokens)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x, chosen = normal(n_tokens, 64).to(dtype), normal(n_tokens, 8).topk(2).indices.int().contiguous()
    gate, up, down = (normal(8, *s).mul(0.1).to(dtype) for s in ((96, 64), (96, 64), (64, 96)))

    def step(tokens, picks):
        groups = ops.group_by_expert(picks, 8)
        return ops.grouped_linear(ops.grouped_gate_up(tokens, groups, gate, up), groups, down)[groups.pair_row.long()]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(x, chosen)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(x, chosen)
    for turn in range(3):
        for n in range(40 * turn + 9, 40 * turn + 49):  # 80 and more different lists
            more = normal(4 * n, 64).to(dtype)
            step(more, normal(4 * n, 8).topk(2).indices.int().contiguous())
        taken = [torch.full((size,), 1 << 20, dtype=torch.int32, device=DEV) for size in range(128, 4096, 16)]  # what was freed, if anything was
        x.copy_(normal(n_tokens, 64))
        graph.replay()
        assert torch.equal(out, step(x, chosen)), turn
        del taken
