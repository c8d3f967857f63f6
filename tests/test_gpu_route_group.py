"""The router's product, the choice and the grouping of few tokens in one launch: the bits of the three launches it stands for."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check(chosen, weights, logits, top, scores, correction, scale, renormalize, groups):
    """Choices and weights against float64.  A logit is a float32 sum of k products, whose sizes add up to less than 80: some
    units of 2^-24 of that, 1e-4 at most, and a chosen score is then off by no more, a weight by 4e-4 of itself."""
    slack = 1e-4
    by = logits if scores == "softmax_chosen" else torch.softmax(logits, -1)
    value = by + correction.double() if correction is not None else by
    value, clear = value.cpu(), 0
    for t in range(value.shape[0]):
        row = value[t]
        if groups:
            best = row.reshape(groups[0], -1).amax(1)
            order = best.argsort(descending=True)
            if float(best[order[groups[1] - 1]] - best[order[groups[1]]]) <= 2 * slack:
                continue  # which group is closed hangs on the last bits
            row = row.clone().reshape(groups[0], -1)
            row[order[groups[1] :]] = float("-inf")
            row = row.flatten()
        clear += 1
        got = chosen[t].cpu().long()
        assert got.unique().numel() == top
        assert bool(((row[got] - row.sort(descending=True).values[:top]).abs() <= 2 * slack).all())
        picked = by[t].cpu()[got]
        want = torch.softmax(picked, 0) if scores == "softmax_chosen" else scale * picked / (picked.sum() if renormalize else 1.0)
        assert bool(((weights[t].cpu().double() - want).abs() <= 4 * slack * want).all())
    assert 2 * clear >= value.shape[0]


@pytest.mark.parametrize("tokens", [1, 2, 8, 15, 16])
@pytest.mark.parametrize("experts,top,groups", [(1, 1, None), (8, 2, None), (16, 4, (4, 2)), (40, 6, (8, 3)), (64, 16, None)])
@pytest.mark.parametrize("k", [32, 480, 2048, 8192])
def test_the_same_as_three_launches(tokens, experts, top, groups, k):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(tokens + experts + k)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x, router = normal(tokens, k).bfloat16(), (normal(experts, k) * k ** -0.5).bfloat16()
    copy = ops.stream_layout(router)
    bias, correction = normal(experts), 0.1 * normal(experts)
    for extra in ((None, ("softmax_chosen", None, 1.0, False, groups)), (bias, ("softmax_all", correction, 2.5, True, groups)), (None, ("softmax_all", None, 1.0, False, groups))):
        b, rule = extra
        want_logits = x.double() @ router.double().T + (b.double() if b is not None else 0)
        # the streaming product's logits (the two add in the same order; K up to 6,144 is one group of its wavefronts)
        logits = ops.gemm_bf16_stream(x, router, b, torch.float32)
        chosen, weights, lists = ops.route_and_group(x, copy, b, experts, top, *rule)
        want, want_weights = ops.route_top(logits, top, *rule)
        if k <= 6144:
            assert torch.equal(chosen, want) and torch.equal(weights, want_weights)
        check(chosen, weights, want_logits, top, *rule)
        other = ops.group_by_expert(chosen, experts)
        assert lists.n_tiles == other.n_tiles and torch.equal(lists.tile_expert, other.tile_expert) and torch.equal(lists.used, other.used)
        # a group's rows are in any order: every pair has a row of its own that names its token, in a tile of its expert
        rows = lists.pair_row.long()
        assert rows.unique().numel() == tokens * top and int((lists.row_token >= 0).sum()) == tokens * top
        assert torch.equal(lists.row_token[rows].long(), torch.arange(tokens * top, device=DEV) // top)
        assert torch.equal(lists.tile_expert[rows // 16], chosen.flatten())


def test_what_it_does_not_take():
    from cwm_amd import ops

    x, router = torch.zeros((17, 64), device=DEV, dtype=torch.bfloat16), torch.zeros((8, 64), device=DEV, dtype=torch.bfloat16)
    copy = ops.stream_layout(router)
    with pytest.raises(ops.KernelError, match="T <= 16"):
        ops.route_and_group(x, copy, None, 8, 2)
    with pytest.raises(ops.KernelError, match="does not fit"):
        ops.route_and_group(x[:4], copy, None, 24, 2)
    with pytest.raises(ops.KernelError, match="groups"):
        ops.route_and_group(x[:4], copy, None, 8, 4, groups=(4, 1))
