"""The router's product, the choice and the grouping of few tokens in one launch: the bits of the three launches it stands for."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


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
        else:  # sums of k products: a few units of 2^-24 of their size decide only between close scores
            assert bool((torch.gather(want_logits, 1, chosen.long()) - torch.gather(want_logits, 1, want.long())).abs().max() <= 1e-4) or groups
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
