"""A router's logits and choice of many tokens in one launch: for every 16 tokens what the launch for few tokens gives."""

import pytest
import torch

from cwm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# a lone token, one block, a last block of one token, many blocks; K of one step, of fewer steps than wavefronts, and long
@pytest.mark.parametrize("tokens", [1, 16, 17, 300])
@pytest.mark.parametrize("experts,top,groups", [(1, 1, None), (16, 4, (4, 2)), (40, 6, None)])
@pytest.mark.parametrize("k", [32, 480, 4096])
def test_the_bits_of_sixteen_at_a_time(tokens, experts, top, groups, k):
    g = torch.Generator(device=DEV).manual_seed(tokens + experts + k)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = normal(tokens, k + 8).bfloat16()[:, :k]  # rows that lie apart
    copy = ops.stream_layout((normal(experts, k) * k**-0.5).bfloat16())
    for bias, rule in ((None, ("softmax_chosen", None, 1.0, False, groups)), (normal(experts), ("softmax_all", 0.1 * normal(experts), 2.5, True, groups))):
        chosen, weights = ops.route_rows(x, copy, bias, experts, top, *rule)
        for t in range(0, tokens, 16):
            want, want_weights, _ = ops.route_and_group(x[t : t + 16], copy, bias, experts, top, *rule)
            assert torch.equal(chosen[t : t + 16], want) and torch.equal(weights[t : t + 16], want_weights)
