"""Which products of routed experts go to the persistent blocks: points where both kernels were timed, on either side of every line of the rule."""

from __future__ import annotations

import pytest

from cwm_amd.ops.routed import _loop_pays


# tokens, experts, choices a token, columns, K, with gates and ups; (us, the other kernel and the persistent blocks)
@pytest.mark.parametrize("tokens,n_experts,top,columns,k,gated,takes", [
    (2048, 16, 4, 1024, 2048, True, True),  # 2.25 rounds (77 / 72)
    (1500, 16, 4, 1024, 2048, True, False),  # 1.71 (72 / 75)
    (203, 4, 2, 2048, 2048, True, True),  # one round of quarters (34 / 22)
    (203, 4, 2, 2048, 2048, False, True),  # (29 / 19)
    (145, 8, 2, 320, 512, True, True),  # the same with a short K
    (262, 16, 4, 1024, 2048, True, True),  # two rounds of quarters, gated (36 / 36 evenly, 48 / 41 unevenly spread)
    (262, 16, 4, 2048, 1024, False, False),  # and not (20 / 24, 27 / 26)
    (2605, 8, 1, 1024, 1024, False, False),  # (18.1 / 18.7)
    (5128, 8, 2, 320, 512, True, False),  # a short K (18 / 24)
    (8195, 8, 2, 512, 320, False, False),
    (1286, 4, 2, 2048, 2048, True, False),  # 1.4 rounds (59 / 66)
    (8195, 64, 8, 768, 2048, True, False),  # 12.8 rounds (408 / 435)
])
def test_where_they_go(tokens, n_experts, top, columns, k, gated, takes):
    assert _loop_pays(tokens * top, n_experts, columns, k, gated) is takes
