"""The router's choice among at most as many experts as lanes: ties, signed zeros, infinities, groups, NaN."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _order(values):
    return sorted(range(len(values)), key=lambda e: (-values[e], e))


@pytest.mark.parametrize("n_experts,top,groups", [(1, 1, None), (5, 5, None), (16, 4, None), (16, 4, (4, 2)), (63, 7, None), (64, 8, None), (64, 8, (8, 3)), (60, 6, (6, 5)), (65, 8, None)])
def test_choice_and_weights(n_experts, top, groups):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(n_experts + top)
    logits = torch.randint(-3, 4, (37, n_experts), generator=g).float()  # most rows have ties
    logits[0] = 0.0
    logits[0, ::2] = -0.0
    logits[1] = float("-inf")
    logits[1, n_experts // 2] = 1.0
    logits[2:20] += torch.randn((18, n_experts), generator=g)
    if groups is None:
        chosen, weights = ops.route_top(logits.to(DEV), top)
        for t, row in enumerate(logits.tolist()):
            want = _order(row)[:top]
            assert chosen[t].tolist() == want
            soft = torch.softmax(torch.tensor([row[e] for e in want], dtype=torch.float64), 0)
            # an exponential, up to eight additions and a division in float32
            assert bool(((weights[t].cpu().double() - soft).abs() <= 2.0 ** -20 * soft).all())
    correction = torch.randint(-2, 3, (n_experts,), generator=g).float()
    chosen, weights = ops.route_top(logits[2:].to(DEV), top, "softmax_all", correction.to(DEV), 2.5, True, groups)
    scores = torch.softmax(logits[2:].double(), -1)
    by = scores + correction.double()
    for t in range(by.shape[0]):
        values = by[t].tolist()
        if groups:
            size = n_experts // groups[0]
            ranked = _order(values)
            keep = list(dict.fromkeys(e // size for e in ranked))[: groups[1]]
            values = [v if e // size in keep else float("-inf") for e, v in enumerate(values)]
        got = chosen[t].tolist()
        assert len(set(got)) == top
        # float32 scores may tie or change places where float64's lie within a few units of 2^-22
        for a, b in zip(got, _order(values)[:top]):
            assert abs(values[a] - values[b]) <= 2.0 ** -20
        picked = scores[t, chosen[t].cpu().long()]
        assert bool(((weights[t].cpu().double() - 2.5 * picked / picked.sum()).abs() <= 2.0 ** -18 * 2.5 * picked / picked.sum()).all())


def test_a_row_with_nan_still_names_experts():
    from cwm_amd import ops

    logits = torch.randn(6, 16, device=DEV)
    logits[0], logits[1, 3], logits[2, 0], logits[3, 15] = float("nan"), float("nan"), -float("nan"), float("nan")
    chosen, weights = ops.route_top(logits, 4)
    assert all(len(set(row)) == 4 and 0 <= min(row) and max(row) < 16 for row in chosen.tolist())
    assert bool(weights[:4].isnan().all()) and not bool(weights[4:].isnan().any())
