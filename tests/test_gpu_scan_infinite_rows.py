"""The selective scan of long bfloat16 portions with an infinity or a NaN among B or C: the kinds of values that the walk token by
token gives, and nothing before the token or in other groups' heads."""

from __future__ import annotations

import pytest
import torch

from test_gpu_scan_blocks import DEV, _batch

pytestmark = pytest.mark.gpu


def kinds(t):
    return torch.stack([torch.isnan(t), t == float("inf"), t == float("-inf")])


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [1, 14, 64 + 37, 256 + 63, 300])
@pytest.mark.parametrize("rows", [40, 128])
@pytest.mark.parametrize("which", ["B", "C"])
def test_as_the_walk_leaves_it(which, rows, at, bad):
    from cwm_amd import ops

    heads, width, groups, n = 4, 48, 2, 600
    inner = heads * width
    g = torch.Generator().manual_seed(at + rows)
    normal = lambda *shape: torch.randn(shape, generator=g)  # noqa: E731
    xbc, dt = normal(n, inner + 2 * groups * rows).bfloat16().to(DEV), (normal(n, heads) - 3).bfloat16().to(DEV)
    # rates that keep something over the whole portion, so that an infinity is never multiplied by a decay of 0
    bias, d_skip, a_log = normal(heads).to(DEV), normal(heads).to(DEV), torch.linspace(-5.0, -3.0, heads, device=DEV)
    spoilt = xbc.clone()
    spoilt[at, inner + (0 if which == "B" else groups * rows) + 3] = bad  # row 3 of the first group's
    start = torch.stack([ops.scan_state_pack(normal(heads, rows, width) * 0.3)]).to(DEV)
    fine, poisoned, walked = start.clone(), start.clone(), start.clone()
    want = ops.selective_scan(xbc, dt, bias, a_log, d_skip, fine, _batch([n], [0]), heads, width, rows, groups)
    got = ops.selective_scan(spoilt, dt, bias, a_log, d_skip, poisoned, _batch([n], [0]), heads, width, rows, groups)
    cuts = [0, 256, 512, n]
    y = torch.cat([ops.selective_scan(spoilt[a:b], dt[a:b], bias, a_log, d_skip, walked, _batch([b - a], [0]), heads, width, rows, groups) for a, b in zip(cuts, cuts[1:])])
    size = 4e-6 * want.abs().amax()
    assert bool(((got - want)[:at].abs() <= size).all()) and bool(((got - want)[:, inner // 2 :].abs() <= size).all())
    if which == "B":
        # the infinite row of B stays in the state: infinite results and states of the walk's signs, and no NaN where it has none
        assert bool((~torch.isfinite(got[at:, : inner // 2])).all())
        assert torch.equal(kinds(got), kinds(y))
        states = [ops.scan_state_unpack(t[0].cpu(), heads, width, rows) for t in (poisoned, walked)]
        assert torch.equal(*(kinds(t) for t in states)) and (bad != bad or bool(torch.isinf(states[0]).any()))
    else:
        # an infinite C is its own token's alone; its scores with the block's other tokens may be of either sign, so infinity or NaN
        assert not bool(torch.isfinite(got[at, : inner // 2]).any()) and torch.equal(torch.isfinite(got), torch.isfinite(y))
        assert bool(((poisoned - walked).abs() <= 4e-6 * walked.abs().amax()).all())
