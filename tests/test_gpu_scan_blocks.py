"""The selective scan of long bfloat16 portions, 64 tokens at a time on the matrix cores, against the recurrence in float64:
portions that end inside a block of tokens, at its edge and one past it, states whose rows fill no tile of 16, columns that
fill no block of 64, decays that forget within a token and ones that keep a state for thousands."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _batch(q_lens, slots):
    cu = torch.tensor([0] + q_lens).cumsum(0).int()
    seq = torch.repeat_interleave(torch.arange(len(q_lens)), torch.tensor(q_lens)).int()
    return SimpleNamespace(
        n_tokens=sum(q_lens), n_seqs=len(q_lens), q_lens=list(q_lens), cu_q=cu.to(DEV), seq_of_token=seq.to(DEV),
        state_slots=torch.tensor(slots, dtype=torch.int32, device=DEV), scratch={},
    )


def _exact(xbc, dt, bias, a_log, d_skip, state, q_lens, slots, heads, width, rows, groups):
    """float64 on the CPU; `state` [slots, heads, rows, width] is updated."""
    inner = heads * width
    xs = xbc[:, :inner].reshape(-1, heads, width)
    b, c = (t.reshape(-1, groups, rows).repeat_interleave(heads // groups, 1) for t in (xbc[:, inner : inner + groups * rows], xbc[:, inner + groups * rows :]))
    dt = torch.nn.functional.softplus(dt + bias, threshold=100.0)
    keep = torch.exp(-torch.exp(a_log) * dt)
    y, at = torch.zeros_like(xs), 0
    for q, slot in zip(q_lens, slots):
        S = state[slot]
        for t in range(at, at + q):
            S = keep[t][:, None, None] * S + (dt[t][:, None] * b[t])[:, :, None] * xs[t][:, None, :]
            y[t] = (S * c[t][:, :, None]).sum(1) + d_skip[:, None] * xs[t]
        state[slot] = S
        at += q
    return y.reshape(-1, inner)


@pytest.mark.parametrize("heads,width,rows,groups", [(4, 64, 128, 2), (2, 16, 8, 1), (3, 48, 72, 3), (2, 80, 64, 1), (1, 128, 24, 1)])
@pytest.mark.parametrize("q_lens", [[257], [320, 1, 64], [5, 511, 768], [1025, 256]])
def test_long_portions_against_float64(heads, width, rows, groups, q_lens):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(sum(q_lens) + rows)
    normal = lambda *shape: torch.randn(shape, generator=g)  # noqa: E731
    slots = [2, 0, 1][: len(q_lens)]
    total = heads * width + 2 * groups * rows
    bias, d_skip = normal(heads) * 0.5, normal(heads)
    a_log = torch.linspace(-7.0, 2.5, heads) if heads > 1 else torch.tensor([-2.0])
    state = normal(3, heads, rows, width) * 0.3
    packed = torch.stack([ops.scan_state_pack(s) for s in state]).to(DEV)
    exact_state = state.double()
    for _ in range(2):  # the second step goes on from the first one's states
        n = sum(q_lens)
        xbc, dt = normal(n, total).bfloat16(), (normal(n, heads) - 1).bfloat16()
        dt[::97] += 24.0  # steps beyond the softplus' linear part
        wide = torch.zeros((n, total + 24), dtype=torch.bfloat16, device=DEV)  # rows that lie apart
        wide[:, :total] = xbc.to(DEV)
        got = ops.selective_scan(wide[:, :total], dt.to(DEV), bias.to(DEV), a_log.to(DEV), d_skip.to(DEV), packed, _batch(q_lens, slots), heads, width, rows, groups)
        want = _exact(xbc.double(), dt.double(), bias.double(), a_log.double(), d_skip.double(), exact_state, q_lens, slots, heads, width, rows, groups)
        # float32 sums of at most some thousand terms: 64 roundings of 2^-24 of the values' size
        scale = want.reshape(n, heads, width).abs().amax((0, 2)).clamp(min=1.0)
        assert bool(((got.double().cpu() - want).reshape(n, heads, width).abs().amax((0, 2)) <= 4e-6 * scale).all())
        for slot in range(3):
            mine = ops.scan_state_unpack(packed[slot].cpu(), heads, width, rows).double()
            size = exact_state[slot].abs().amax((1, 2)).clamp(min=1.0)
            assert bool(((mine.reshape(heads, rows, width) - exact_state[slot]).abs().amax((1, 2)) <= 4e-6 * size).all())


@pytest.mark.parametrize("heads,width,rows,groups", [(4, 64, 128, 2), (3, 48, 72, 3)])
@pytest.mark.parametrize("q_lens", [[320, 1, 64], [1, 256, 257], [1, 1, 600]])
def test_short_portions_beside_a_long_one_keep_their_bits(heads, width, rows, groups, q_lens):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(sum(q_lens))
    normal = lambda *shape: torch.randn(shape, generator=g)  # noqa: E731
    n = sum(q_lens)
    xbc, dt = normal(n, heads * width + 2 * groups * rows).bfloat16().to(DEV), (normal(n, heads) - 1).bfloat16().to(DEV)
    bias, d_skip, a_log = (normal(heads).to(DEV) for _ in range(3))
    state = torch.stack([ops.scan_state_pack(normal(heads, rows, width) * 0.3) for _ in range(3)]).to(DEV)
    slots, beside = [1, 2, 0], state.clone()
    together = ops.selective_scan(xbc, dt, bias, a_log, d_skip, beside, _batch(q_lens, slots), heads, width, rows, groups)
    at = 0
    for q, slot in zip(q_lens, slots):
        if q <= 256:
            alone = state.clone()
            y = ops.selective_scan(xbc[at : at + q], dt[at : at + q], bias, a_log, d_skip, alone, _batch([q], [slot]), heads, width, rows, groups)
            assert torch.equal(y, together[at : at + q]) and torch.equal(alone[slot], beside[slot])
        at += q


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [1, 14, 64 + 37, 256 + 63, 300])
def test_a_value_that_is_not_finite_reaches_no_earlier_token(bad, at):
    from cwm_amd import ops

    heads, width, rows, groups, n = 2, 48, 40, 1, 350
    g = torch.Generator().manual_seed(at)
    normal = lambda *shape: torch.randn(shape, generator=g)  # noqa: E731
    xbc, dt = normal(n, heads * width + 2 * groups * rows).bfloat16().to(DEV), (normal(n, heads) - 1).bfloat16().to(DEV)
    bias, d_skip, a_log = (normal(heads).to(DEV) for _ in range(3))
    spoilt = xbc.clone()
    spoilt[at, 5] = bad  # x of the first head
    start = torch.stack([ops.scan_state_pack(normal(heads, rows, width) * 0.3)]).to(DEV)
    fine, poisoned = start.clone(), start.clone()
    want = ops.selective_scan(xbc, dt, bias, a_log, d_skip, fine, _batch([n], [0]), heads, width, rows, groups)
    got = ops.selective_scan(spoilt, dt, bias, a_log, d_skip, poisoned, _batch([n], [0]), heads, width, rows, groups)
    others = torch.arange(heads * width, device=DEV) != 5
    assert torch.equal(got[:, others], want[:, others]) or bool(((got - want)[:, others].abs() <= 4e-6 * want.abs().amax()).all())
    # the tokens before it, whose sums may come in another order
    assert bool(((got - want)[:at].abs() <= 4e-6 * want.abs().amax()).all())
    assert not bool(torch.isfinite(got[at, 5]))
    # and as the walk leaves it: the same tokens in portions of one segment
    walked = start.clone()
    y = torch.cat([ops.selective_scan(spoilt[a:b], dt[a:b], bias, a_log, d_skip, walked, _batch([b - a], [0]), heads, width, rows, groups) for a, b in ((0, 200), (200, n))])
    assert torch.equal(torch.isfinite(y), torch.isfinite(got))


def test_decays_of_nothing_left():
    """Rates whose logarithms are huge or infinite: the walk's decay is 0, and so is the blocks'."""
    from cwm_amd import ops

    heads, width, rows, groups, n = 4, 16, 24, 1, 400
    g = torch.Generator().manual_seed(7)
    normal = lambda *shape: torch.randn(shape, generator=g)  # noqa: E731
    xbc, dt = normal(n, heads * width + 2 * groups * rows).bfloat16().to(DEV), normal(n, heads).bfloat16()
    dt[100] = -60.0  # a step of e^-60: nothing added, and at the lesser rates nothing forgotten
    a_log = torch.tensor([100.0, 88.0, 30.0, 5.0], device=DEV)
    bias, d_skip, dt = normal(heads).to(DEV), normal(heads).to(DEV), dt.to(DEV)
    start = torch.stack([ops.scan_state_pack(normal(heads, rows, width))]).to(DEV)
    whole, walked = start.clone(), start.clone()
    got = ops.selective_scan(xbc, dt, bias, a_log, d_skip, whole, _batch([n], [0]), heads, width, rows, groups)
    want = torch.cat([ops.selective_scan(xbc[a:b], dt[a:b], bias, a_log, d_skip, walked, _batch([b - a], [0]), heads, width, rows, groups) for a, b in ((0, 256), (256, n))])
    assert bool(torch.isfinite(want).all())
    assert bool(((got - want).abs() <= 4e-6 * want.abs().amax()).all())
    assert bool(((whole - walked).abs() <= 4e-6 * walked.abs().amax().clamp(min=1.0)).all())
