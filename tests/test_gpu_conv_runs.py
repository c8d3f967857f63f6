"""Convolutions over time of whole portions, whose rows a thread reads once for four tokens: portions shorter than the taps, ends
inside and at the borders of four tokens, states of any slot, against the same tokens one a step (the kernels of a decode step)."""

from __future__ import annotations

import pytest
import torch

from test_gpu_digasun import DEV, step_batch

pytestmark = pytest.mark.gpu
LENGTHS = [1, 2, 3, 4, 5, 7, 8, 9, 31, 64]


def _alone(n_seqs, at, lens, slots):
    """The step of the sequences that still have a token at place `at`."""
    left = [i for i in range(n_seqs) if lens[i] > at]
    return left, step_batch([10] * len(left), [1] * len(left), [slots[i] for i in left])


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("dim,pad", [(8, 0), (24, 8), (2048, 0), (1032, 16)])
@pytest.mark.parametrize("two,write", [(True, True), (False, True), (True, False)])
def test_short_convolutions(taps, dim, pad, two, write):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(dim + taps)
    slots = [len(LENGTHS) - i for i in range(len(LENGTHS))]
    wide = torch.randn((sum(LENGTHS), dim + pad), generator=g).bfloat16().to(DEV)
    x = wide[:, :dim]
    w = [torch.randn((taps, dim), generator=g).to(DEV) for _ in range(2 if two else 1)]
    state = torch.randn((len(LENGTHS) + 1, (taps - 1) * dim + 8), generator=g).to(DEV)
    before, steps = state.clone(), state.clone()
    got = ops.short_conv(x, w, state, step_batch([10] * len(LENGTHS), LENGTHS, slots), write_state=write)
    starts = [sum(LENGTHS[:i]) for i in range(len(LENGTHS))]
    for at in range(max(LENGTHS)):
        left, batch = _alone(len(LENGTHS), at, LENGTHS, slots)
        rows = [starts[i] + at for i in left]
        one = ops.short_conv(x[rows].contiguous(), w, steps, batch)
        for a, b in zip(got, one):
            assert torch.equal(a[rows], b), at
    assert torch.equal(state, steps if write else before)


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("channels,lead", [(8, 0), (40, 8), (2056, 24)])
def test_convolutions_with_an_activation(taps, channels, lead):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(channels + taps)
    slots = [len(LENGTHS) - i for i in range(len(LENGTHS))]
    wide = torch.randn((sum(LENGTHS), channels + lead), generator=g).bfloat16().to(DEV)
    x = wide[:, lead:]
    w, b = torch.randn((channels, taps), generator=g).to(DEV), torch.randn(channels, generator=g).to(DEV)
    by_tap, offset = w.t().contiguous(), 16
    state = torch.randn((len(LENGTHS) + 1, offset + (taps - 1) * channels), generator=g).to(DEV)
    steps = state.clone()
    got = ops.causal_conv_silu(x, w, b, state, offset, step_batch([10] * len(LENGTHS), LENGTHS, slots), by_tap)
    starts = [sum(LENGTHS[:i]) for i in range(len(LENGTHS))]
    for at in range(max(LENGTHS)):
        left, batch = _alone(len(LENGTHS), at, LENGTHS, slots)
        rows = [starts[i] + at for i in left]
        one = ops.causal_conv_silu(x[rows].contiguous(), w, b, steps, offset, batch, by_tap)
        assert torch.equal(got[rows], one), at
    assert torch.equal(state, steps)
