"""Which steps the convolutions take in runs of four tokens: portions of a prompt whose threads 31 bits number.  Larger steps are answered
as before, by the kernels of a thread a channel."""

from __future__ import annotations

import pytest

from cwm_amd.ops import build


@pytest.mark.parametrize(
    "n_tokens,n_seqs,channels,runs",
    [
        (2048, 1, 6144, True), (16, 16, 6144, False), (17, 16, 6144, True), (2048, 1, 6140, False), (2, 0, 8, None),
        (11184804, 1, 6144, True), (11184805, 1, 6144, False), (4 * 2 ** 21, 1, 8192, False), (4 * (2 ** 21 - 2), 1, 8192, True), (2 ** 24 - 1, 1, 4096, False),
        (2 ** 24 - 1, 1, 2048, True), (5, 4, 8, True),
    ],
)
def test_steps_in_runs(n_tokens, n_seqs, channels, runs):
    silu = build.load("state_space").cwm_conv_silu_in_runs
    short = build.load("short_conv").cwm_short_conv_in_runs
    if runs is None:  # no sequences at all: no state to leave
        assert not silu(n_tokens, n_seqs, channels)
        return
    assert bool(silu(n_tokens, n_seqs, channels)) == runs
    for taps in (2, 3, 4):
        assert bool(short(n_tokens, n_seqs, taps, channels)) == runs
    assert not short(n_tokens, n_seqs, 1, channels) and not short(n_tokens, n_seqs, 5, channels)
