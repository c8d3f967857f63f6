"""Sampling of rows that are cut into segments: vocabularies at the edges of segments and of 16-byte loads, distributions
whose nucleus ends in a bin of few entries, of thousands and of equal ones, masked logits, extreme temperatures, and rows
that one block does alone."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from plain import llama3_plain as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(vocab, g):
    """Rows of logits by kind."""
    normal = lambda std: torch.randn(vocab, generator=g) * std  # noqa: E731
    peaked = normal(0.3)
    peaked[vocab // 3] += 14.0
    masked = torch.full((vocab,), -math.inf)
    masked[vocab // 2 : vocab // 2 + 40] = normal(2.0)[:40]  # whole segments without an entry
    far = normal(1.0) + 3000.0
    few = torch.round(normal(2.0))  # many equal ones in every bin
    return {"normal": normal(3.0), "flat": normal(0.02), "peaked": peaked, "masked": masked, "far": far, "equal": torch.zeros(vocab), "few": few}


@pytest.mark.parametrize("vocab", [8192, 8193, 8256, 10243, 32768, 100003, 131072])
def test_draws_follow_the_inverse_cdf_of_the_nucleus(vocab):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(vocab)
    rows, temps, tops, kinds = [], [], [], []
    for kind, row in _rows(vocab, g).items():
        for temp, top_p in ((0.0, 0.9), (0.7, 0.95), (1.0, 0.5), (1.3, 1.0), (0.9, 1e-6), (0.05, 0.9), (50.0, 0.8), (1.0, 0.9999)):
            rows.append(row), temps.append(temp), tops.append(top_p), kinds.append(kind)
    logits = torch.stack(rows)
    n = len(rows)
    us = torch.rand(n, generator=g)
    us[::7], us[3::11] = 0.0, 1.0 - 2.0 ** -24
    args = [t.to(DEV) for t in (logits, torch.tensor(temps), torch.tensor(tops), us)]
    packed = ops.sample_packed(*args)
    assert torch.equal(packed, ops.sample_packed(*args))  # the same bits every time
    toks, lp, slp = (t.cpu() for t in ops.unpack_sampled(packed))
    logp = torch.log_softmax(logits.double(), -1)
    for r in range(n):
        tok, where = int(toks[r]), f"vocabulary {vocab}, {kinds[r]}, temperature {temps[r]}, top_p {tops[r]}"
        assert 0 <= tok < vocab, where
        # 2^-24 of the logit itself (the far ones) beside the sum's rounding
        np.testing.assert_allclose(float(lp[r]), float(logp[r, tok]), rtol=1e-4, atol=5e-4 if kinds[r] == "far" else 1e-4, err_msg=where)
        if temps[r] <= 0:
            assert tok == plain.greedy(logits[r]), where
            continue
        probs = torch.softmax(logits[r].double() / temps[r], -1)
        values = torch.sort(probs, descending=True).values
        above = torch.cumsum(values, 0) - values
        # entries that are kept for certain and those that may be: equal ones are all kept, and a sum of float32 values is
        # off by up to 1e-5 of the mass; float32 exponents of (x - max) / T are off by 1e-6 and, far from 0, by x's own rounding
        off = 2e-5 if kinds[r] != "far" else 1e-3
        least = float(values[above <= tops[r] + off][-1]) * (1 - 1e-4)
        assert float(probs[tok]) >= least, where
        kept = torch.where(probs >= float(values[above <= tops[r]][-1]) * (1 - 1e-6), probs, torch.zeros_like(probs))
        total = float(kept.sum())
        np.testing.assert_allclose(float(slp[r]), math.log(float(probs[tok]) / total), rtol=2e-3, atol=2e-3 if kinds[r] != "far" else 2e-2, err_msg=where)
        cdf = torch.cumsum(kept / total, 0)
        slack = 2e-3 if kinds[r] == "far" else 1e-4
        assert float(cdf[tok] - kept[tok] / total) <= float(us[r]) + slack and float(cdf[tok]) >= float(us[r]) - slack, where


def test_rows_that_one_block_does_alone():
    """NaN, infinities and temperatures beyond the bins' range give what they gave in a row of one segment."""
    from cwm_amd import ops

    short = 2000
    g = torch.Generator().manual_seed(5)
    base = torch.randn(short, generator=g)
    rows = []
    for kind in range(6):
        row = base.clone()
        if kind == 0:
            row[700] = math.nan
        elif kind == 1:
            row[:] = -math.inf
        elif kind == 2:
            row[[300, 900]] = math.inf
        elif kind == 3:
            row[:] = math.nan
        elif kind == 4:
            row *= 1e30
        rows.append(row)
    rows = torch.stack(rows).repeat_interleave(4, 0)
    n = rows.shape[0]
    temps = torch.tensor([0.0, 0.8, 0.8, 1e-9]).repeat(n // 4)
    tops = torch.tensor([1.0, 0.9, 1.0, 0.9]).repeat(n // 4)
    us = torch.full((n,), 0.4)
    want = ops.sample(*(t.to(DEV) for t in (rows, temps, tops, us)))
    # the same rows with entries behind them that nothing chooses
    longer = torch.full((n, 9001), -math.inf)
    longer[:, :short] = rows
    got = ops.sample(*(t.to(DEV) for t in (longer, temps, tops, us)))
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("value,temp", [(25.0, 0.001), (650.25, 0.05), (-25.0, 0.001), (650.25, 0.01), (3.1, 1.0)])
@pytest.mark.parametrize("ties", [600, 1025, 1500, 4096, 6000])
def test_ties_that_a_rounded_product_leaves_at_a_bins_edge(value, temp, ties):
    """More entries of the decisive bin than are put in order, far from 0, where x / T lies a rounding above a bin's edge."""
    from cwm_amd import ops

    vocab = 20000
    g = torch.Generator().manual_seed(ties)
    base = torch.tensor(value)
    step = base.abs() * 2.0 ** -22  # a few units of the last place
    row = torch.full((vocab,), value - 60 * temp)
    order = torch.randperm(vocab, generator=g)
    row[order[:ties]] = base
    row[order[ties : 2 * ties]] = base + step  # in the same bin, in another part or the same
    row[order[2 * ties]] = value + 2 * temp
    n = 24
    us, tops = torch.rand(n, generator=g), torch.tensor([0.2, 0.5, 0.999]).repeat(n // 3)
    temps = torch.full((n,), temp)
    toks, lp, slp = (t.cpu() for t in ops.sample(row.repeat(n, 1).to(DEV), temps.to(DEV), tops.to(DEV), us.to(DEV)))
    x = (row.double() - row.double().max()) * float(1.0 / torch.tensor(temp))
    probs = torch.softmax(x, -1)
    values = torch.sort(probs, descending=True).values
    above = torch.cumsum(values, 0) - values
    for r in range(n):
        least = float(values[above <= float(tops[r])][-1])
        kept = torch.where(probs >= least * (1 - 1e-9), probs, torch.zeros_like(probs))
        cdf = torch.cumsum(kept / kept.sum(), 0)
        tok = int(toks[r])
        # the weights' exponents are float32 numbers of at most 60, and sums of thousands of equal weights are off by 1e-6
        assert kept[tok] > 0, (r, tok)
        assert float(cdf[tok] - kept[tok] / kept.sum()) <= float(us[r]) + 2e-5 and float(cdf[tok]) >= float(us[r]) - 2e-5, (r, tok)
        np.testing.assert_allclose(float(slp[r]), math.log(float(kept[tok] / kept.sum())), atol=2e-5)


@pytest.mark.parametrize("levels", [None, 6])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 255, 256, 257, 511, 513, 1024])
def test_the_nucleus_ends_in_a_bin_of_so_many_entries(count, levels):
    """At the numbers of entries where the way of putting them in order changes, all different and with ties."""
    from cwm_amd import ops

    vocab, n = 32768, 64
    g = torch.Generator().manual_seed(count)
    within = torch.rand(count, generator=g)
    if levels:
        within = torch.floor(within * levels) / levels
    logits = torch.full((vocab,), -20.0)  # all others together: 32768 exp(-29.9), below 1e-8 of the mass
    where = torch.randperm(vocab, generator=g)[:count]
    logits[where] = (115.05 + 0.9 * within) * (math.log(2.0) / 8.0)  # one eighth of an octave, away from its edges
    us = (torch.arange(n) + 0.5) / n
    args = [logits.expand(n, vocab).contiguous(), torch.ones(n), torch.full((n,), 0.6), us]
    toks, _, slp = (t.cpu() for t in ops.unpack_sampled(ops.sample_packed(*(t.to(DEV) for t in args))))
    probs = torch.softmax(logits.double(), -1)
    values = torch.sort(probs, descending=True).values
    above = torch.cumsum(values, 0) - values
    # 2^-24 for each of the at most 12 additions that a mass goes through and for the exponential: 1e-6 of the target
    kept = [probs >= float(values[above <= 0.6 + off][-1]) * (1 - 1e-6) for off in (-1e-6, 1e-6)]
    least, most = (float((probs * k).sum()) for k in kept)
    for u, tok, s in zip(us.tolist(), toks.tolist(), slp.tolist()):
        assert bool(kept[1][tok])
        assert math.log(float(probs[tok]) / most) - 1e-5 <= s <= math.log(float(probs[tok]) / least) + 1e-5
        upto = torch.cumsum(probs * kept[1], 0)
        slack = 1e-5 + (most - least) / least  # an entry at the threshold may be in or out
        assert float(upto[tok] - probs[tok]) / most <= u + slack and float(upto[tok]) / most >= u - slack
