"""Blocks of 64 rows in the attention of few long portions: which steps take them, their work lists, and their bits."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from cwm_amd.ops.attention_plan import WIDE_TILES, build_plan, wide_item_tiles

DEV = "cuda:0"


@pytest.mark.parametrize("q,kv,tiles", [
    ([129], [129], 4), ([128], [128], 8), ([1, 1], [900, 30], 8), ([2048], [2048], 4), ([300, 1], [300, 5000], 4),
    ([300], [2049], 8), ([16384], [16384], 8), ([6000], [6000], 8), ([300, 130], [300, 40000], 8),
])
def test_which_steps_take_halves(q, kv, tiles):
    assert wide_item_tiles(q, kv, 1, 16, 128, 32, 256) == tiles
    assert wide_item_tiles(q, kv, 1, 16, 96, 32, 256) == WIDE_TILES  # not built


@pytest.mark.parametrize("q,kv,group,window,chunk", [([129, 1, 700], [129, 40, 1900], 1, None, None), ([65, 400], [65, 1000], 3, 100, None), ([500], [777], 2, None, 128)])
def test_halves_cover_the_same_rows_and_keys(q, kv, group, window, chunk):
    whole, halves = (build_plan(q, kv, group, window, 0, chunk, wide_tiles=t) for t in (8, 4))
    assert np.array_equal(whole.work, halves.work) and halves.n_partials == whole.n_partials
    rows = lambda plan, t: {(b, r) for b, r0, *_ in plan.work_wide.tolist() for r in range(r0, min(r0 + 16 * t, q[b] * group))}  # noqa: E731
    assert rows(whole, 8) == rows(halves, 4) == {(b, r) for b, n in enumerate(q) if n * group > 128 for r in range(n * group)}
    spans = {(b, r0 // 128): (lo, hi) for b, r0, lo, hi, *_ in whole.work_wide.tolist()}
    for b, r0, lo, hi, slot, _ in halves.work_wide.tolist():
        assert spans[b, r0 // 128][0] <= lo < hi <= spans[b, r0 // 128][1] and slot < 0
        assert hi == kv[b] - q[b] + (min(r0 + 64, q[b] * group) - 1) // group + 1


@pytest.mark.gpu
@pytest.mark.parametrize("hd,n_q,n_kv", [(64, 4, 2), (128, 3, 1), (256, 2, 1)])
@pytest.mark.parametrize("page", [32, 256])
@pytest.mark.parametrize("mask", [{}, {"window": 90}, {"chunk": 64}, {"softcap": 5.0}, {"sink": True}])
def test_the_same_bits(hd, n_q, n_kv, page, mask, monkeypatch):
    from cwm_amd import ops

    new, old = [129, 1, 260, 63, 200], [0, 300, 37, 70, 1801]
    lens = [a + b for a, b in zip(new, old)]
    g = torch.Generator(device=DEV).manual_seed(hd + page)
    per = [-(-n // page) for n in lens]
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32)
    order, used = torch.randperm(sum(per), generator=torch.Generator().manual_seed(1)).int(), 0
    for i, p in enumerate(per):
        table[i, :p] = order[used : used + p]
        used += p
    cache = torch.randn((sum(per), 2, n_kv, page * hd), generator=g, device=DEV).bfloat16()
    q = torch.randn((sum(new), n_q, hd), generator=g, device=DEV).bfloat16()
    mask = {k: torch.randn(n_q, generator=g, device=DEV) if k == "sink" else v for k, v in mask.items()}
    cu = torch.tensor([0, *np.cumsum(new)], dtype=torch.int32, device=DEV)
    window = mask.pop("window", None)

    def run():
        batch = SimpleNamespace(q_lens=new, kv_lens=lens, n_seqs=len(new), n_tokens=sum(new), scratch={}, cu_q=cu, kv_len=torch.tensor(lens, dtype=torch.int32, device=DEV))
        return ops.paged_attention_mfma(q, cache, table.to(DEV), batch, window, hd ** -0.5, **mask)

    from cwm_amd.ops import attention_plan

    halves = run()
    monkeypatch.setattr(attention_plan, "WIDE_HALF_BLOCKS", {})
    assert torch.equal(halves, run()) and bool(torch.isfinite(halves).all())
