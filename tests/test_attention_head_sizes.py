"""Layers of several head sizes in one step: each has the attention work list that its own size asks for."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from cwm_amd import ops
from cwm_amd.ops.attention_plan import WIDE_TILES

DEV = "cuda:0"


@pytest.mark.parametrize("first,second", [((64, 8), (96, 8)), ((96, 8), (64, 8)), ((128, 8), (96, 8)), ((256, 1), (192, 1)), ((64, 8), (128, 8))])
@pytest.mark.parametrize("q,halves", [([600], (64, 128, 256)), ([4000, 9000], (64,))])
def test_each_head_size_has_its_own_list(first, second, q, halves, monkeypatch):
    """Host arithmetic alone, on 256 stand-in compute units: blocks of 64 rows by the head size's own limit (up to 960 blocks of
    128 rows for 64, 691 for 128, none for 96 and 192), whichever layer asked first; 13,000 tokens are 824 blocks of eight
    heads, and one head alone has the keys of its 9,000 cut."""
    monkeypatch.setattr(ops, "_compute_units", lambda device: 256)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    monkeypatch.setattr(torch.Tensor, "to", lambda self, *args, **kwargs: self)
    batch = SimpleNamespace(q_lens=q, kv_lens=q, scratch={}, static=None)
    for hd, n_kv in (first, second, first):
        built = ops._half_blocks_built(n_kv, hd, 256)
        plan = ops._attention_plan(batch, 1, n_kv, hd, None, SimpleNamespace(type="cuda"), halves=built)
        tiles = WIDE_TILES // 2 if hd in halves else WIDE_TILES
        assert plan.item_tiles == tiles and built == (hd in (64, 128, 256))
        assert n_kv == 1 or plan.n_wide == sum(-(-n // (16 * tiles)) for n in q)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(128, 96), (64, 48), (256, 96), (64, 128)])
def test_two_head_sizes_share_a_batch(sizes):
    """One batch object for both layers, as in a step, against a batch object each."""
    new, old, page = [300, 1, 140], [0, 70, 33], 32
    lens = [a + b for a, b in zip(new, old)]
    per = [-(-n // page) for n in lens]
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32)
    for i, p in enumerate(per):
        table[i, :p] = torch.arange(sum(per[:i]), sum(per[: i + 1]), dtype=torch.int32)
    table = table.to(DEV)
    cu = torch.tensor([0, *np.cumsum(new)], dtype=torch.int32, device=DEV)

    def batch():
        return SimpleNamespace(q_lens=new, kv_lens=lens, n_seqs=len(new), n_tokens=sum(new), scratch={}, cu_q=cu, kv_len=torch.tensor(lens, dtype=torch.int32, device=DEV))

    shared = batch()
    for order in (sizes, sizes[::-1]):
        for hd in order:
            g = torch.Generator(device=DEV).manual_seed(hd)
            cache = torch.randn((sum(per), 2, 2, page * hd), generator=g, device=DEV).bfloat16()
            q = torch.randn((sum(new), 4, hd), generator=g, device=DEV).bfloat16()
            together, apart = (ops.paged_attention_mfma(q, cache, table, b, None, hd ** -0.5) for b in (shared, batch()))
            assert torch.equal(together, apart) and bool(torch.isfinite(together).all())
