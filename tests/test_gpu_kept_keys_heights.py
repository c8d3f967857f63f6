"""Kept first keys beside a window: a row's bits do not depend on what else is in the step (which decides on the height of the
blocks of long portions), also where a block's first key lies among the kept ones' first tile."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("window,keep", [(50, 16), (34, 5), (64, 40), (90, 70)])
def test_a_portion_alone_and_among_many(hd, window, keep):
    """192 tokens alone, and beside a portion long enough that the launch has more blocks than 64-row ones would be taken for;
    with these windows a block of 64 rows would start at keys 1 to 31 where the one of 128 starts at 0."""
    from cwm_amd import ops

    n_kv, page, portion = 16, 32, 192
    outs = []
    for other in (0, 8192):
        new = [portion] + [other] * (other > 0)
        per = [n // page for n in new]
        g = torch.Generator(device=DEV).manual_seed(hd + window)
        cache = torch.randn((6, 2, n_kv, page * hd), generator=g, device=DEV).bfloat16()
        q = torch.randn((portion, n_kv, hd), generator=g, device=DEV).bfloat16()
        table = torch.full((len(new), max(per)), -1, dtype=torch.int32)
        table[0, : per[0]] = torch.arange(6, dtype=torch.int32)
        if other:
            cache = torch.cat([cache, torch.randn((per[1], 2, n_kv, page * hd), generator=g, device=DEV).bfloat16()])
            q = torch.cat([q, torch.randn((other, n_kv, hd), generator=g, device=DEV).bfloat16()])
            table[1] = 6 + torch.arange(per[1], dtype=torch.int32)
        cu = torch.tensor([0, *np.cumsum(new)], dtype=torch.int32, device=DEV)
        batch = SimpleNamespace(q_lens=new, kv_lens=new, n_seqs=len(new), n_tokens=sum(new), scratch={}, cu_q=cu, kv_len=torch.tensor(new, dtype=torch.int32, device=DEV))
        outs.append(ops.paged_attention_mfma(q, cache, table.to(DEV), batch, window, hd ** -0.5, keep_first=keep)[:portion])
    assert torch.equal(*outs) and bool(torch.isfinite(outs[0]).all())
