"""Row-wise passes of 16 bytes a lane against the same passes on rows that start off such a boundary, and against float64."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _normal(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return lambda *shape: torch.randn(shape, generator=g, device=DEV)


@pytest.mark.parametrize("n_tokens", [1, 7, 8, 9, 600])
@pytest.mark.parametrize("n_q,n_kv,qk,vd,hd,source", [(16, 4, 128, 128, 128, torch.bfloat16), (3, 1, 20, 8, 32, torch.bfloat16), (5, 2, 256, 192, 256, torch.float32), (6, 3, 64, 64, 64, None)])
def test_head_norm_rope_write(n_tokens, n_q, n_kv, qk, vd, hd, source):
    from cwm_amd import ops

    normal = _normal(n_tokens + hd)
    width, page, dtype = (n_q + n_kv) * qk + n_kv * vd, 16, torch.float32 if source == torch.float32 else torch.bfloat16
    src = normal(3, n_tokens, width) if source is None else normal(n_tokens, width + 8).to(source)[:, :width]
    # the same rows one element off the boundary: the pass of one element a load
    off = torch.empty(n_tokens, width + 9, device=DEV, dtype=torch.float32 if source is None else source)[:, 1 : 1 + width]
    off.copy_(src.sum(0) if source is None else src)
    bias, wq, wk = normal(width), normal(qk).abs() + 0.2, normal(qk).abs() + 0.2
    positions = torch.arange(5, 5 + n_tokens, device=DEV, dtype=torch.int32)
    n_pages = (n_tokens + 5 + page - 1) // page
    table = torch.arange(n_pages, device=DEV, dtype=torch.int32).flip(0).reshape(1, -1).contiguous()
    seq = torch.zeros(n_tokens, device=DEV, dtype=torch.int32)
    other, mix = normal(n_tokens, n_kv * vd).to(dtype), torch.tensor([0.375], device=DEV)
    inv_freq = torch.where(torch.arange(hd // 2, device=DEV) < qk // 4, 0.01 * normal(hd // 2).abs(), torch.zeros(hd // 2, device=DEV))

    def run(rows):
        cache = torch.zeros(n_pages, 2, n_kv, hd * page, device=DEV, dtype=dtype)
        q, kept = ops.head_norm_rope_write(rows, n_q, n_kv, qk, vd, hd, bias, wq, wk, 1e-5, positions, inv_freq, dtype, cache, table, seq, v_other=other,
                                           v_mix=mix, keep_values=True, temperature=(0.1, 64))
        return q, cache, kept

    # float32 sums of a head's squares in another order, the partial sums' rounding: a few units of 2^-24 of values up to about
    # 10, which may round to the neighbouring bfloat16 value (a step of 2^-7 of it)
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 0.0
    for got, want in zip(run(src), run(off)):
        assert bool(((got.float() - want.float()).abs() <= step * want.float().abs() + 2e-5).all())
        assert float((got.float() - want.float()).abs().mean()) <= 2e-4 * float(want.float().abs().mean()) + 1e-7


@pytest.mark.parametrize("rows,hidden", [(1, 1 << 20), (1, (1 << 20) - 8), (1033, 1024), (4100, 264)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.float32, torch.float32)])
def test_activations_are_the_same_bits(rows, hidden, dtype, out_dtype):
    from cwm_amd import ops

    normal = _normal(rows)
    x = normal(rows, hidden).to(dtype)
    off = torch.empty(rows * hidden + 1, device=DEV, dtype=dtype)[1:].view(rows, hidden)
    off.copy_(x)
    for kind in ("relu2", "silu"):
        assert torch.equal(ops.act_rows(x, kind, out_dtype), ops.act_rows(off, kind, out_dtype))
    gated = normal(rows, 2 * hidden + 8).to(dtype)
    off = torch.empty(rows, 2 * hidden + 9, device=DEV, dtype=dtype)[:, : 2 * hidden + 8]
    off.copy_(gated)
    for activation in (ops.GatedActivation(), ops.GatedActivation("clamped_swish", 1.7, 1.0)):
        for column in (None, 2 * hidden + 3):
            assert torch.equal(ops.gated_act_rows(gated, hidden, activation, out_dtype, column), ops.gated_act_rows(off, hidden, activation, out_dtype, column))
    if dtype == torch.float32:
        partials = normal(3, rows, hidden)
        want = torch.relu((partials[0] + partials[1]) + partials[2]).square().to(out_dtype)
        assert torch.equal(ops.act_rows(partials, "relu2", out_dtype), want)


@pytest.mark.parametrize("top", [1, 3, 4, 6])
@pytest.mark.parametrize("n_tokens,dim", [(1, 4), (5, 1020), (33, 2052)])
def test_combined_rows(top, n_tokens, dim):
    from cwm_amd.ops import routed

    normal = _normal(top + dim)
    rows, weights = normal(n_tokens * top, dim), normal(n_tokens, top)
    pair_row = torch.randperm(n_tokens * top, device=DEV).int()
    pair_row[torch.rand(n_tokens * top, device=DEV) < 0.3] = -1  # choices whose expert is elsewhere
    got = routed.combine_routed(rows, SimpleNamespace(pair_row=pair_row, top=top), weights)
    chosen = rows.double()[pair_row.clamp(min=0).long()] * (pair_row >= 0).double()[:, None]
    terms = chosen.view(n_tokens, top, dim) * weights.double()[:, :, None]
    # `top` float32 products and sums, each within half a unit (2^-24) of what it adds up
    assert bool(((got.double() - terms.sum(1)).abs() <= top * 2.0 ** -24 * 1.01 * terms.abs().sum(1)).all())
