"""Portions of a prompt whose heads mix their weights without a table in memory: every room for heads and share of a wavefront, edges
of tiles and ranges, windows, several portions beside short ones and decoded tokens, and more portions than one launch takes."""

from __future__ import annotations

import pytest
import torch

from test_gpu_digasun import DEV, _talking_case

pytestmark = pytest.mark.gpu


def _bound(case, window):
    """What the kernels' roundings can add up to, float64 [T, H * hd]: the mixed weights and the result in bfloat16 (seven bits after
    the first: half of the last is at most 2^-8 of the value) and, far below them, float32 scores, exponentials and sums (2^-15 of the unmixed weights' size)."""
    q, cache, table, batch, scale, sink, mix, want = case
    hd, n_q = q.shape[2], q.shape[1]
    n_kv, page, per = cache.shape[2], cache.shape[3] // hd, n_q // cache.shape[2]
    rows, t0 = [], 0
    for b, (n, kv) in enumerate(zip(batch.q_lens, batch.kv_lens)):
        pos = torch.arange(kv, device=DEV)
        pages, slots = table[b].long()[pos // page], pos % page
        k = cache[:, 0].view(-1, n_kv, page, hd)[pages, :, slots].double().permute(1, 2, 0)
        v = cache[:, 1].view(-1, n_kv, page // 8, hd, 8)[pages, :, slots // 8, :, slots % 8].double().abs().transpose(0, 1)
        s = torch.stack([q[t0 : t0 + n, h].double() @ k[h // per] for h in range(n_q)]) * scale
        at = torch.arange(kv - n, kv, device=DEV)[:, None]
        seen = (pos <= at) & (pos > (at - window if window is not None else -1))
        s = s.masked_fill(~seen, float("-inf"))
        top = torch.maximum(s.amax(-1), sink.double()[:, None])
        p = torch.exp(s - top[..., None])
        p = p / (p.sum(-1) + torch.exp(sink.double()[:, None] - top))[..., None]
        mixed, unmixed = (m.double() @ p.flatten(1) for m in (mix, mix.abs()))
        size = [torch.stack([w.reshape(p.shape)[h].abs() @ v[h // per] for h in range(n_q)], 1).reshape(n, -1) for w in (mixed, unmixed)]
        rows.append(2.0 ** -8 * size[0] + 2.0 ** -15 * size[1])
        t0 += n
    return torch.cat(rows).cpu() + 2.0 ** -7.99 * want.abs() + 1e-30


@pytest.mark.parametrize(
    "n_q,n_kv,hd,page_size,lens_old,lens_new,window",
    [
        (8, 8, 128, 32, [0], [128], None),
        (16, 8, 128, 256, [0, 77, 5], [1500, 1, 129], None),
        (16, 8, 128, 64, [300, 31], [143, 700], 64),
        (12, 4, 64, 64, [511], [257], None),
        (9, 3, 128, 64, [0, 1000], [160, 300], 129),
        (24, 8, 128, 256, [640], [400], None),
        (32, 8, 64, 32, [0, 33], [200, 128], 200),
        (20, 4, 64, 96, [100], [333], 1),
        (16, 1, 128, 64, [0], [255], None),
        (5, 5, 64, 32, [2000], [130], 513),
        (8, 8, 64, 32, [3 * i for i in range(18)], [16 + 7 * i for i in range(18)], None),
        (16, 8, 128, 256, [900, 0, 40], [16, 15, 33], None),
    ],
)
def test_portions_without_a_table(n_q, n_kv, hd, page_size, lens_old, lens_new, window):
    from cwm_amd import ops
    from cwm_amd.ops import mixing

    assert mixing._talk_tiles_built(n_q, n_kv, hd)
    case = _talking_case(torch.bfloat16, n_q, n_kv, hd, page_size, lens_old, lens_new, window, seed=n_q + hd)
    q, cache, table, batch, scale, sink, mix, want = case
    got = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu().double()
    long = torch.tensor([n >= mixing.TALK_TILE_FROM for n in lens_new]).repeat_interleave(torch.tensor(lens_new))
    assert bool(((got - want).abs() <= _bound(case, window))[long].all())
    again = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu().double()
    assert torch.equal(got, again)
    # a portion's bits are its own, whatever else the step holds
    if len(lens_new) > 1:
        b = max(range(len(lens_new)), key=lambda i: lens_new[i])
        t0 = sum(lens_new[:b])
        from test_gpu_digasun import step_batch

        alone = ops.talking_attention(q[t0 : t0 + lens_new[b]], cache, table[b : b + 1], step_batch([lens_old[b]], [lens_new[b]]), window, scale, sink=sink, talk=mix)
        assert torch.equal(alone.cpu().double(), got[t0 : t0 + lens_new[b]])


def test_a_missing_page_of_a_long_portion():
    from cwm_amd import ops

    q, cache, table, batch, scale, sink, mix, want = _talking_case(torch.bfloat16, 8, 4, 64, 32, [400], [200], 100, seed=2)
    gone = table.clone()
    gone[0, :9] = -1  # keys 0..287: before every row's window (301 on)
    got = ops.talking_attention(q, cache, gone, batch, 100, scale, sink=sink, talk=mix)
    assert torch.equal(got, ops.talking_attention(q, cache, table, batch, 100, scale, sink=sink, talk=mix))
    gone[0, 15] = cache.shape[0]  # keys 480..511, out of range: rows 80 to 199 read one or more (and rows of their tile of 32 may answer so too)
    got = ops.talking_attention(q, cache, gone, batch, 100, scale, sink=sink, talk=mix)
    assert torch.isnan(got[80:]).all() and torch.isfinite(got[:64]).all()
