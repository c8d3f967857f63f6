"""Portions of a prompt whose heads mix their weights without a table in memory: every room for heads and share of a wavefront, edges
of tiles and ranges, windows, several portions beside short ones and decoded tokens, and more portions than one launch takes."""

from __future__ import annotations

import pytest
import torch

from test_gpu_digasun import DEV, _talking_case

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_portion_in_tiles(monkeypatch):
    """Sizes that the rule leaves to the table of scores and the library's products as well."""
    from cwm_amd.ops import mixing

    monkeypatch.setattr(mixing, "talk_tiles_take", lambda tokens, keys, groups, n_q, n_kv, hd: groups > 0 and tokens >= mixing.TALK_TILE_FROM)


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
    gone[0, 15] = cache.shape[0]  # keys 480..511, out of range: rows 80 to 199 read one or more
    got = ops.talking_attention(q, cache, gone, batch, 100, scale, sink=sink, talk=mix)
    assert torch.isnan(got[80:]).all() and torch.isfinite(got[:80]).all()


def _value_of(cache, table, b, key, n_kv, hd):
    """The place of a key's values in the cache, [Hkv, hd]."""
    page = cache.shape[3] // hd
    slot = key % page
    return cache[int(table[b, key // page]), 1].view(n_kv, page // 8, hd, 8)[:, slot // 8, :, slot % 8]


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("n_q,n_kv,hd,old,new,window", [(16, 8, 128, 5, 40, None), (8, 4, 64, 70, 100, 33), (24, 8, 128, 40, 130, 64), (9, 3, 128, 0, 16, None), (20, 4, 64, 300, 77, 1)])
def test_a_value_that_is_not_finite_reaches_its_readers_only(bad, n_q, n_kv, hd, old, new, window):
    """One element of one token's values: of the heads and elements that it lies in, the rows that read the token are not
    finite; all else keeps its bits."""
    from cwm_amd import ops

    case = _talking_case(torch.bfloat16, n_q, n_kv, hd, 64, [old], [new], window, seed=n_q + new)
    q, cache, table, batch, scale, sink, mix, want = case
    clean = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu()
    key, head, d, per = old + new * 2 // 3, n_kv - 1, hd - 3, n_q // n_kv
    _value_of(cache, table, 0, key, n_kv, hd)[head, d] = bad
    got = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu()
    at = torch.arange(old, old + new)
    reads = (at >= key) & (at - key < (window if window is not None else old + new))
    assert reads.any() and not reads.all()
    there = torch.zeros((n_q, hd), dtype=torch.bool)
    there[head * per :, d] = True
    there = there.flatten()
    assert not torch.isfinite(got[reads][:, there]).any()
    assert torch.equal(got[~reads], clean[~reads])
    assert torch.equal(got[:, ~there][reads], clean[:, ~there][reads])


@pytest.mark.parametrize("place", ["q", "k"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_queries_and_keys_that_are_not_finite(place, bad):
    from cwm_amd import ops

    n_q, n_kv, hd, old, new, window = 16, 8, 128, 20, 90, 48
    q, cache, table, batch, scale, sink, mix, want = _talking_case(torch.bfloat16, n_q, n_kv, hd, 64, [old], [new], window, seed=4)
    clean = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu()
    key = old + 50
    if place == "q":
        q[50, 3, 7] = bad
    else:
        cache[int(table[0, key // 64]), 0].view(n_kv, 64, hd)[2, key % 64, 7] = bad
    got = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix).cpu()
    at = torch.arange(old, old + new)
    reads = at == key if place == "q" else (at >= key) & (at - key < window)
    assert torch.equal(got[~reads], clean[~reads])
    if place == "q" or bad != bad:
        assert torch.isnan(got[reads]).all()  # every head has a share of the bad one's weights
    else:  # a score of an infinity either way: all weight or none
        assert bool((~torch.isfinite(got[reads])).any())


def test_a_block_table_that_ends_before_the_last_key():
    """The rows whose keys the table does not reach have no result, the others theirs; nothing is refused."""
    from cwm_amd import ops

    for new in (40, 200):
        q, cache, table, batch, scale, sink, mix, want = _talking_case(torch.bfloat16, 8, 4, 64, 32, [100], [new], None, seed=6)
        whole = ops.talking_attention(q, cache, table, batch, None, scale, sink=sink, talk=mix)
        pages = 4  # keys 0..127: rows 0..27
        got = ops.talking_attention(q, cache, table[:, :pages].contiguous(), batch, None, scale, sink=sink, talk=mix)
        assert torch.isnan(got[28:]).all() and torch.equal(got[:28], whole[:28])


@pytest.mark.parametrize("new", [20, 150])
def test_scales_that_are_not_positive(new):
    """Scores of minus the scale are those of minus the queries; a scale of zero gives all keys the same score."""
    from cwm_amd import ops

    q, cache, table, batch, scale, sink, mix, want = _talking_case(torch.bfloat16, 8, 4, 64, 32, [100], [new], 60, seed=7)
    got = ops.talking_attention(-q, cache, table, batch, 60, -scale, sink=sink, talk=mix).cpu().double()
    torch.testing.assert_close(got, want, rtol=3e-2, atol=3e-2)
    none = ops.talking_attention(q, cache, table, batch, 60, 0.0, sink=sink, talk=mix)
    zero = ops.talking_attention(torch.zeros_like(q), cache, table, batch, 60, scale, sink=sink, talk=mix)
    torch.testing.assert_close(none.float(), zero.float(), rtol=2 ** -6, atol=2 ** -6)  # bfloat16 weights and results


@pytest.mark.parametrize("n_q,n_kv,hd,lens_old,lens_new,window", [
    (16, 8, 128, [300, 31], [700, 143], None), (16, 8, 128, [300, 31], [143, 700], 64), (24, 8, 64, [0, 100], [333, 200], None), (24, 8, 128, [40, 5], [97, 260], 50),
])
def test_portions_over_several_launches(n_q, n_kv, hd, lens_old, lens_new, window, monkeypatch):
    """A table of weights that holds a few tiles of rows: the portions go over many launches, with the bits of one."""
    from cwm_amd import ops
    from cwm_amd.ops import mixing

    q, cache, table, batch, scale, sink, mix, want = _talking_case(torch.bfloat16, n_q, n_kv, hd, 64, lens_old, lens_new, window, seed=n_q + sum(lens_new))
    lib, launches = mixing._build.load("attention_talk_tile"), []

    class Counting:
        def __getattr__(self, name):
            return getattr(lib, name)

        def cwm_talking_tiles(self, *args):
            launches.append(args)
            return lib.cwm_talking_tiles(*args)

    mixing._build._loaded["attention_talk_tile"] = Counting()
    try:
        whole = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix)
        assert len(launches) == 1
        for table_bytes in (1, 300_000, 1_000_000):
            monkeypatch.setattr(mixing, "TALK_TABLE_BYTES", table_bytes)
            del launches[:]
            got = ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix)
            assert len(launches) > 1, table_bytes
            assert torch.equal(got, whole), table_bytes
        monkeypatch.setattr(mixing, "TALK_TABLE_BYTES", 1)
        del launches[:]
        ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix)
        assert len(launches) == sum(-(-n // 32) for n in lens_new)  # a tile of rows each
    finally:
        mixing._build._loaded["attention_talk_tile"] = lib


@pytest.mark.parametrize("n_q,n_kv,hd,old,new,window", [(16, 8, 128, 77, 130, None), (24, 8, 64, 300, 45, 64), (9, 3, 128, 0, 16, None)])
def test_without_a_sink(n_q, n_kv, hd, old, new, window):
    """A sink far below every score adds nothing, so it gives the bits of none; a quiet one gives others."""
    from cwm_amd import ops

    case = _talking_case(torch.bfloat16, n_q, n_kv, hd, 64, [old], [new], window, seed=n_q)
    q, cache, table, batch, scale, sink, mix, want = case
    none = ops.talking_attention(q, cache, table, batch, window, scale, sink=None, talk=mix)
    low = ops.talking_attention(q, cache, table, batch, window, scale, sink=torch.full_like(sink, -1e30), talk=mix)
    assert torch.equal(none, low)
    assert not torch.equal(none, ops.talking_attention(q, cache, table, batch, window, scale, sink=sink, talk=mix))
