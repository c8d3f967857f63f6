"""Norms of rows around the widths at which a block's number of threads and elements a thread change, with numbers of partial
sums and of experts' rows around the four that are under way at a time, and around the number of rows that takes other blocks."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
WIDTHS = [4, 252, 260, 1024, 1028, 4092, 4096, 4100, 8192]
SLABS = [1, 2, 4, 5, 9]


def drawn(dim, slabs, rows):
    g = torch.Generator(device=DEV).manual_seed(dim + slabs)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    return normal(rows, dim), normal(slabs, rows, dim), 1 + 0.1 * normal(dim)


def check(got, want, size):
    # float32: a few units of 2^-24 for the serial part of each sum and the logarithmic rest, relative to the terms' size
    # (a sum of slabs may cancel)
    assert bool(((got.double() - want).abs() <= 2.0 ** -18 * size + 1e-6).all())


@pytest.mark.parametrize("dim", WIDTHS)
@pytest.mark.parametrize("slabs", SLABS)
def test_sums_and_norms(dim, slabs):
    from cwm_amd import ops

    for rows in (1, 3, 600):
        h, parts, w = drawn(dim, slabs, rows)
        x = h.double() + parts.double().sum(0)
        size = h.double().abs() + parts.double().abs().sum(0)
        scale = torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5)
        pending = parts if slabs > 1 else parts[0]
        kept = h.clone()
        check(ops.add_rmsnorm(kept, pending, w, 1e-5, torch.float32), x * scale * w, size * scale * w.abs())
        check(kept, x, size)
        kept = h.clone()
        check(ops.stream_mix_norm(kept, 1, pending, None, None, None, w, 1e-5, torch.float32), x * scale * w, size * scale * w.abs())
        check(kept, x, size)
        kept, bias = h.clone(), w.flip(0).contiguous()
        out = ops.add_layernorm(kept, ops.ScaledSum([(pending, 1.0)]), w, bias, 1e-5, torch.float32)
        d = x - x.mean(-1, keepdim=True)
        scale = torch.rsqrt((d * d).mean(-1, keepdim=True) + 1e-5)
        check(out, d * scale * w + bias, (size + size.mean(-1, keepdim=True)) * scale * w.abs() + bias.abs())
        check(kept, x, size)


@pytest.mark.parametrize("top", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("dim", [1024, 1028, 4100])
def test_a_sum_of_experts_rows_is_the_combined_one(dim, top):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(top)
    for tokens in (1, 7):
        chosen = torch.rand((tokens, 16), generator=g, device=DEV).argsort(-1)[:, :top].int().contiguous()
        groups = ops.group_by_expert(chosen, 16)
        groups.pair_row[top - 1] = -1  # a choice that names no row
        rows = torch.randn((groups.n_tiles * 16, dim), generator=g, device=DEV)
        weights = torch.rand((tokens, top), generator=g, device=DEV)
        pending = ops.RoutedSum(rows, groups, weights)
        h, w = torch.randn((tokens, dim), generator=g, device=DEV), torch.ones(dim, device=DEV)
        one, two = h.clone(), h.clone()
        a = ops.stream_mix_norm(one, 1, pending, None, None, None, w, 1e-5, torch.float32)
        b = ops.stream_mix_norm(two, 1, pending.combine(), None, None, None, w, 1e-5, torch.float32)
        assert torch.equal(one, two) and torch.equal(a, b)


@pytest.mark.parametrize("heads,slabs", [((4, 1), 1), ((6, 2), 5), ((40, 8), 4)])
def test_queries_and_keys_share_no_sum(heads, slabs):
    """Queries and keys normalised over their whole projections, where a block has more and fewer threads than pieces."""
    from cwm_amd import ops

    nq, nk = heads
    g = torch.Generator(device=DEV).manual_seed(nq)
    for tokens in (3, 520):
        parts = torch.randn((slabs, tokens, (nq + 2 * nk) * 128), generator=g, device=DEV)
        qw, kw = (1 + 0.1 * torch.randn((n * 128,), generator=g, device=DEV) for n in heads)
        positions = torch.arange(tokens, device=DEV, dtype=torch.int32)
        cache = torch.zeros((-(-tokens // 16), 2, nk, 16 * 128), device=DEV)
        table = torch.arange(cache.shape[0], device=DEV, dtype=torch.int32)[None]
        q = ops.qk_norm_rope_write(parts if slabs > 1 else parts[0], nq, nk, 128, 128, 128, qw, kw, 1e-5, positions, None, torch.float32, cache, table,
                                   torch.zeros(tokens, device=DEV, dtype=torch.int32))
        x, size = parts.double().sum(0), parts.double().abs().sum(0)
        for got, at, w in ((q.reshape(tokens, -1), 0, qw), (cache[:, 0].reshape(-1, nk, 16, 128).permute(0, 2, 1, 3).reshape(-1, nk * 128)[:tokens], nq * 128, kw)):
            n = w.numel()
            scale = torch.rsqrt((x[:, at : at + n] ** 2).mean(-1, keepdim=True) + 1e-5)
            check(got, x[:, at : at + n] * scale * w, size[:, at : at + n] * scale * w.abs())
