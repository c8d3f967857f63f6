"""The streaming product with 9 to 32 rows: its block of two row tiles, the fused epilogues on it, and which sizes go to it."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def drawn(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    return normal(m, k).bfloat16(), (normal(n, k) * k ** -0.5).bfloat16()


def rounded(got, want):
    # one rounding to bfloat16 (half a unit, 2^-9 of the binade's top) after float32 sums of values of order one
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13).all())


@pytest.mark.parametrize("m", [16, 17, 31, 32])
@pytest.mark.parametrize("k", [64, 2048, 2056, 3072])
def test_fused_epilogues(m, k):
    from cwm_amd import ops

    n_q, n_kv, hd = 3, 1, 64
    x, w = drawn(m, (n_q + 2 * n_kv) * hd, k)
    positions = torch.arange(m, device=DEV, dtype=torch.int32) * 7 % 61
    seq = torch.arange(m, device=DEV, dtype=torch.int32)
    table = torch.arange(4 * m, device=DEV, dtype=torch.int32).reshape(m, 4)
    freq = torch.rand(hd // 2, device=DEV)
    caches = [torch.zeros((4 * m, 2, n_kv, 16 * hd), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    rope = (positions, seq, freq, caches[0], table, n_q, n_kv, hd)
    fused = ops.gemm_bf16_stream(x, torch.full_like(w, float("nan")), None, torch.bfloat16, rope=rope, streamed=ops.stream_layout(w))
    apart = ops.gemm_bf16_stream(x, w)  # the same sums where K is not split, by other roundings where it is
    rounded(apart, x.double() @ w.double().T)
    q, kk, v = (apart[:, a * hd : b * hd].unflatten(1, (-1, hd)) for a, b in ((0, n_q), (n_q, n_q + n_kv), (n_q + n_kv, n_q + 2 * n_kv)))
    ops.rope_kv_write(q, kk, v, positions, freq, caches[1], table, seq)
    if k <= 2048:
        assert torch.equal(fused, apart) and torch.equal(caches[0], caches[1])
    else:  # rotated sums of two values, each off by a unit at most
        size = apart.abs().float().unflatten(1, (-1, 2)).sum(-1, keepdim=True).expand(-1, -1, 2).flatten(1)
        assert bool(((fused.float() - apart.float()).abs() <= 2.0 ** -6 * size + 2.0 ** -12).all())

    x, w = drawn(m, 2 * 40, k)
    got = ops.gemm_bf16_stream(x, torch.full_like(w, float("nan")), None, torch.bfloat16, glu=True, streamed=ops.stream_layout(w))
    both = (x.double() @ w.double().T).reshape(m, -1, 2, 8)
    both = ops.gemm_bf16_stream(x, w).double().reshape(m, -1, 2, 8) if k <= 2048 else both
    want = (torch.nn.functional.silu(both[:, :, 0]) * both[:, :, 1]).reshape(m, -1)
    # gate and up are rounded first: where K is split they may each be off by a unit
    assert bool(((got.double() - want).abs() <= 2.0 ** (-8 if k <= 2048 else -5) * (want.abs() + 2.0 ** -5)).all())


@pytest.mark.parametrize("m", [9, 16, 17, 32, 33])
def test_which_products_stream(m):
    from cwm_amd import ops

    for n, k, streams in ((208, 128, False), (256, 512, True), (1024, 512, True), (1 << 12, (1 << 13) + 64, False), ((1 << 15) - 16, 1 << 12, m <= 16)):
        x, w = drawn(m, n, k)
        copy = ops.stream_layout(w)
        got = ops.linear(x, w, None, torch.float32, partials_ok=True, streamed=copy)
        tiled = ops.gemm_bf16_tile(x, w, None, torch.float32, partials_ok=True)
        chosen = ops.gemm_bf16_stream(x, w, None, torch.float32, partials_ok=True, streamed=copy) if m <= 32 and streams else tiled
        assert torch.equal(got, chosen)
        without = ops.linear(x, w, None, torch.float32, partials_ok=True)
        assert torch.equal(without, chosen if n * k < 1 << 22 else tiled)


@pytest.mark.parametrize("m", [9, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(512, 64), (320, 512), (768, 1088), (1024, 4032), (256, 8192)])
def test_a_copy_changes_no_bit_below_its_limit(m, n, k):
    """Every way a product of these sizes is called: plain, as partial sums, with the gate, with the rotation and cache write."""
    from cwm_amd import ops

    x, w = drawn(m, n, k)
    copy = ops.stream_layout(w)
    assert torch.equal(ops.linear(x, w), ops.linear(x, w, streamed=copy))
    assert torch.equal(ops.linear(x, w, None, partials_ok=True), ops.linear(x, w, None, partials_ok=True, streamed=copy))
    assert torch.equal(ops.gate_up_silu(x, w, None, True), ops.gate_up_silu(x, w, None, True, streamed=copy))
    hd, n_kv = 32, n // 128
    positions = torch.arange(m, device=DEV, dtype=torch.int32) % 16
    seq = torch.arange(m, device=DEV, dtype=torch.int32)
    caches = [torch.zeros((m, 2, n_kv, 16 * hd), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    wq = w[: 4 * n_kv * hd].contiguous()
    got = [ops.qkv_rope_write(x, wq, None, 2 * n_kv, n_kv, hd, positions, torch.rand(hd // 2, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)),
                              cache, seq[:, None].contiguous(), seq, streamed=s) for cache, s in zip(caches, (None, ops.stream_layout(wq)))]
    assert torch.equal(*got) and torch.equal(*caches)
