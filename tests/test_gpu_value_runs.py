"""Values of many tokens written a value block at a time, where the heads are many enough: the bits of calls of few tokens, which write
each token's own."""

import pytest
import torch

from cwm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (first position, tokens) of each sequence in a step of 512 tokens and more: one that fits the windows of eight tokens, starts
# inside a value block and ends inside one, decoded tokens before and between (which shift the windows), runs shorter than a block
STEPS = [[(0, 512)], [(5, 523)], [(7, 1), (30, 1), (0, 300), (11, 1), (3, 221)], [(1, 7), (8, 8), (3, 13), (0, 505), (16, 7)]]


@pytest.mark.parametrize("step", STEPS)
@pytest.mark.parametrize("page", [8, 24, 12])
@pytest.mark.parametrize("n_kv,qk,vd,hd,kind", [(4, 128, 128, 128, "rows"), (1, 20, 12, 32, "mixed"), (3, 64, 64, 64, "partials"), (2, 4, 4, 4, "rows"),
                                                  (16, 20, 12, 32, "mixed"), (8, 64, 64, 64, "partials"), (128, 4, 4, 4, "rows")])
def test_the_bits_of_few_tokens(step, page, n_kv, qk, vd, hd, kind):
    n_q, total = 2, sum(n for _, n in step)
    g = torch.Generator(device=DEV).manual_seed(total + page + hd)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    width = (n_q + n_kv) * qk + n_kv * vd
    src = normal(3, total, width) if kind == "partials" else normal(total, width + 4).bfloat16()[:, :width]
    other = normal(total, n_kv * vd + 4).bfloat16()[:, : n_kv * vd] if kind == "mixed" else None
    mix = torch.tensor([0.375], device=DEV) if kind == "mixed" else None
    bias, weight, inv_freq = normal(width), normal(qk).abs(), 0.01 * normal(hd // 2).abs()
    wide = max((p + n + page - 1) // page for p, n in step)
    table = torch.randperm(len(step) * wide, generator=g, device=DEV).int().reshape(len(step), wide)
    table[0, 1 if wide > 1 else 0] = -1  # tokens of a page that is not there are left out
    positions = torch.cat([torch.arange(p, p + n, device=DEV) for p, n in step]).int()
    seq = torch.cat([torch.full((n,), i, device=DEV) for i, (_, n) in enumerate(step)]).int()

    def run(cache, lo, hi):
        rows = src[:, lo:hi].contiguous() if kind == "partials" else src[lo:hi]
        return ops.head_norm_rope_write(rows, n_q, n_kv, qk, vd, hd, bias, weight, weight, 1e-5, positions[lo:hi], inv_freq, torch.bfloat16, cache, table, seq[lo:hi],
                                        v_other=None if other is None else other[lo:hi], v_mix=mix, keep_values=True)

    lib = ops._build.load("rope_kv")
    assert not lib.cwm_value_runs_pay(100, 1, n_q, n_kv, hd) and bool(lib.cwm_value_runs_pay(total, len(step), n_q, n_kv, hd)) == (n_kv * hd >= 512)
    caches = [torch.full((table.numel(), 2, n_kv, hd * page), 9.0, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    q, kept = run(caches[0], 0, total)
    parts = [run(caches[1], lo, min(lo + 100, total)) for lo in range(0, total, 100)]
    assert torch.equal(caches[0], caches[1])
    assert torch.equal(q, torch.cat([p[0] for p in parts])) and torch.equal(kept, torch.cat([p[1] for p in parts]))
