"""A layer's token input on the matrix cores: numbers of tokens around a block's, side values that split the wavefronts evenly
and not, widths of few and many tiles, pending addends of either type."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_tokens", [255, 256, 257, 303, 4100])
@pytest.mark.parametrize("dim,side", [(64, 32), (192, 64), (2048, 64), (2112, 96), (4096, 128)])
def test_against_float64(n_tokens, dim, side):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(n_tokens + dim)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    vocab, column0 = 61, 24
    h, tokens = normal(n_tokens, dim), torch.randint(vocab, (n_tokens,), generator=g, device=DEV, dtype=torch.int32)
    gate, proj, table = normal(side, dim).mul(dim ** -0.5).bfloat16(), normal(dim, side).bfloat16(), normal(vocab, column0 + side + 8).bfloat16()
    weight = normal(dim).abs() + 0.3
    wide = normal(n_tokens, dim + 16).bfloat16()
    pending = ops.ScaledSum([(normal(2, n_tokens, dim), 1.0), (wide[:, 8 : 8 + dim], 0.5)])
    x = h.double() + sum(c * (t.double().sum(0) if t.dim() == 3 else t.double()) for t, c in pending.terms)
    args = (tokens, table, column0, gate, proj.t().contiguous(), weight, 1e-6, True)
    got, before = h.clone(), h.clone()
    ops.token_side(got, *args, pending=pending, w_proj=proj)
    ops.token_side(before, *args, pending=pending)
    z = (x.float().bfloat16().double() @ gate.double().T).float().bfloat16().double()
    e = table[tokens.long(), column0 : column0 + side].double()
    gated = (torch.nn.functional.gelu(z, approximate="tanh") * e).float().bfloat16().double()
    y = gated @ proj.double().T
    want = x + y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6) * weight.double()
    # a gate's sum or a rounded x in another order may round to the neighbouring bfloat16 value (2^-8 of one of the side
    # values, and of their result over the root of their number); the kernel without matrix cores is held to the same
    bound = 2.0 ** -8 * 6.0 * weight.double() + 1e-5
    for result in (got, before):
        off = (result.double() - want).abs()
        assert bool((off <= bound).all())
        assert float(off.square().mean().sqrt()) <= 2e-3


@pytest.mark.parametrize("q_lens", [[3, 300, 1], [1] * 260 + [256], [127, 256], [128, 256], [257, 255], [1] * 300, [400, 260], [17, 4100, 0, 2]])
@pytest.mark.parametrize("dim", [192, 2112])
def test_a_portions_bits_do_not_depend_on_the_step(q_lens, dim):
    from cwm_amd import ops

    g = torch.Generator(device=DEV).manual_seed(sum(q_lens))
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    side, vocab, n = 64, 61, sum(q_lens)
    h, tokens = normal(n, dim), torch.randint(vocab, (n,), generator=g, device=DEV, dtype=torch.int32)
    gate, proj, table = normal(side, dim).mul(dim ** -0.5).bfloat16(), normal(dim, side).bfloat16(), normal(vocab, side).bfloat16()
    args = (table, 0, gate, proj.t().contiguous(), normal(dim).abs() + 0.3, 1e-6, True)
    parts = normal(2, n, dim)

    def step(lens, first, last):
        lengths = torch.tensor(lens)
        batch = SimpleNamespace(
            q_lens=list(lens), cu_q=torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).int().to(DEV),
            seq_of_token=torch.repeat_interleave(torch.arange(len(lens)), lengths).int().to(DEV),
        )
        out = h[first:last].clone()
        ops.token_side(out, tokens[first:last], *args, pending=parts[:, first:last].contiguous(), w_proj=proj, batch=batch)
        return out

    together, first = step(q_lens, 0, n), 0
    for b, q in enumerate(q_lens):
        if q and (b < 6 or b >= len(q_lens) - 2):
            assert torch.equal(together[first : first + q], step([q], first, first + q)), b
        first += q
