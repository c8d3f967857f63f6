"""A layer's token input with four, eight and sixteen tokens a block: the same bits, at widths of every build and its edges."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from test_gpu_token_side_tiles import test_against_float64 as against_float64

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_tokens,dim,side", [(256, 256, 32), (300, 320, 128), (2049, 512, 96), (2050, 576, 32), (263, 1024, 64), (2063, 1088, 128), (2049, 3136, 64), (4097, 3520, 32), (1024, 3520, 64)])
def test_against_float64_at_every_build(n_tokens, dim, side):
    against_float64(n_tokens, dim, side)


@pytest.mark.parametrize("dim,side", [(64, 32), (256, 128), (320, 64), (512, 96), (1024, 32), (2048, 64), (3136, 128), (3520, 64), (4096, 32)])
@pytest.mark.parametrize("pending", [True, False])
def test_blocks_of_any_size_give_the_same_bits(dim, side, pending):
    """A portion alone, behind a portion that makes the step's blocks larger, and with short ones between."""
    from cwm_amd import ops
    from cwm_amd.ops import build

    lib, first = build.load("token_side"), 300
    steps = [[first], [first, 1500], [first, 2000], [7, first, 3, 1800]]
    toks = {lib.cwm_token_side_tile_tokens(sum(s), dim, side) for s in steps}
    assert toks == ({4, 8, 16} if dim > 3456 else {8, 16})
    g = torch.Generator(device=DEV).manual_seed(dim + side)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    vocab, n = 61, 2400
    h, tokens = normal(n, dim), torch.randint(vocab, (n,), generator=g, device=DEV, dtype=torch.int32)
    gate, proj, table = normal(side, dim).mul(dim ** -0.5).bfloat16(), normal(dim, side).bfloat16(), normal(vocab, side).bfloat16()
    args = (table, 0, gate, proj.t().contiguous(), normal(dim).abs() + 0.3, 1e-6, True)
    parts, other = normal(2, n, dim), normal(n, dim).bfloat16()

    def run(lens):
        lengths = torch.tensor(lens)
        batch = SimpleNamespace(
            q_lens=list(lens), cu_q=torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).int().to(DEV),
            seq_of_token=torch.repeat_interleave(torch.arange(len(lens)), lengths).int().to(DEV),
        )
        at = sum(lens[: lens.index(first)])  # the portion's rows are the first of the data wherever it lies in the step
        order = torch.cat([torch.arange(first, first + at), torch.arange(first), torch.arange(first + at, sum(lens))]).to(DEV)
        out = h[order].contiguous()
        sums = ops.ScaledSum([(parts[:, order].contiguous(), 1.0), (other[order].contiguous(), 0.5)]) if pending else None
        ops.token_side(out, tokens[order].contiguous(), *args, pending=sums, w_proj=proj, batch=batch)
        return out[at : at + first]

    want = run(steps[0])
    for lens in steps[1:]:
        assert torch.equal(run(lens), want), lens
