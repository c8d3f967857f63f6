"""Passes over rows that take several values a thread: widths with and without whole pieces give the same values, those of float32 torch."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("width", [8, 24, 2040, 2048, 2056, 6152, 7, 2044])
@pytest.mark.parametrize("rows", [1, 5, 300])
def test_sigmoid_gate_and_embedding(width, rows):
    from cwm_amd import ops

    g = torch.Generator().manual_seed(width + rows)
    a, z = (torch.randn((rows, width), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    got = ops.sigmoid_mul(a, z)
    want = a.float() * torch.sigmoid(z.float())
    torch.testing.assert_close(got.float(), want, rtol=2 ** -8, atol=1e-6)  # one rounding to bfloat16
    table = torch.randn((50, width), generator=g).to(torch.bfloat16).to(DEV)
    tokens = torch.randint(50, (rows,), generator=g).to(torch.int32)
    out = ops.embedding(tokens.to(DEV), table, 1.5)
    assert torch.equal(out.cpu(), table.cpu().float()[tokens.long()] * 1.5)
