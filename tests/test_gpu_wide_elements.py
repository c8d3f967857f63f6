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


@pytest.mark.parametrize("width", [8, 2056, 7, 2044])
def test_ids_outside_the_vocabulary(width):
    from cwm_amd import ops

    table = torch.randn((5, width), generator=torch.Generator().manual_seed(width)).to(torch.bfloat16).to(DEV)
    out = ops.embedding(torch.tensor([4, -1, 0, 5, 2 ** 31 - 1, -(2 ** 31)], dtype=torch.int32, device=DEV), table, 0.5)
    assert torch.isnan(out[[1, 3, 4, 5]]).all()
    assert torch.equal(out[[0, 2]], table[[4, 0]].float() * 0.5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [4, 7, 201, 1028, 2048, 4099])
@pytest.mark.parametrize("write_state", [True, False])
def test_token_shift(dtype, dim, write_state):
    """Four values a thread (widths that are multiples of four) and one."""
    from cwm_amd import ops
    from test_gpu_sequence_kernels import _both

    g = torch.Generator().manual_seed(dim)
    gb, _ = _both([1, 5, 2, 1, 3], [0, 0, 9, 4, 7], [3, 0, 2, 1, -1])
    gb.state_slots[4] = 6  # a slot that the state does not have: nothing is read or written
    h, mu, state = torch.randn((12, dim), generator=g), torch.rand(dim, generator=g), torch.randn((6, dim), generator=g)
    before = state.clone()
    sd = state.to(DEV)
    got = ops.token_shift(h.to(DEV), mu.to(DEV), sd, gb, dtype, write_state).float().cpu()
    prev = torch.cat([torch.zeros(1, dim), h[:-1]])
    prev[[0, 1, 6, 8, 9]] = torch.stack([torch.zeros(dim), torch.zeros(dim), state[2], state[1], torch.zeros(dim)])
    want = h.double() + (prev.double() - h.double()) * mu.double()
    # one rounding to bfloat16; in float32 one each of the difference, the product and the sum, which may be less than either
    size = h.double().abs() + 2.0 * (prev - h).double().abs()
    assert bool(((got.double() - want).abs() <= (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0) + 2.0 ** -23 * size).all())
    after = before.clone()
    if write_state:
        after[[3, 0, 2, 1]] = h[[0, 5, 7, 8]]
    assert torch.equal(sd.cpu(), after)
