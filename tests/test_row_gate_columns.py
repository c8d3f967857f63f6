"""A gated feed-forward with a row's gate: its matrix has its own number of columns for up to as many rows as the streaming product takes,
and whole groups of 16 above."""

from __future__ import annotations

import pytest
import torch

from cwm_amd import ops
from cwm_amd.parts.base import Runtime
from cwm_amd.parts.feedforward import GatedMLP


def _part(dim, hidden, device, dtype, stream_copies):
    part = GatedMLP(dim, hidden, row_gate="sg")
    gen = torch.Generator().manual_seed(hidden)
    tensors = {name: (torch.randn(spec.shape, generator=gen) * dim**-0.5).to(dtype).to(device) for name, spec in part.tensor_specs().items()}
    part.bind(tensors, Runtime(device=torch.device(device), act_dtype=dtype, stream_copies=stream_copies))
    return part, tensors


def test_both_forms_share_their_memory():
    part, tensors = _part(64, 40, "cpu", torch.float32, False)
    own, wide = part.gate_up.weight, part.gate_up_wide.weight
    assert own.shape == (81, 64) and wide.shape == (96, 64) and own.data_ptr() == wide.data_ptr()
    assert torch.equal(own, torch.cat([tensors["gate"], tensors["up"], tensors["sg"]])) and not wide[81:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [False, True])
@pytest.mark.parametrize("rows", [1, 12, 33, 64, 65, 129, 256, 257, 700])
def test_rows_of_either_form(rows, copies):
    dim, hidden = 512, 256
    part, tensors = _part(dim, hidden, "cuda:0", torch.bfloat16, copies)
    x = torch.randn(rows, dim, generator=torch.Generator().manual_seed(rows)).bfloat16().to("cuda:0")
    got = part.forward(x, None)
    got = got.sum(0) if got.dim() == 3 else got
    if rows <= 64:  # the bits of the matrix without zeros
        weight = torch.cat([tensors["gate"], tensors["up"], tensors["sg"]])
        joined = ops.linear(x, weight, None, None, True, streamed=ops.stream_layout(weight) if copies else None)
        same = part.down(ops.gated_act_rows(joined, hidden, part.activation, x.dtype, 2 * hidden), partials_ok=True)
        assert torch.equal(got, same.sum(0) if same.dim() == 3 else same)
    gate, up, row, down = (tensors[n].double() for n in ("gate", "up", "sg", "down"))
    a = x.double()
    want = torch.sigmoid(a @ row.t()) * (torch.nn.functional.silu(a @ gate.t()) * (a @ up.t())) @ down.t()
    # gate, up, hidden row and result are rounded to bfloat16, 2^-9 of each; a sum of `hidden` of them
    assert float((got.double() - want).norm() / want.norm()) <= 2.0**-6
