"""Streamed products of 9 to 32 rows whose consumer adds float32 sums leave float32 sums, also where K is not split: what follows is
computed on them and rounded once."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def drawn(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    normal = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x, w = normal(m, k).bfloat16(), (normal(n, k) * k ** -0.5).bfloat16()
    return x, w, x.double() @ w.double().T


# N of 8,192 and more or K below 1,024: K is not split.  The others: it is.
SIZES = [(10240, 2048), (8208, 1024), (9216, 3072), (2048, 512), (1024, 2048)]


@pytest.mark.parametrize("m", [9, 12, 16, 17, 24, 32])
@pytest.mark.parametrize("n,k", SIZES)
def test_activations_round_once(m, n, k):
    from cwm_amd import ops

    x, w, want = drawn(m, n, k)
    joined = ops.linear(x, w, None, partials_ok=True, streamed=ops.stream_layout(w))
    assert joined.dtype == torch.float32 and joined.dim() == 3

    # one rounding to bfloat16, at most 2^-8 of the value; float32 sums off by at most 2^-18 of values of order one
    def once(got, exact, slope):
        return bool(((got.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 2.0 ** -18 * slope).all())

    assert once(ops.act_rows(joined, "relu2", torch.bfloat16), want.clamp_min(0) ** 2, 2 * want.abs() + 1)
    gate, up = want[:, : n // 2], want[:, n // 2 :]
    got = ops.gated_act_rows(joined, n // 2, ops.GatedActivation("silu"), torch.bfloat16, None)
    assert once(got, torch.nn.functional.silu(gate) * up, 1.1 * up.abs() + gate.abs() + 1)


@pytest.mark.parametrize("m", [9, 16, 17, 32])
@pytest.mark.parametrize("n,k", SIZES)
def test_a_residual_takes_the_sums_as_they_are(m, n, k):
    from cwm_amd import ops

    x, w, want = drawn(m, n, k)
    h = torch.zeros((m, n), device=DEV)
    ops.add_rmsnorm(h, ops.linear(x, w, None, partials_ok=True, streamed=ops.stream_layout(w)), torch.ones(n, device=DEV), 1e-5, torch.bfloat16)
    assert bool(((h.double() - want).abs() <= 2.0 ** -18 * (want.abs() + 1)).all())
