"""The float32 product whose operands go to the matrix cores in three bfloat16 parts: sizes at the edges of its tiles and steps,
values that need all 24 bits, of very different sizes, and ones that round to infinity in bfloat16."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _normal(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


@pytest.mark.parametrize("m", [1, 17, 32, 33, 64, 65, 130, 300])
@pytest.mark.parametrize("n,k", [(1, 32), (63, 64), (129, 96), (520, 1056)])
@pytest.mark.parametrize("c_dtype", [torch.float32, torch.bfloat16])
def test_against_float64(m, n, k, c_dtype):
    from cwm_amd import ops

    a, w, b = _normal((m, k), m), _normal((n, k), n), _normal((n,), k)
    got = ops.gemm_f32(a, w, b, out_dtype=c_dtype).double()
    want = a.double() @ w.double().T + b.double()
    # each of the k products is off by less than 2^-23 of itself, each of the 6 k / 32 sums by 2^-24 of the running sum
    bound = (a.double().abs() @ w.double().abs().T) * 2.0 ** -23 + (0.2 * k + 2) * 2.0 ** -24 * (k ** 0.5 + 4)
    if c_dtype == torch.bfloat16:
        bound = bound + want.abs() * 2.0 ** -8
    assert bool(((got - want).abs() <= bound).all())
    # a row's bits do not depend on the others
    for rows in (slice(0, 1), slice(m // 2, m)):
        assert torch.equal(ops.gemm_f32(a[rows].contiguous(), w, b, out_dtype=c_dtype).double(), got[rows])


def test_rows_that_lie_apart_and_values_of_all_sizes():
    from cwm_amd import ops

    m, n, k = 70, 200, 128
    scale = 10.0 ** torch.linspace(-18, 18, k, device=DEV)  # the products are of order one, their parts from 1e-22 to 1e22
    wide = _normal((m, k + 36), 1)
    a = wide[:, 4 : 4 + k]
    a *= scale
    w = _normal((n, k), 2) / scale
    got, want = ops.gemm_f32(a, w).double(), a.double() @ w.double().T
    assert bool(((got - want).abs() <= (a.double().abs() @ w.double().abs().T) * 2.0 ** -21).all())
    # numbers with all 24 bits set: a part less would show
    a, w = torch.full((40, 32), 1.0 + 2.0 ** -23, device=DEV), torch.full((40, 32), 1.0 - 2.0 ** -24, device=DEV)
    exact = 32.0 * (1.0 + 2.0 ** -23) * (1.0 - 2.0 ** -24)
    assert float((ops.gemm_f32(a, w).double() - exact).abs().max()) <= 32 * 2.0 ** -23


def test_values_beyond_the_parts():
    """Infinities, NaN and the largest float32 values give what float32 gives."""
    from cwm_amd import ops

    m, n, k = 140, 150, 64
    a, w = _normal((m, k), 3), _normal((n, k), 4)
    a[5, 7], a[20, 1], a[139, 60] = math.inf, -math.inf, math.nan
    a[60] = 0.0
    a[60, 3] = 3.4e38
    w[8, 3], w[9, 3] = 1.0, 0.5
    w[100, 7] = 0.0
    got, want = ops.gemm_f32(a, w), (a.double() @ w.double().T).float()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    fine = torch.isfinite(want)
    torch.testing.assert_close(got[fine], want[fine], rtol=1e-5, atol=2e-5)
    assert bool((got[~fine & ~torch.isnan(want)] == want[~fine & ~torch.isnan(want)]).all())


@pytest.mark.parametrize("m", [17, 40, 300])
@pytest.mark.parametrize("a_size,w_size", [(1e-30, 1e3), (1e-36, 1e4), (1e-38, 1e9), (3e-43, 1e9), (1e-19, 1e-18), (1e-25, 1e-9), (1e9, 1e-36), (4e9, 4e9)])
def test_sizes_at_the_ends_of_float32(m, a_size, w_size):
    """Operands and products down to the smallest normal numbers and below, where a part more than the last bit would be lost."""
    from cwm_amd import ops

    n, k = 130, 96
    a, w = _normal((m, k), 5) * a_size, _normal((n, k), 6).clamp(-1, 1) * w_size
    a[:, ::7] = 0.0
    got, want = ops.gemm_f32(a, w).double(), a.double() @ w.double().T
    # as in the first test, and half of the smallest float32 number for a result below the normal ones
    bound = (a.double().abs() @ w.double().abs().T) * (2.0 ** -23 + 0.2 * k * 2.0 ** -24) + 2.0 ** -150
    assert bool(((got - want).abs() <= bound).all())


def test_a_value_beyond_the_parts_changes_no_other_row():
    from cwm_amd import ops

    m, n, k = 140, 150, 64
    a, w, b = _normal((m, k), 3), _normal((n, k), 4), _normal((n,), 5)
    fine = ops.gemm_f32(a, w, b)
    odd, odd_w = a.clone(), w.clone()
    odd[5, 7], odd[20, 1], odd[139, 60], odd[60, 3], odd[61, 3] = math.inf, -math.inf, math.nan, 3.4e38, 2.0 ** 32
    odd_w[8, 3], odd_w[149, 0] = 1e30, math.inf
    got = ops.gemm_f32(odd, odd_w, b)
    rows = [i for i in range(m) if i not in (5, 20, 139, 60, 61)]
    columns = [i for i in range(n) if i not in (8, 149)]
    assert torch.equal(got[rows][:, columns], fine[rows][:, columns])
    # and the odd rows and columns are the same in any company
    assert torch.equal(ops.gemm_f32(odd[60:62].contiguous(), odd_w, b), got[60:62])
    assert torch.equal(ops.gemm_f32(odd, odd_w[8:9].contiguous(), b[8:9].contiguous())[:, 0][rows], got[:, 8][rows])


@pytest.mark.parametrize("m,n", [(20, 2048), (227, 3072), (700, 9000)])
@pytest.mark.parametrize("k", [512, 2048, 2080, 8192, 14336])
def test_results_are_not_all_low_or_high(m, n, k):
    """Roundings of an instruction that rounds down add up to the same amount in every result, and over a model's layers."""
    from cwm_amd import ops

    a, w = _normal((m, k), k), _normal((n, k), k + 1)
    off = ops.gemm_f32(a, w).double() - a.double() @ w.double().T
    # unbiased errors have a mean of their size over the root of their number, here at most 1 / 200 (five deviations: 0.025)
    assert abs(float(off.mean())) <= 0.025 * float(off.square().mean().sqrt())
