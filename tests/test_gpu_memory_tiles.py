"""The matrix memory's blocks of bfloat16 rows on the matrix cores: whole pieces of 16 bytes and rows without them give what float64
gives, and an infinity or a NaN stays where the recurrence leaves it."""

from __future__ import annotations

import pytest
import torch

from test_gpu_dogotar import MemoryCase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,d,e", [(2, 8, 8), (3, 32, 24), (2, 40, 64), (1, 128, 128), (1, 136, 8), (1, 256, 32)])
@pytest.mark.parametrize("lengths", [[33, 600, 9], [1060]])
def test_whole_pieces(heads, d, e, lengths):
    from cwm_amd import ops

    case = MemoryCase(heads, d, e, 6.0, lengths, torch.bfloat16, seed=sum(lengths) + d)
    slots = list(range(len(lengths)))
    whole, state = case.run([list(enumerate(lengths))], slots)
    case.check(whole, "whole")
    _, walked = case.run([[(s, 1) for s, n in enumerate(lengths) if i < n] for i in range(40)] + [[(s, n - 40) for s, n in enumerate(lengths) if n > 40]], slots)
    for s in slots:
        a, b = (ops.matrix_memory_state_unpack(t[s], heads, d, e) for t in (state, walked))
        # float32 sums of up to a thousand products, weights of at most one, as tests of segments have it
        torch.testing.assert_close(a[0], b[0], rtol=1e-4, atol=1e-5)
        torch.testing.assert_close(a[1], b[1], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("place", ["q", "v"])
def test_values_that_are_not_finite(bad, place):
    heads, d, e, n, at = 2, 64, 32, 640, 300
    case = MemoryCase(heads, d, e, 6.0, [n], torch.bfloat16, seed=5)
    clean, _ = case.run([[(0, n)]], [0])
    proj = case.proj[0].clone()
    column = 0 if place == "q" else 2 * heads * d
    case.proj[0][at, column] = bad
    got, _ = case.run([[(0, n)]], [0])
    case.proj[0] = proj
    first = at - at % 32  # tokens of the blocks before have the same bits, and the other head's all have
    assert torch.equal(got[0][:first], clean[0][:first])
    assert torch.equal(got[0][:, e:], clean[0][:, e:])
    row = got[0][at, :e].float()
    assert torch.isnan(row).any()
    if place == "q":  # a query reaches its own token only
        keep = [t for t in range(n) if t != at]
        torch.testing.assert_close(got[0][keep].float(), clean[0][keep].float(), rtol=2e-2, atol=2e-2)  # bfloat16 results
    else:  # a value stays in the state
        assert (~torch.isfinite(got[0][at:, :e].float())).any(1).all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [300, 100])
def test_a_key_that_is_not_finite(bad, at):
    """It reaches the state, so its head's later tokens, over the segments' borders (256 and 512) too, and nothing else."""
    from cwm_amd import ops

    heads, d, e, n, row = 2, 64, 32, 640, 5
    case = MemoryCase(heads, d, e, 6.0, [n], torch.bfloat16, seed=6)
    clean, clean_state = case.run([[(0, n)]], [0])
    case.proj[0][at, heads * d + row] = bad
    want = case.from_inputs(0)
    got, state = case.run([[(0, n)]], [0])
    first = at - at % 32  # tokens of the blocks before have the same bits, and the other head's all have
    assert torch.equal(got[0][:first], clean[0][:first])
    assert torch.equal(got[0][:, e:], clean[0][:, e:])
    torch.testing.assert_close(got[0][first:at].float(), clean[0][first:at].float(), rtol=2e-2, atol=2e-2)  # bfloat16 results
    assert torch.equal(torch.isfinite(got[0]), torch.isfinite(want))
    assert not torch.isfinite(got[0][at:, :e]).any()
    (s, norm, m), (s0, norm0, m0) = (ops.matrix_memory_state_unpack(t[0], heads, d, e) for t in (state, clean_state))
    assert not torch.isfinite(s[0, row]).any() and not torch.isfinite(norm[0, row])
    others = [r for r in range(d) if r != row]
    torch.testing.assert_close(s[0, others], s0[0, others], rtol=1e-4, atol=1e-5)  # as tests of segments have it
    torch.testing.assert_close(norm[0, others], norm0[0, others], rtol=1e-4, atol=1e-5)
    assert torch.equal(s[1], s0[1]) and torch.equal(norm[1], norm0[1]) and torch.equal(m, m0)
