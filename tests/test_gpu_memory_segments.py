"""The matrix memory's long portions in segments walked side by side: lengths around whole segments and blocks, several portions
of which some have one segment, states that are carried in and out, and gates that decide what survives a segment's border."""

from __future__ import annotations

import pytest
import torch

from test_gpu_dogotar import MemoryCase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,d,e", [(2, 20, 12), (1, 64, 32), (1, 130, 40)])
@pytest.mark.parametrize("lengths", [[512, 1, 256], [3, 513, 255, 257], [767, 600], [40, 1056]])
def test_segments_and_the_walk(heads, d, e, lengths):
    from cwm_amd import ops

    case = MemoryCase(heads, d, e, 6.0, lengths, torch.float32, seed=sum(lengths) + d)
    slots = list(range(len(lengths)))[::-1]
    whole, state = case.run([list(enumerate(lengths))], slots)
    case.check(whole, "whole")
    # a first step of one token each, so that the segments start from a state, and a last one that continues from theirs
    middle = [(s, n - 2) for s, n in enumerate(lengths) if n > 2]
    parts, carried = case.run([[(s, 1) for s in range(len(lengths))], middle, [(s, 1) for s, n in enumerate(lengths) if n > 1]], slots)
    case.check(parts, "from a state")
    for s in slots:
        a, b = (ops.matrix_memory_state_unpack(t[s], heads, d, e) for t in (state, carried))
        assert torch.equal(a[2], b[2])  # the maximum is the walk's to the bit
        # float32 sums of up to a thousand products, weights of at most one: as far apart as blocks and the walk are
        torch.testing.assert_close(a[0], b[0], rtol=1e-4, atol=1e-5)
        torch.testing.assert_close(a[1], b[1], rtol=1e-4, atol=1e-5)
