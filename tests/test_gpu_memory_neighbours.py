"""The matrix memory cuts a portion by its own length: a portion's results and state have the same bits alone and beside others,
and scratch grows with the tokens, not with the sequences."""

from __future__ import annotations

import ctypes

import pytest
import torch

from test_gpu_dogotar import MemoryCase

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,d,e", [(2, 20, 12), (1, 64, 32), (1, 128, 64), (1, 200, 40)])
@pytest.mark.parametrize("lengths", [[300, 600], [513, 257, 511, 1], [9, 512, 33, 768, 256], [1, 1, 1100, 1, 255, 1]])
def test_a_portion_alone_and_beside_others(heads, d, e, lengths, dtype):
    from cwm_amd import ops

    case = MemoryCase(heads, d, e, 6.0, lengths, dtype, seed=sum(lengths) + d)
    for gates in case.gates:
        gates[:, heads:] += 12.0  # capped forget gates close to one: what lies hundreds of tokens back still counts
    slots = [(3 * s + 1) % len(lengths) if len(lengths) % 3 else s for s in range(len(lengths))]
    # a first step of one token each, so that every portion starts from a state
    first = [(s, 1) for s, n in enumerate(lengths) if n > 8]
    rest = [(s, n - 1 if n > 8 else n) for s, n in enumerate(lengths)]
    together, state = case.run([first, rest], slots)
    alone, apart = case.run([first] + [[portion] for portion in rest], slots)
    for s, n in enumerate(lengths):
        if n > 9:  # shorter portions alone are walked token by token, which differs by rounding
            assert torch.equal(together[s], alone[s]), n
            for a, b in zip(*(ops.matrix_memory_state_unpack(t[slots[s]], heads, d, e) for t in (state, apart))):
                assert torch.equal(a, b), n


def test_places_of_segments_hold_any_cut():
    """The library's scratch is by tokens alone; every long portion's segments lie before the place of what follows it."""
    from cwm_amd.ops import build

    lib = build.load("matrix_memory")
    lib.cwm_matrix_memory_saved_floats.restype = ctypes.c_long
    a_place = 32 * 32  # one head of 1 to 31 columns and up to 32 rows
    place = lambda t: lib.cwm_matrix_memory_saved_floats(ctypes.c_int(t), ctypes.c_int(1), ctypes.c_int(20), ctypes.c_int(12)) // a_place  # noqa: E731
    starts = [0, 1, 170, 171, 255, 256, 341, 342, 511, 512, 1000, 123457, 2 ** 31 - 1 - 70000]
    for start in starts:
        for n in [*range(512, 1400), 4095, 4096, 4097, 65535, 65537]:
            assert place(start) + -(-n // 256) <= place(start + n), (start, n)
