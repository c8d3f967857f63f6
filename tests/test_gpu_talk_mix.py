"""Normalising and mixing a table of scores: tables narrower than a load, odd widths, rows that read a part of them and rows beyond
what a wavefront keeps, few and many heads, and widths whose last block has only threads that start in the block before."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_q,n_kv", [(4, 2), (7, 7), (16, 4), (20, 5)])
@pytest.mark.parametrize(
    "rows,columns,base,window",
    [(1, 1, 0, None), (2, 3, 5, 1), (4, 4, 0, None), (37, 130, 9, 60), (300, 1001, 11, 500), (260, 1024, 0, None), (9, 4099, 3, None), (5, 2052, 0, 2049),
     (513, 513, 0, None), (514, 514, 0, None), (515, 515, 7, None), (769, 769, 0, None), (400, 770, 0, 300)],
)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_against_float64(n_q, n_kv, rows, columns, base, window, dtype):
    from cwm_amd.ops import _check, _code, _ptr, _stream
    from cwm_amd.ops import build

    g = torch.Generator(device=DEV).manual_seed(columns + n_q)
    per, pos0 = n_q // n_kv, base + columns - rows
    scores = 30 * torch.randn((n_kv, rows, per, columns), generator=g, device=DEV)
    sink, talk = torch.randn(n_q, generator=g, device=DEV), torch.randn((n_q, n_q), generator=g, device=DEV)
    key, at = base + torch.arange(columns, device=DEV), pos0 + torch.arange(rows, device=DEV)
    reads = (key[None] <= at[:, None]) & (key[None] >= (0 if window is None else at[:, None] - (window - 1)))
    by_row = scores.permute(1, 0, 2, 3).reshape(rows, n_q, columns)
    lib = build.load("attention_talk")
    for use_sink, use_talk in ((True, True), (False, False)):
        weights, stats = torch.full((n_kv, rows, per, columns), 7.0, device=DEV, dtype=dtype), torch.empty(rows, n_q, 2, device=DEV)
        # columns a row does not read may hold anything
        dirty = scores.masked_fill(~reads[None, :, None], float("nan"))
        _check(lib, lib.cwm_talking_mix(
            _ptr(dirty), _ptr(weights), ctypes.c_int(_code(dtype)), _ptr(stats), ctypes.c_int(rows), ctypes.c_int(columns), ctypes.c_int(n_q), ctypes.c_int(n_kv),
            ctypes.c_int(pos0), ctypes.c_int(base), ctypes.c_int(-1 if window is None else window - 1), ctypes.c_float(0.1), _ptr(sink if use_sink else None),
            _ptr(talk if use_talk else None), _stream()))
        s = (by_row.double() * 0.1).masked_fill(~reads[:, None], float("-inf"))
        top = s.amax(-1, keepdim=True)
        top = torch.maximum(top, sink.double()[None, :, None]) if use_sink else top
        e = torch.exp(s - top)
        p = e / (e.sum(-1, keepdim=True) + (torch.exp(sink.double()[None, :, None] - top) if use_sink else 0.0))
        want = torch.matmul(talk.double(), p) if use_talk else p
        size = torch.matmul(talk.double().abs(), p) if use_talk else p
        got = weights.permute(1, 0, 2, 3).reshape(rows, n_q, columns).double()
        # an exponent's argument of up to about 20 has an error of 20 x 2^-24 and the fast exponential a few units more, the sums of
        # up to 4,099 weights the logarithm of that; bfloat16 rounds once more
        assert bool(((got - want).abs() <= (2.0 ** -17) * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0) + 1e-37).all())
        assert bool((got.masked_select(~reads[:, None].expand_as(got)) == 0).all())
