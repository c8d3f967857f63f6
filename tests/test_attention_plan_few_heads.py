"""The work lists of attention with one large key/value head, whose keys are cut finer (host arithmetic only)."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from cwm_amd import ops
from cwm_amd.ops.attention_plan import NULL_ROW, build_plan, capacity_until, pad_plan


@pytest.mark.parametrize("window", [None, 100, 8192])
@pytest.mark.parametrize("kv", [[1], [256], [257, 3], [8192, 8193, 40], [65536, 65537], [70000, 511, 513]])
def test_keys_are_covered_once_at_every_length_of_the_rule(kv, window):
    q = [1] * len(kv)
    plan = build_plan(q, kv, 16, window, few_heads=True)
    for b, n in enumerate(kv):
        items = sorted(w[2:5] for w in plan.work.tolist() if w[0] == b)
        lo = 0 if window is None else max(0, n - window)
        cut = 256 if n - lo <= 8192 else 512 if n - lo <= 65536 else 1024
        assert items[0][0] == lo and items[-1][1] == n and all(a[1] == c[0] for a, c in zip(items, items[1:]))
        assert all(end - first <= cut and (first % cut == 0 or first == lo) for first, end, _ in items)
        assert (len(items) == 1) == (items[0][2] == -1)


@pytest.mark.parametrize("window", [None, 300])
def test_captured_lists_hold_every_later_step(window):
    q, kv, most = [1, 1, 1], [8000, 200, 255], 9000
    plan, capacity = capacity_until(q, kv, 16, window, 0, most, few_heads=True)
    for t in [0, 1, 2, 56, 57, 191, 192, 193, 194, 500, most - 8000]:
        flat = pad_plan(build_plan(q, [n + t for n in kv], 16, window, few_heads=True), capacity)
        assert flat is not None and flat.size == capacity.ints
        work = flat[: capacity.work * 6].reshape(-1, 6)
        assert np.all((work[:, 1] == NULL_ROW) | (work[:, 3] > work[:, 2]))


@pytest.mark.parametrize("few_heads,window,chunk", [(True, 8192, None), (True, 16384, None), (True, 16500, None), (False, 32768, None), (True, None, 8320), (True, 7936, None), (True, 8191, None)])
@pytest.mark.parametrize("past", [0, 1, 255, 256, 512, 700])
def test_captured_lists_hold_a_window_at_every_place(few_heads, window, chunk, past):
    """A window's chunks are counted differently from step to step, also across the border between the two lists of merges."""
    span = window if chunk is None else chunk
    q, kv, most = [1, 1], [span + past, span + past + 256], 2 * span + 4096
    _, capacity = capacity_until(q, kv, 16, window, 0, most, chunk, few_heads)
    for t in [*range(0, 1100, 3), most - max(kv)]:
        assert pad_plan(build_plan(q, [n + t for n in kv], 16, window, 0, chunk, few_heads), capacity) is not None, t


def test_short_windows_leave_no_room_for_many_partials():
    _, capacity = capacity_until([1], [9000], 16, 4096, 0, 16384, few_heads=True)
    assert capacity.merge_many == 0 and capacity.merge_mid == 1


@pytest.mark.parametrize("n_kv,head_dim,finer", [(1, 256, True), (1, 192, True), (1, 128, False), (2, 128, False), (2, 256, False), (8, 128, False)])
def test_keys_are_cut_finer_for_one_large_head_alone(n_kv, head_dim, finer):
    batch = SimpleNamespace(q_lens=[1, 1], kv_lens=[2000, 700], scratch={}, static=None)
    plan = ops._attention_plan(batch, 16, n_kv, head_dim, None, torch.device("cpu"))
    assert plan.n_work == (11 if finer else 2)
    # lists of other sizes of head are others, in a captured step as well
    other = ops._attention_plan(batch, 16, n_kv, 64, None, torch.device("cpu"))
    assert other.n_work == 2 and (other is plan) == (not finer)
