"""A decode step of linear attention with five inputs in two kernels, at the row counts beyond one tile of 16: where the streaming
product's blocks change (17, 33) and end (32, 64), with K split and not."""

from __future__ import annotations

import pytest

from test_gpu_sunusun import test_a_decode_step_in_two_kernels as decode_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,dim,rank,width,batch", [(2, 64, 16, 256, 17), (3, 32, 8, 4096, 32), (2, 48, 40, 2048, 33), (4, 64, 64, 512, 64), (1, 16, 5, 2176, 25)])
def test_more_rows_than_a_tile(heads, dim, rank, width, batch):
    decode_step(heads, dim, rank, width, batch)
