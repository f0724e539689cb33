"""The weight-streaming product's packed loop, which keeps loads on their way, against the one for plain weights: the same sums in the same order, so the same bits."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import rnd

pytestmark = pytest.mark.gpu


# a wave has no step at all, fewer than are on their way, as many, whole turns of them and every number left behind the last
@pytest.mark.parametrize("steps", [1, 3, 8, 9, 17, 24, 31, 33, 40, 63, 64, 65, 72, 81, 97])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16, 17, 24, 25, 32])
@pytest.mark.parametrize("tiles,waves", [(1, 8), (1, 4), (2, 8), (2, 4), (4, 4)])
def test_packed_rows_have_the_bits_of_plain_ones(steps, m, tiles, waves):
    from llama_cu_amd.kernels import ops
    n, k = 16 * tiles + 16, 128 * steps
    x, w = rnd(m, k, seed=1).bfloat16().cuda(), rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda()
    kw = dict(out_dtype=torch.float32, tiles=tiles, waves=waves)
    assert torch.equal(ops.gemm_skinny(x, ops.pack_weight(w), packed=True, **kw), ops.gemm_skinny(x, w, **kw))
