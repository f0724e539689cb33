"""The delta rule's preparation, eight tokens a workgroup and one: the same bits whatever the rank is, at the edges of its quarters and of the sixteen that are loaded together."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import hand_step, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rank", [1, 3, 63, 64, 65, 129, 257, 400, 512])
def test_tokens_together_and_apart(rank, dtype):
    from llama_cu_amd.kernels import ops
    heads, dim, requests, each = 4, 24, 257, 4                   # 4,112 tokens' heads, and 1,028
    hd = heads * dim
    off = {"r": 0, "k": hd, "v": 2 * hd, "g": 3 * hd, "a": 4 * hd, "l": 5 * hd}
    args = tuple(t.cuda() for t in (rnd(rank, hd, seed=3, std=rank ** -0.5), rnd(hd, seed=4), rnd(hd, seed=5), rnd(hd, seed=6) * 0.1 + 1))
    proj = rnd(requests * each, 5 * hd + rank, seed=1).to(dtype).cuda()
    before = rnd(requests, heads, dim, dim, seed=2).cuda()

    def run(first, last):
        n = last - first
        state = before[first:last].clone()
        step = hand_step([each] * n, [each + 7] * n, list(range(n)))
        return ops.delta_rule(proj[first * each:last * each], off, *args, state, step, heads, dim, dim, 1e-5), state

    out, state = run(0, requests)
    for first in range(0, requests, 64):
        last = min(requests, first + 64)
        few, few_state = run(first, last)
        assert torch.equal(out[first * each:last * each], few) and torch.equal(state[first:last], few_state)
