"""Recurrence with a bonus in steps of single tokens: the kernel's two forms, which differ in when they ask for what they read."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import TYPES, hand_step, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,dim,rank", [(12, 64, 1), (12, 48, 5), (12, 20, 64), (12, 64, 100), (4, 100, 17)])
def test_many_requests_have_the_bits_of_few(dtype, heads, dim, rank):
    """A request's outputs and state in a step of 128 requests, which fill a round of workgroups where nothing is asked for in front, and in a step of eight."""
    from llama_cu_amd.kernels import build, ops
    tdt, n, hd = TYPES[dtype], 128, heads * dim
    units = torch.cuda.get_device_properties(0).multi_processor_count
    front = build.load("wkv").lcu_wkv_front
    assert front(8, heads, dim, units) and (units != 256 or bool(front(n, heads, dim, units)) == (heads != 12))
    rows, low = rnd(n, 4 * hd, seed=1).to(tdt).cuda(), rnd(n, rank, seed=2).cuda()
    w2, w0, u, norm = rnd(rank, hd, seed=3, std=0.3).cuda(), rnd(hd, seed=4).cuda(), rnd(hd, seed=5).cuda(), rnd(hd, seed=6).cuda()
    off = {name: i * hd for i, name in enumerate("rkvg")}
    start, ctx = rnd(n, hd * dim, seed=7).cuda(), [1 + i % 5 for i in range(n)]
    one, two = start.clone(), start.clone()
    run = lambda k, state: ops.wkv(rows[:k], off, low[:k], w2, w0, u, norm, state, hand_step([1] * k, ctx[:k], list(range(k))), heads, dim, 1e-5, tdt)
    many, few = run(n, one), run(8, two)
    assert torch.equal(many[:8], few) and torch.equal(one[:8], two[:8]) and torch.equal(two[8:], start[8:]) and torch.isfinite(many.float()).all()
