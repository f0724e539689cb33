"""The router over rows of whole chunks, one or four tokens a workgroup, against the general kernel (the same rows with eight zeros behind them), bit for bit."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import F64, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,n,experts,extra,top,how", [
    (2048, 1, 16, 1, 2, {}), (2048, 256, 4, 0, 4, {"softmax_chosen": True}), (2048, 257, 17, 8, 3, {}), (2048, 976, 16, 0, 2, {}),
    (2048, 977, 16, 1, 2, {"softmax_all": True, "groups": 4, "keep": 2, "scale": 2.5}), (1024, 1955, 18, 0, 2, {"softmax_all": True}), (1024, 258, 3, 0, 1, {}), (1024, 9, 4, 0, 2, {}),
    (512, 3907, 1, 0, 1, {}), (512, 3910, 1024, 8, 8, {"softmax_all": True, "renorm": False}), (2048, 260, 300, 0, 300, {"softmax_chosen": True}),
])
def test_route(dtype, d, n, experts, extra, top, how):
    from llama_cu_amd.kernels import ops
    h, w = rnd(n, d, seed=1).to(dtype).cuda(), rnd(experts + extra, d, seed=2, std=d ** -0.5).cuda()
    bias = rnd(experts, seed=3, std=0.1).cuda()
    more = lambda x: torch.cat([x, torch.zeros(x.shape[0], 8, dtype=x.dtype, device="cuda")], dim=1)
    got = ops.moe_route(h, w, top, bias, extra=extra, **how)
    want = ops.moe_route(more(h), more(w), top, bias, extra=extra, **how)
    assert len(got) == len(want) == (3 if extra else 2)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # the best expert by 64-bit logits, where no other comes near it
    z = h.to(F64) @ w[:experts].to(F64).T
    if how.get("softmax_all"):
        z = torch.softmax(z, dim=-1)
    z = z + bias
    if "groups" not in how and experts > 1:
        best = z.topk(2, dim=-1)
        sure = best.values[:, 0] - best.values[:, 1] > 1e-4
        assert torch.equal(got[0][sure, 0].long(), best.indices[sure, 0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,n,experts,extra,how", [
    (512, 1954, 64, 0, {}), (1024, 977, 17, 1, {"softmax_chosen": True}), (1024, 2930, 18, 0, {}), (1536, 300, 5, 8, {}), (1536, 652, 64, 0, {"softmax_all": True}),
    (1536, 1954, 16, 1, {}), (2048, 489, 1024, 0, {"softmax_all": True, "renorm": False}), (2560, 257, 16, 1, {}), (3072, 515, 64, 0, {"softmax_chosen": True}),
    (3584, 513, 300, 3, {}), (4096, 512, 16, 1, {}), (4096, 513, 16, 1, {}), (2048, 1000, 5, 0, {}),
])
def test_route_in_steps_of_few_tokens(dtype, d, n, experts, extra, how):
    """One, two and four tokens a workgroup at every whole number of chunks: a token's bits are those that it has in a step of few tokens, which has a kernel of its own."""
    from llama_cu_amd.kernels import ops
    h, w = rnd(n, d, seed=4).to(dtype).cuda(), rnd(experts + extra, d, seed=5, std=d ** -0.5).cuda()
    bias = rnd(experts, seed=6, std=0.1).cuda()
    for b in (bias, None):
        got = ops.moe_route(h, w, 3, b, extra=extra, **how)
        parts = [ops.moe_route(part, w, 3, b, extra=extra, **how) for part in h.split(250)]
        for k, a in enumerate(got):
            assert torch.equal(a, torch.cat([p[k] for p in parts]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,n", [(1536, 3), (2560, 1), (2560, 130), (3584, 900), (2048, 900), (2048, 1100)])
def test_route_to_few_experts(dtype, d, n):
    """Four experts, a wave each: against the general kernel, as above."""
    from llama_cu_amd.kernels import ops
    h, w, bias = rnd(n, d, seed=7).to(dtype).cuda(), rnd(4, d, seed=8, std=d ** -0.5).cuda(), rnd(4, seed=9).cuda()
    more = lambda x: torch.nn.functional.pad(x, (0, 8))
    for a, b in zip(ops.moe_route(h, w, 2, bias), ops.moe_route(more(h), more(w), 2, bias)):
        assert torch.equal(a, b)
