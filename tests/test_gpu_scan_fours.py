"""The selective scan of 16 states, four tokens at a time, against the general kernel, bit for bit, and against the recurrence in 64 bits."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, hand_step, rnd

pytestmark = pytest.mark.gpu


def recurrence(x, dt_raw, bias, bc, a, d, z, state):
    x, dt_raw, bias, bc, a, d, z, S = (v.to(F64).cpu() for v in (x, dt_raw, bias, bc, a, d, z, state))
    dt, rows = torch.nn.functional.softplus(dt_raw + bias), []
    for t in range(x.shape[0]):
        S = torch.exp(dt[t][:, None] * a) * S + (dt[t] * x[t])[:, None] * bc[t, :16]
        rows.append((S @ bc[t, 16:] + d * x[t]) * torch.nn.functional.silu(z[t]))
    return torch.stack(rows), S


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels,lens,fresh", [
    (64, [5], [True]), (72, [1, 2, 3, 4], [True, False, False, True]), (1, [9, 1], [False, True]),                # within a block's channels, single tokens beside others
    (130, [515, 1, 6, 514], [True, False, True, False]), (47, [512], [False]), (2048, [4, 1000], [False, True]),  # walked in runs, of uneven lengths
])
def test_tokens_in_fours(dtype, channels, lens, fresh):
    from llama_cu_amd.kernels import ops
    n = sum(lens)
    x, dt, z = (rnd(n, channels + 3, seed=s).to(t).cuda()[:, 1:channels + 1] for s, t in ((1, dtype), (2, torch.float32), (3, torch.float32)))
    wide = rnd(n, 44, seed=4).cuda()
    bias, d, a = rnd(channels, seed=5).cuda(), rnd(channels, seed=6).cuda(), -rnd(channels, 16, seed=7).abs().cuda()
    step = hand_step(lens, [k if f else k + 11 for k, f in zip(lens, fresh)], list(range(len(lens))))
    before, got = rnd(len(lens), channels, 16, seed=8, std=3.0).cuda(), []
    for offset in (8, 5):                                            # B and C at sixteen bytes, and beside them: the general kernel
        room = wide.clone()
        room[:, offset:offset + 32] = wide[:, 8:40]
        state = before.clone()
        got.append((ops.selective_scan(x, dt, bias, room[:, offset:offset + 32], a, d, z, state, step), state))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    at = 0
    for r, k in enumerate(lens):
        rows = slice(at, at + k)
        start = torch.zeros_like(before[r]) if fresh[r] else before[r]
        want, state = recurrence(x[rows], dt[rows], bias, wide[rows, 8:40], a, d, z[rows], start)
        assert_close(got[0][0][rows], want, 1e-5 if dtype == torch.float32 else 2.0 ** -8, f"request {r}")
        assert_close(got[0][1][r], state, 1e-5, f"state {r}")
        at += k
