"""Short convolutions over many tokens, eight to a thread, against the same tokens in steps too small for that, bit for bit, and against 64 bits."""
from __future__ import annotations

import pytest
import torch

import plain_divasun as PD
import plain_mufotar as PM
from divasun_common import assert_close
from test_gpu_divasun import F64, hand_step, rnd

pytestmark = pytest.mark.gpu
LENS = [200, 3, 70, 1, 2, 65, 8]                         # runs of eight that begin inside a request, at its start, and over several requests


def in_portions(lens, forward, most=20):
    """``forward(rows of each request [(request, from, to)], step)`` over portions of at most ``most`` tokens; the outputs, request by request."""
    done, got = [0] * len(lens), [[] for _ in lens]
    while any(a < n for a, n in zip(done, lens)):
        live = [r for r in range(len(lens)) if done[r] < lens[r]][:2]
        take = [min(most, lens[r] - done[r]) for r in live]
        parts = [(r, done[r], done[r] + k) for r, k in zip(live, take)]
        out = forward(parts, hand_step(take, [b for _, _, b in parts], live))
        for (r, _, _), o in zip(parts, out.split(take, dim=-2)):
            got[r].append(o)
        for r, k in zip(live, take):
            done[r] += k
    return torch.cat([torch.cat(g, dim=-2) for g in got], dim=-2)


@pytest.mark.parametrize("types", [(torch.float32, torch.float32, torch.float32), (torch.float32, torch.float32, torch.bfloat16), (torch.bfloat16,) * 3])
@pytest.mark.parametrize("d,taps", [(40, 2), (1028, 3), (2048, 4), (39, 4), (40, 5), (64, 1)])
def test_short_convolution(types, d, taps):
    from llama_cu_amd.kernels import ops
    ti, tw, to = types
    sets, n = 2, sum(LENS)
    h, w = rnd(sets, n, d, seed=1).to(ti), rnd(sets, d, taps, seed=2, std=0.5).to(tw)
    starts = [sum(LENS[:r]) for r in range(len(LENS))]

    def forward(parts, step, state):
        rows = torch.cat([h[:, starts[r] + a:starts[r] + b] for r, a, b in parts], dim=1).contiguous().cuda()
        return ops.short_conv(rows, w.cuda(), state, torch.empty(rows.shape, dtype=to, device="cuda"), step)

    states = [torch.full((len(LENS), sets, taps - 1, d), 9.0, device="cuda") for _ in range(2)]
    whole = forward([(r, 0, k) for r, k in enumerate(LENS)], hand_step(LENS, LENS, list(range(len(LENS)))), states[0])
    cut = in_portions(LENS, lambda parts, step: forward(parts, step, states[1]))
    assert torch.equal(whole, cut) and torch.equal(*states)
    for r, part in enumerate(whole.split(LENS, dim=1)):
        want = torch.stack([PD.short_conv(h[s, starts[r]:starts[r] + LENS[r]].to(F64), w[s].to(F64)) for s in range(sets)])
        assert_close(part, want, 1e-6 if to == torch.float32 else 2.0 ** -8, f"request {r}")


@pytest.mark.parametrize("ti,to", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("d,taps,long", [(516, 2, 90), (520, 3, 300), (1024, 4, 300), (512, 4, 497), (512, 4, 498), (40, 2, 6600)])
def test_short_convolution_of_single_tokens_beside_a_prompt(ti, to, d, taps, long):
    """Eight tokens a thread, each its request's only one, at their first position, within the convolution's reach of it and behind it, then a prompt that
    begins inside a run: the bits and the states of the same requests in steps of fewer than 64 tokens, on both sides of the line for few channels."""
    from llama_cu_amd.kernels import ops
    sets, lens = 2, [1] * 13 + [long, 1]
    ctx = [k + (i % 4 if k == 1 else 0) for i, k in enumerate(lens)]
    h, w = rnd(sets, sum(lens), d, seed=11).to(ti).cuda(), rnd(sets, d, taps, seed=12, std=0.5).cuda().to(ti)
    before = rnd(len(lens), sets, taps - 1, d, seed=13).cuda()
    states = [before.clone() for _ in range(2)]
    run = lambda rows, state, step: ops.short_conv(rows.contiguous(), w, state, torch.empty(rows.shape, dtype=to, device="cuda"), step)
    whole = run(h, states[0], hand_step(lens, ctx, list(range(len(lens)))))
    parts = [run(h[:, :13], states[1], hand_step(lens[:13], ctx[:13], list(range(13))))]
    for a in range(0, long, 50):
        k = min(50, long - a)
        parts.append(run(h[:, 13 + a:13 + a + k], states[1], hand_step([k], [a + k], [13])))
    parts.append(run(h[:, -1:], states[1], hand_step([1], ctx[-1:], [14])))
    assert torch.equal(whole, torch.cat(parts, dim=1)) and torch.equal(*states)


@pytest.mark.parametrize("types", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("channels,taps,offset,bias,act", [(40, 2, 8, True, "silu"), (3072, 4, 0, False, "silu"), (1100, 3, 4, True, None), (40, 4, 3, True, None),
                                                           (38, 4, 0, False, None), (64, 6, 0, True, "silu")])
def test_causal_convolution(types, channels, taps, offset, bias, act):
    from llama_cu_amd.kernels import ops
    ti, to = types
    lens = [max(200, (1 << 20) // channels)] + LENS[1:]         # a million values
    x = rnd(sum(lens), channels + 8, seed=3).to(ti)
    w, b = rnd(channels, taps, seed=4, std=0.6).cuda(), (rnd(channels, seed=5, std=0.3).cuda() if bias else None)
    starts = [sum(lens[:r]) for r in range(len(lens))]

    def forward(parts, step, state):
        rows = torch.cat([x[starts[r] + a:starts[r] + e] for r, a, e in parts]).cuda()
        return ops.causal_conv(rows, offset, w, b, state, step, to, activation=act)

    states = [rnd(len(lens), taps - 1, channels, seed=6, std=9.0).cuda() for _ in range(2)]
    whole = forward([(r, 0, k) for r, k in enumerate(lens)], hand_step(lens, lens, list(range(len(lens)))), states[0])
    cut = in_portions(lens, lambda parts, step: forward(parts, step, states[1]), max(20, (1 << 18) // channels))
    assert torch.equal(whole, cut) and torch.equal(*states)
    for r, part in enumerate(whole.split(lens)):
        f64 = lambda t: t.cpu().to(F64).numpy()
        y = torch.from_numpy(PM.causal_conv(f64(x[starts[r]:starts[r] + lens[r], offset:offset + channels]), f64(w), f64(b) if bias else None))
        assert_close(part, y * torch.sigmoid(y) if act else y, 2e-6 if to == torch.float32 else 2.0 ** -8, f"request {r}")
