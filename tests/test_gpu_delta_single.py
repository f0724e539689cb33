"""Delta rules in steps in which every request feeds one token (kernels of their own) against the same tokens beside a request that feeds two, which go
through the scan: the same bits, outputs and states."""
import pytest
import torch

from test_gpu_divasun import TYPES, hand_step, rnd
from test_gpu_mufotar import built

pytestmark = pytest.mark.gpu

REQUESTS = 5


def steps(slots_of):
    """Three tokens of every request in steps of single tokens, then the same with a last request that feeds two a step: ``(q_lens, ctx, slots)``."""
    for k in range(3):
        ctx = [1 + k + 3 * (r % 2) for r in range(REQUESTS)]            # (some requests' first token, some with tokens before it)
        yield ([1] * REQUESTS, ctx, slots_of[:REQUESTS]), ([1] * REQUESTS + [2], ctx + [2 * k + 2], slots_of)


# every size of key channels; columns in whole sets of 128, with a rest of less than a wave's 32, fewer than a wave's, the most there are
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,dk,dv,rank", [(2, 128, 128, 64), (3, 32, 132, 3), (1, 64, 4, 1), (2, 96, 300, 9), (1, 128, 512, 33)])
def test_the_generalised_rule(dtype, heads, dk, dv, rank):
    from llama_cu_amd.kernels import build, ops
    assert build.load("delta_rule").lcu_delta_single_takes(heads, dk, dv) and not build.load("delta_rule").lcu_delta_single_takes(heads, dk + 16, dv)
    hk, hv, tdt = heads * dk, heads * dv, TYPES[dtype]
    off = {"r": 0, "k": hk, "v": 2 * hk, "g": 2 * hk + hv, "a": 2 * hk + 2 * hv, "l": 3 * hk + 2 * hv}
    args = (rnd(rank, hk, seed=3).cuda(), rnd(hk, seed=4).cuda(), rnd(hk, seed=5).cuda(), (rnd(hv, seed=6) + 1).cuda())
    a = rnd(REQUESTS + 1, heads, dk, dv, seed=7).cuda()
    b = a.clone()
    for k, (one, two) in enumerate(steps([3, 0, 5, 1, 4, 2])):
        rows = rnd(REQUESTS + 2, 3 * hk + 2 * hv + rank, seed=10 + k).to(tdt).cuda()
        got = ops.delta_rule(rows[:REQUESTS].contiguous(), off, *args, a, hand_step(*one), heads, dk, dv, 1e-4)
        want = ops.delta_rule(rows, off, *args, b, hand_step(*two), heads, dk, dv, 1e-4)
        assert torch.equal(got, want[:REQUESTS]) and torch.equal(a[[3, 0, 5, 1, 4]], b[[3, 0, 5, 1, 4]]), k


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,qk_heads,dk,dv,taps", [(4, 2, 128, 128, 4), (3, 3, 32, 132, 1), (2, 1, 64, 4, 2), (4, 1, 96, 300, 8), (1, 1, 128, 512, 3)])
def test_the_gated_rule(dtype, heads, qk_heads, dk, dv, taps):
    from llama_cu_amd.kernels import ops
    d, tdt = 56, TYPES[dtype]
    shape = {"hidden_size": d, "heads": heads, "qk_heads": qk_heads, "head_dim": dk, "value_dim": dv, "taps": taps, "norm_eps": 1e-5}
    from llama_cu_amd.parts import PartSpec, make_part
    names = make_part("mixer", PartSpec("gated_delta", shape)).tensors()
    part = built("mixer", "gated_delta", shape, {n: rnd(*t.shape, seed=k, std=t.shape[-1] ** -0.5 if len(t.shape) > 1 else 1.0) for k, (n, t) in enumerate(names.items())}, tdt)
    a, b = (part.cache_need().allocate(-1, 0, 0, REQUESTS + 1, tdt, torch.device("cuda")) for _ in range(2))
    a.state.copy_(rnd(*a.state.shape, seed=99))
    b.state.copy_(a.state)
    matrices = a.state[:, :part.state_size].view(-1, heads, dk, dv)
    for k, (one, two) in enumerate(steps([3, 0, 5, 1, 4, 2])):
        rows = rnd(REQUESTS + 2, d, seed=10 + k).to(tdt).cuda()
        assert ops.gated_delta_single_takes(hand_step(*one), matrices, heads, qk_heads, dk, dv, taps) == (a.state.stride(0) % 4 == 0)
        got = part.forward(rows[:REQUESTS].contiguous(), hand_step(*one), a)
        want = part.forward(rows, hand_step(*two), b)
        assert torch.equal(got, want[:REQUESTS]) and torch.equal(a.state[[3, 0, 5, 1, 4]], b.state[[3, 0, 5, 1, 4]]), k


def test_a_state_of_one_slot():
    shape = {"hidden_size": 24, "heads": 2, "qk_heads": 1, "head_dim": 32, "value_dim": 8, "taps": 3, "norm_eps": 1e-5}
    from llama_cu_amd.parts import PartSpec, make_part
    names = make_part("mixer", PartSpec("gated_delta", shape)).tensors()
    part = built("mixer", "gated_delta", shape, {n: rnd(*t.shape, seed=k) for k, (n, t) in enumerate(names.items())}, torch.float32)
    a, b = (part.cache_need().allocate(-1, 0, 0, n, torch.float32, torch.device("cuda")) for n in (1, 2))
    rows = rnd(4, 24, seed=9).cuda()
    want = part.forward(rows, hand_step([4], [4], [1]), b)
    got = torch.cat([part.forward(rows[k:k + 1].contiguous(), hand_step([1], [k + 1], [0]), a) for k in range(4)])
    assert torch.equal(got, want) and torch.equal(a.state[0], b.state[1])


def test_states_that_no_cache_holds():
    """A step whose states are streamed past the caches (48 MB and more) against its halves, whose are not: the same bits."""
    from llama_cu_amd.kernels import ops
    n, heads, dk, dv, rank = 25, 8, 128, 512, 5
    hk, hv = heads * dk, heads * dv
    off = {"r": 0, "k": hk, "v": 2 * hk, "g": 2 * hk + hv, "a": 2 * hk + 2 * hv, "l": 3 * hk + 2 * hv}
    args = (rnd(rank, hk, seed=3).cuda(), rnd(hk, seed=4).cuda(), rnd(hk, seed=5).cuda(), (rnd(hv, seed=6) + 1).cuda())
    gated = (rnd(heads, seed=13).cuda(), rnd(heads, seed=14).cuda(), rnd(dv, seed=15).cuda())
    channels = 2 * hk + hv
    conv_w = rnd(channels, 3, seed=16).cuda()
    rows, wide = rnd(n, 3 * hk + 2 * hv + rank, seed=7).cuda(), rnd(n, channels + 2 * heads + hv, seed=8).cuda()
    a = torch.randn(n, heads, dk, dv, generator=torch.Generator("cuda").manual_seed(9), device="cuda")
    slots = torch.randn(n, heads * dk * dv + 2 * channels, generator=torch.Generator("cuda").manual_seed(10), device="cuda")

    def run(first, last, state, both):
        step = hand_step([1] * (last - first), [1 + r % 3 for r in range(first, last)], list(range(first, last)))
        y = ops.delta_rule(rows[first:last].contiguous(), off, *args, state, step, heads, dk, dv, 1e-4)
        m = heads * dk * dv
        z = ops.gated_delta_single(wide[first:last].contiguous(), channels, channels + heads, channels + 2 * heads, conv_w, both[:, m:].view(n, 2, channels), *gated,
                                   both[:, :m].view(n, heads, dk, dv), step, heads, heads, dk, dv, 1e-4, torch.bfloat16)
        return y, z
    b, both = a.clone(), slots.clone()
    got = run(0, n, a, slots)
    halves = [run(0, 12, b, both), run(12, n, b, both)]
    for k in range(2):
        assert torch.equal(got[k], torch.cat([h[k] for h in halves]))
    assert torch.equal(a, b) and torch.equal(slots, both)


def test_steps_that_the_other_kernels_take_in_less_time():
    """Many heads of few columns, and few workgroups with the longest columns behind long ranks or the convolution of many channels: both sides of the lines."""
    from llama_cu_amd.kernels import build, ops
    lib = build.load("delta_rule")
    for (n, heads, dk, dv, rank), pays in [((200, 16, 128, 128, 64), 1), ((256, 64, 64, 4, 8), 0), ((16, 64, 64, 4, 8), 1), ((64, 64, 32, 16, 64), 1), ((65, 64, 32, 16, 64), 0),
                                           ((64, 16, 64, 16, 512), 0), ((63, 16, 64, 16, 512), 1), ((256, 32, 32, 32, 512), 0), ((256, 32, 32, 32, 256), 1), ((96, 32, 32, 32, 512), 1),
                                           ((256, 32, 128, 32, 512), 1), ((1, 8, 128, 512, 512), 0), ((1, 9, 128, 512, 512), 1), ((1, 8, 128, 512, 256), 1), ((1, 1, 128, 384, 512), 1)]:
        assert lib.lcu_delta_single_pays(n, heads, dk, dv, rank) == pays, (n, heads, dk, dv, rank)
    for (n, heads, qk_heads, dk, dv), pays in [((1, 32, 16, 128, 128), 1), ((200, 8, 2, 128, 128), 1), ((256, 64, 16, 64, 4), 0), ((32, 64, 16, 64, 4), 1), ((128, 16, 4, 128, 16), 1),
                                               ((129, 16, 4, 128, 16), 0), ((256, 64, 64, 64, 16), 1), ((1, 8, 1, 128, 512), 0), ((8, 8, 1, 128, 512), 0), ((9, 8, 1, 128, 512), 1),
                                               ((1, 8, 2, 128, 512), 0), ((5, 8, 2, 128, 512), 1), ((1, 8, 8, 128, 512), 1)]:
        assert lib.lcu_gated_delta_single_pays(n, heads, qk_heads, dk, dv) == pays, (n, heads, qk_heads, dk, dv)
    state = torch.zeros(64, 64, 64, 4, device="cuda")
    assert ops.gated_delta_single_takes(hand_step([1] * 32, [2] * 32, list(range(32))), state, 64, 16, 64, 4, 4)
    assert not ops.gated_delta_single_takes(hand_step([1] * 64, [2] * 64, list(range(64))), state, 64, 16, 64, 4, 4)


@pytest.mark.parametrize("n,part,heads,dk,dv,rank", [(65, 13, 64, 32, 4, 5), (9, 3, 2, 128, 512, 300)])
def test_single_tokens_that_go_the_other_way(n, part, heads, dk, dv, rank):
    """Of a step and its parts one side goes through the one kernel, the other through the three: the same bits."""
    from llama_cu_amd.kernels import build, ops
    lib = build.load("delta_rule")
    assert lib.lcu_delta_single_pays(n, heads, dk, dv, rank) != lib.lcu_delta_single_pays(part, heads, dk, dv, rank)
    hk, hv = heads * dk, heads * dv
    off = {"r": 0, "k": hk, "v": 2 * hk, "g": 2 * hk + hv, "a": 2 * hk + 2 * hv, "l": 3 * hk + 2 * hv}
    args = (rnd(rank, hk, seed=3).cuda(), rnd(hk, seed=4).cuda(), rnd(hk, seed=5).cuda(), (rnd(hv, seed=6) + 1).cuda())
    rows = rnd(n, 3 * hk + 2 * hv + rank, seed=7).cuda()
    a = rnd(n, heads, dk, dv, seed=8).cuda()
    b, ctx = a.clone(), [1 + r % 3 for r in range(n)]
    got = ops.delta_rule(rows, off, *args, a, hand_step([1] * n, ctx, list(range(n))), heads, dk, dv, 1e-4)
    want = torch.cat([ops.delta_rule(rows[f:f + part].contiguous(), off, *args, b, hand_step([1] * part, ctx[f:f + part], list(range(f, f + part))), heads, dk, dv, 1e-4)
                      for f in range(0, n, part)])
    assert torch.equal(got, want) and torch.equal(a, b)
