"""The delta rules' chunks (csrc/kernels/delta_chunks.h) against the recurrences in 64 bits, beside the token-by-token scan:
at the chunks' edges, from states of earlier portions, and where decays are as small as they can be."""
from __future__ import annotations

import math

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import hand_step, rnd

pytestmark = pytest.mark.gpu
F64 = torch.float64
EPS = 1e-5


def unit_rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def walk(w, al, u, k, v, r):
    """o [T, heads, dv] and the last state of S <- diag(w) S - al (u^T S) + k v^T from zeros; all [T, heads, .]."""
    S = torch.zeros(w.shape[1], w.shape[2], v.shape[2], dtype=F64)
    outs = []
    for t in range(w.shape[0]):
        seen = u[t][:, None, :] @ S
        S = w[t][:, :, None] * S - al[t][:, :, None] * seen + k[t][:, :, None] * v[t][:, None, :]
        outs.append((r[t][:, None, :] @ S)[:, 0])
    return torch.stack(outs), S


def general(T, heads, dim, rank, decay, seed):
    """(arguments of ops.delta_rule, a row maker, the expected outputs and state); ``decay``: added to w0."""
    hd = heads * dim
    off = {"r": 0, "k": hd, "v": 2 * hd, "g": 3 * hd, "a": 4 * hd, "l": 5 * hd}
    proj = rnd(T, 5 * hd + rank, seed=seed).bfloat16()
    w2, w0, ab, nw = rnd(hd, rank, seed=3), rnd(hd, seed=4) + decay, rnd(hd, seed=5), rnd(hd, seed=6) * 0.1 + 1
    x = proj.to(F64)
    r, k, v, g, a = (x[:, off[c]:off[c] + hd].view(T, heads, dim) for c in "rkvga")
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(x[:, 5 * hd:]) @ w2.to(F64).T + w0.to(F64))).view(T, heads, dim)
    u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    o, S = walk(w, torch.sigmoid(a + ab.to(F64).view(heads, dim)) * u, u, k, v, r)
    want = unit_rms(o).reshape(T, hd) * nw.to(F64) * torch.sigmoid(g.reshape(T, hd))
    return (off, w2.t().contiguous().cuda(), w0.cuda(), ab.cuda(), nw.cuda()), proj, want, S


def run_general(args, proj, heads, dim, portions):
    """Outputs and last state of the rows in portions, from a slot that holds other values; a short request walks beside."""
    from llama_cu_amd.kernels import ops
    state = torch.full((3, heads, dim, dim), 7.0, device="cuda")
    outs, at = [], 0
    for n in portions:
        rows = torch.cat([proj[:2], proj[at:at + n]]).cuda()
        outs.append(ops.delta_rule(rows, *args, state, hand_step([2, n], [2, at + n], [0, 2]), heads, dim, dim, EPS)[2:].clone())
        at += n
    assert (state[1] == 7.0).all()
    return torch.cat(outs), state[2]


@pytest.mark.parametrize("heads,dim,portions,decay", [
    (2, 128, [64], 0.0), (1, 128, [65, 63, 64], 0.0), (2, 128, [129], 9.0), (2, 64, [127, 1, 66], -3.0),
    (3, 20, [200, 129], 0.0), (1, 72, [128, 128], 9.0), (2, 16, [191], -9.0), (1, 112, [100, 70], 0.0),
    (2, 128, [128, 127, 130], 0.0), (1, 64, [192, 1, 193], 3.0), (1, 48, [255], 0.0)])
def test_the_generalised_rule_in_chunks(heads, dim, portions, decay):
    """``decay`` 9: every decay is as small as the rule allows (0.545 a token); -9: close to 1."""
    args, proj, want, S = general(sum(portions), heads, dim, 3, decay, seed=11)
    got, state = run_general(args, proj, heads, dim, portions)
    # the state: sums of some hundred 32-bit products of either sign, 2e-7 to 17e-7 of the largest value off as measured (the
    # scan's 2e-7 to 18e-7); the outputs are rounded to 8 bits: half a unit of the last is up to 2^-8 of the value, and what
    # the 32-bit value is off adds to it
    assert_close(state, S, 5e-6, "state")
    assert_close(got, want, 2.0 ** -8 + 1e-5, "outputs")


def gated(T, heads, qk_heads, dk, dv, gate, seed):
    width, hv = 2 * qk_heads * dk + heads * dv, heads * dv
    qkv = rnd(T, width, seed=seed)
    rows = rnd(T, 2 * heads + hv, seed=seed + 1)                        # a, b, gate
    a_log, bias, weight = rnd(heads, seed=7), rnd(heads, seed=8) + gate, rnd(dv, seed=9) * 0.1 + 1
    x, y = qkv.to(F64), rows.to(F64)
    rep = heads // qk_heads
    q, k = (x[:, i * qk_heads * dk:(i + 1) * qk_heads * dk].view(T, qk_heads, dk) for i in (0, 1))
    q, k = ((z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(rep, 1) for z in (q, k))
    v = x[:, 2 * qk_heads * dk:].view(T, heads, dv)
    g = torch.exp(-torch.exp(a_log.to(F64)) * torch.nn.functional.softplus(y[:, :heads] + bias.to(F64)))[..., None]
    beta = torch.sigmoid(y[:, heads:2 * heads])[..., None]
    o, S = walk(g.expand(T, heads, dk), beta * g * k, k, k, beta * v, q * dk ** -0.5)
    z = y[:, 2 * heads:].view(T, heads, dv)
    want = (unit_rms(o) * weight.to(F64) * (z * torch.sigmoid(z))).reshape(T, hv)
    return (a_log.cuda(), bias.cuda(), weight.cuda()), qkv, rows, want, S


@pytest.mark.parametrize("heads,qk_heads,dk,dv,portions,gate", [
    (2, 1, 128, 128, [64], 0.0), (2, 2, 128, 128, [65, 63, 130], -4.0), (4, 2, 64, 20, [127, 1, 66], 0.0), (1, 1, 24, 40, [200], 80.0),
    (3, 1, 72, 136, [128, 65], 3.0), (2, 2, 16, 16, [191], -9.0), (1, 1, 128, 272, [100], 0.0),
    (2, 1, 128, 128, [128, 127, 191], -4.0), (1, 1, 64, 20, [192, 1, 193], 0.0), (1, 1, 128, 272, [255], 0.0)])
def test_the_gated_rule_in_chunks(heads, qk_heads, dk, dv, portions, gate):
    """``gate`` 80: a token's decay is 0 in 32 bits; -9: it is 1 but for the fourth digit."""
    from llama_cu_amd.kernels import ops
    T = sum(portions)
    args, qkv, rows, want, S = gated(T, heads, qk_heads, dk, dv, gate, seed=21)
    state = torch.full((3, heads, dk, dv), 7.0, device="cuda")
    outs, at = [], 0
    for n in portions:
        pick = torch.cat([torch.arange(at, at + n), torch.arange(3)])
        outs.append(ops.gated_delta_rule(qkv[pick].cuda(), rows[pick].cuda(), 0, heads, 2 * heads, *args, state,
                                         hand_step([n, 3], [at + n, 3], [1, 2]), heads, qk_heads, dk, dv, EPS, torch.bfloat16)[:n].clone())
        at += n
    assert (state[0] == 7.0).all()
    assert_close(state[1], S, 5e-6, "state")
    assert_close(torch.cat(outs), want, 2.0 ** -8 + 1e-5, "outputs")


def rms_off(got, want):
    return float((got.cpu().to(F64) - want).norm() / want.norm())


def raw(kind, dim, decay, T, chunks, seed):
    """How far the last state and the outputs, both in 32 bits, are off the recurrence in 64 bits (2-norm): scanned, or in chunks."""
    import ctypes
    from llama_cu_amd.kernels import build, ops
    lib, p, heads, step = build.load("delta_rule"), ops._ptr, 2, hand_step([T], [T], [0])
    hv = heads * dim
    state, o, out = torch.zeros(1, heads, dim, dim, device="cuda"), torch.empty(T, hv, device="cuda"), torch.empty(T, hv, device="cuda")
    lib.lcu_delta_work_floats.restype = ctypes.c_longlong
    floats = lib.lcu_delta_work_floats(T, 1, heads, dim, dim, int(kind == "gated"))
    assert floats > 0
    work = torch.empty(floats, device="cuda") if chunks else None
    steps = (p(step.q_start), p(step.ctx_len), p(step.state_slot), T, 1, heads)
    if kind == "gated":
        args, qkv, rows, want, S = gated(T, heads, heads, dim, dim, decay, seed)
        q, r = qkv.cuda(), rows.cuda()
        prep, vb = torch.empty(T, heads, 2 * dim + 4, device="cuda"), torch.empty(T, hv, device="cuda")
        rc = lib.lcu_gated_delta_rule(p(q), p(r), r.stride(0), 0, heads, 2 * heads, *(p(a) for a in args), p(prep), p(vb), p(work), p(o), p(state),
                                      ctypes.c_longlong(hv * dim), p(out), ops._type(out, "out"), *steps, heads, dim, dim, ctypes.c_float(EPS), ops._stream())
    else:
        (off, *args), proj, want, S = general(T, heads, dim, 8, decay, seed)
        rows = proj.float().cuda()
        prep = torch.empty(T, heads, 5, dim, device="cuda")
        rc = lib.lcu_delta_rule(p(rows), ops._type(rows, "rows"), rows.stride(0), *(off[c] for c in "rkvgal"), *(p(a) for a in args), p(prep), p(work),
                                p(o), p(state), p(out), *steps, dim, dim, 8, ctypes.c_float(EPS), ops._stream())
    assert rc == 0
    return rms_off(out, want), rms_off(state[0], S)


@pytest.mark.parametrize("kind,decay", [("general", 9.0), ("general", 0.0), ("general", -3.0), ("general", -9.0), ("gated", 3.0), ("gated", 0.0),
                                        ("gated", -4.0), ("gated", -9.0)])
@pytest.mark.parametrize("dim", [64, 128])
def test_chunks_are_no_further_off_than_the_scan(kind, decay, dim):
    """Decays from the smallest to almost 1: what chunks make, before anything is rounded to bfloat16, beside what the scan makes (mean of three
    seeds; a tenth and 1e-8 for what seeds differ by)."""
    scan, chunk = ([raw(kind, dim, decay, 320, c, s) for s in (1, 2, 3)] for c in (False, True))
    for what, a, b in zip(("outputs", "state"), zip(*scan), zip(*chunk)):
        assert sum(b) <= 1.1 * sum(a) + 3e-8, f"{what}: scanned {sum(a) / 3:.2e}, in chunks {sum(b) / 3:.2e}"


@pytest.mark.parametrize("dim,heads,requests", [(16, 40, 4), (64, 8, 17)])
def test_many_long_requests_of_small_heads_are_scanned(dim, heads, requests):
    """More long requests than chunks are good for: the bits that every request has scanned alone in portions too short for chunks."""
    from llama_cu_amd.kernels import ops
    T = 130
    args, qkv, rows, want, S = gated(T, heads, heads, dim, dim, -4.0, seed=3)
    q, r = qkv.cuda(), rows.cuda()
    state = torch.full((requests, heads, dim, dim), 7.0, device="cuda")
    all_of = ops.gated_delta_rule(q.repeat(requests, 1), r.repeat(requests, 1), 0, heads, 2 * heads, *args, state,
                                  hand_step([T] * requests, [T] * requests, list(range(requests))), heads, heads, dim, dim, EPS, torch.bfloat16)
    alone, one = torch.full((1, heads, dim, dim), 7.0, device="cuda"), []
    for a, b in ((0, 60), (60, T)):
        one.append(ops.gated_delta_rule(q[a:b].contiguous(), r[a:b].contiguous(), 0, heads, 2 * heads, *args, alone, hand_step([b - a], [b], [0]),
                                        heads, heads, dim, dim, EPS, torch.bfloat16))
    one = torch.cat(one)
    for k in range(requests):
        assert torch.equal(all_of[k * T:(k + 1) * T], one) and torch.equal(state[k], alone[0])


@pytest.mark.parametrize("what,value", [("r", math.inf), ("k", math.nan), ("v", math.inf), ("v", math.nan), ("a", math.nan), ("l", math.nan),
                                        ("k", 1e30), ("v", -1e35)])
@pytest.mark.parametrize("dim", [40, 128])
def test_the_generalised_rule_passes_nothing_back_in_time(what, value, dim):
    """An infinity, a NaN or a number whose products overflow in one token of 200: in chunks the tokens before it, the other heads and the other
    request are what they are without it, and the token and those behind it what the scan makes of them."""
    heads, T, at = 2, 200, 100
    args, proj, want, S = general(T, heads, dim, 3, 0.0, seed=11)
    proj[at, args[0][what] + (0 if what == "l" else dim + 3)] = value                   # (a channel of the second head; l reaches both)
    whole, state = run_general(args, proj, heads, dim, [T])
    cut, state2 = run_general(args, proj, heads, dim, [60, 60, 60, 20])
    assert_close(whole[:at], want[:at], 2.0 ** -8 + 1e-5, "before")
    if what != "l":
        assert_close(whole[:, :dim], want[:, :dim], 2.0 ** -8 + 1e-5, "the other head")
    same_but_for_rounding(whole, cut, 2.0 ** -8)
    same_but_for_rounding(state, state2, 1e-5)


def same_but_for_rounding(a, b, rel):
    a, b = a.cpu().to(F64), b.cpu().to(F64)
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
    fine = a.isfinite()
    if fine.any():
        assert float((a[fine] - b[fine]).abs().max()) <= rel * max(float(b[fine].abs().max()), 1e-30)


@pytest.mark.parametrize("what,value", [("q", math.nan), ("k", math.inf), ("v", math.inf), ("a", math.nan), ("a", math.inf), ("b", math.nan), ("v", 1e30)])
def test_the_gated_rule_passes_nothing_back_in_time(what, value):
    from llama_cu_amd.kernels import ops
    heads, dk, dv, T, at = 2, 64, 24, 200, 100
    args, qkv, rows, want, S = gated(T, heads, heads, dk, dv, -2.0, seed=21)
    if what in "qkv":
        qkv[at, {"q": 0, "k": heads * dk, "v": 2 * heads * dk}[what] + (dv if what == "v" else dk) + 3] = value
    else:
        rows[at, {"a": 0, "b": heads}[what] + 1] = value
    outs = []
    for portions in ([T], [60, 60, 60, 20]):
        state, got, n0 = torch.full((2, heads, dk, dv), 7.0, device="cuda"), [], 0
        for n in portions:
            got.append(ops.gated_delta_rule(qkv[n0:n0 + n].cuda(), rows[n0:n0 + n].cuda(), 0, heads, 2 * heads, *args, state,
                                            hand_step([n], [n0 + n], [1]), heads, heads, dk, dv, EPS, torch.bfloat16))
            n0 += n
        outs.append((torch.cat(got), state[1]))
    assert_close(outs[0][0][:at], want[:at], 2.0 ** -8 + 1e-5, "before")
    assert_close(outs[0][0][:, :dv], want[:, :dv], 2.0 ** -8 + 1e-5, "the other head")
    for a, b, rel in zip(*outs, (2.0 ** -8, 1e-5)):
        same_but_for_rounding(a, b, rel)


@pytest.mark.parametrize("heads,dk,dv,lens,chunked", [
    (2, 128, 128, [256, 257, 255, 193], True), (1, 128, 272, [400, 64, 63, 1], True), (3, 64, 20, [1, 320, 129, 7], True), (2, 40, 40, [64, 63, 65], True),
    (4, 16, 48, [500, 100], True), (2, 128, 128, [100, 64], False), (2, 64, 64, [63, 1], False), (32, 16, 16, [65] * 5, False)])
def test_long_and_short_requests_in_a_step(heads, dk, dv, lens, chunked):
    """Requests of chunks and of the scan side by side, where chunks pay and where they do not (then each has the bits that it has alone)."""
    from llama_cu_amd.kernels import ops
    n = len(lens)
    each = [gated(T, heads, heads, dk, dv, -2.0, seed=31 + 2 * r) for r, T in enumerate(lens)]
    args, step = each[0][0], hand_step(lens, lens, list(range(n)))
    assert ops.plan_delta(step, heads, dk, dv, True).chunked == chunked
    state = torch.full((n, heads, dk, dv), 7.0, device="cuda")
    out = ops.gated_delta_rule(torch.cat([e[1] for e in each]).cuda(), torch.cat([e[2] for e in each]).cuda(), 0, heads, 2 * heads, *args, state, step,
                               heads, heads, dk, dv, EPS, torch.bfloat16).split(lens)
    for r, (_, qkv, rows, want, S) in enumerate(each):
        assert_close(state[r], S, 5e-6, f"state {r}")
        assert_close(out[r], want, 2.0 ** -8 + 1e-5, f"outputs {r}")
        if not chunked:
            alone, got = torch.full((1, heads, dk, dv), 7.0, device="cuda"), []
            for at in range(0, lens[r], 50):
                to = min(lens[r], at + 50)
                got.append(ops.gated_delta_rule(qkv[at:to].cuda(), rows[at:to].cuda(), 0, heads, 2 * heads, *args, alone, hand_step([to - at], [to], [0]),
                                                heads, heads, dk, dv, EPS, torch.bfloat16))
            assert torch.equal(torch.cat(got), out[r]) and torch.equal(alone[0], state[r])


@pytest.mark.parametrize("name", ["B", "D"])
def test_steps_of_equal_sizes_with_and_without_chunks(name):
    """Captured steps of 126 tokens and two requests, some of which go through chunks: each kind replays its own launches."""
    from divasun_common import tokens_of
    from test_gpu_divasun import model, runner_for
    cfg, _, folder = model(name)
    kinds = [[63, 63], [125, 1], [1, 125], [63, 63], [124, 2]] * 3

    def run(use_graphs):
        r, outs = runner_for(folder, "bfloat16", use_graphs=use_graphs), []
        for i, lens in enumerate(kinds):
            toks = [tokens_of(cfg["vocab"], n, 100 * i + n + k) for k, n in enumerate(lens)]
            outs.append(r.step([2 * i, 2 * i + 1], toks).float().cpu())
            torch.cuda.synchronize()
            for rid in (2 * i, 2 * i + 1):                   # and a step of single tokens on the states
                outs.append(r.step([rid], [[5]]).float().cpu())
                r.end(rid)
        return outs, r
    (eager, _), (graphed, r) = run(False), run(True)
    assert sum(r.step_graph_replays.values()) >= (len(kinds) - 4 if name == "D" else 1) and len(r._step_graphs) >= 2
    for i, (a, b) in enumerate(zip(eager, graphed)):
        assert torch.isfinite(a).all() and torch.equal(a, b), f"step {i}"
