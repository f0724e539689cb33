"""The recurrent unit's gates on the matrix instruction, and its steps of single tokens in one kernel, against the recurrence in 64 bits."""
from __future__ import annotations

import math

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, hand_step, rnd

pytestmark = pytest.mark.gpu


class Unit:
    def __init__(self, width, blocks, taps, seed=1, offsets=(3, 5)):
        bs = width // blocks
        self.y_off, self.x_off = offsets[0], width + offsets[1]
        self.width, self.blocks, self.taps = width, blocks, taps
        self.bias = rnd(2 * width + 8, seed=seed, std=0.3)
        self.conv_w, self.conv_b = rnd(width, taps, seed=seed + 1, std=0.5), rnd(width, seed=seed + 2, std=0.3)
        self.wa, self.wi = (rnd(blocks, bs, bs, seed=seed + k, std=2 / math.sqrt(bs)) for k in (3, 4))
        self.ba, self.bi, self.lam = rnd(width, seed=seed + 5), rnd(width, seed=seed + 6), rnd(width, seed=seed + 7, std=1.5) - 2.0

    def args(self):
        from llama_cu_amd.kernels import ops
        self.gates = ops.pack_rglru_gates(*(t.transpose(1, 2).contiguous().cuda() for t in (self.wa, self.wi)))
        g = [t.cuda() for t in (self.bias, self.conv_w, self.conv_b, self.wa.transpose(1, 2).contiguous(), self.wi.transpose(1, 2).contiguous(),
                                self.ba, self.bi, self.lam)]
        return (self.y_off, self.x_off, *g, 8.0)

    def want(self, rows, state=None):
        """One request's tokens from the state's rows (none: from the beginning): outputs and the state behind them."""
        w, taps = self.width, self.taps
        x = rows.to(F64) + self.bias.to(F64)
        y, x = x[:, self.y_off:self.y_off + w], x[:, self.x_off:self.x_off + w]
        before = torch.zeros(taps - 1, w, dtype=F64) if state is None else state[:taps - 1].to(F64)
        S = torch.zeros(w, dtype=F64) if state is None else state[taps - 1].to(F64)
        x = torch.cat([before, x], 0)
        out = []
        for t in range(rows.shape[0]):
            u = self.conv_b.to(F64) + (x[t:t + taps] * self.conv_w.to(F64).t()).sum(0)
            r, i = (torch.sigmoid(torch.einsum("bi,boi->bo", u.view(self.blocks, -1), m.to(F64)).reshape(w) + b.to(F64))
                    for m, b in ((self.wa, self.ba), (self.wi, self.bi)))
            a = torch.exp(-8.0 * r * torch.nn.functional.softplus(self.lam.to(F64)))
            S = a * S + torch.sqrt(-torch.expm1(2 * torch.log(a))) * i * u
            out.append(S * torch.nn.functional.gelu(y[t], approximate="tanh"))
        return torch.stack(out), torch.cat([x[rows.shape[0]:], S[None]], 0)


@pytest.mark.parametrize("width,blocks,taps", [(64, 4, 4), (96, 2, 1), (256, 2, 3), (384, 2, 4), (128, 1, 2), (2048, 16, 4), (40, 2, 4), (64, 1, 5)])
@pytest.mark.parametrize("n", [1, 7, 16, 17, 64])
@pytest.mark.parametrize("offsets", [(3, 5), (0, 8)])
@pytest.mark.parametrize("out_type", [torch.bfloat16, torch.float32])
def test_steps_of_single_tokens(width, blocks, taps, n, offsets, out_type):
    """Requests at their first token, within the convolution's reach of it and far behind it, from slots in no order; the other slots stay.  With
    32-bit outputs the bits are those of the same tokens without the packed gates, alone or in portions."""
    from llama_cu_amd.kernels import ops
    unit = Unit(width, blocks, taps, offsets=offsets)
    args = unit.args()
    rows = rnd(n, 2 * width + 8, seed=20)
    ctx = [1 + (3 * i) % 7 for i in range(n)]
    slots = torch.randperm(n + 2, generator=torch.Generator().manual_seed(21))[:n].tolist()
    old = rnd(n + 2, taps, width, seed=22)
    state = old.clone().cuda()
    got = ops.rglru(rows.cuda(), *args, state, hand_step([1] * n, ctx, slots), out_type, gates=unit.gates)
    if out_type == torch.float32:
        plain = old.clone().cuda()
        assert torch.equal(got, ops.rglru(rows.cuda(), *args, plain, hand_step([1] * n, ctx, slots), out_type)) and torch.equal(state, plain)
    for i in range(n):
        have = old[slots[i]].clone()
        for k in range(taps - 1):                       # rows of tokens before the request's first are zeros, whatever the slot holds
            if taps - 1 - k > ctx[i] - 1:
                have[k] = 0.0
        want, after = unit.want(rows[i:i + 1], have if ctx[i] > 1 else None)
        assert_close(got[i:i + 1], want, 2e-5 if out_type == torch.float32 else 2.0 ** -8, f"request {i}")
        assert_close(state[slots[i]], after, 2e-5, f"state {i}")
    others = [s for s in range(n + 2) if s not in slots]
    assert torch.equal(state[others].cpu(), old[others])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,blocks,taps", [(64, 4, 4), (512, 4, 3), (192, 1, 4), (1024, 16, 4), (256, 2, 6)])
@pytest.mark.parametrize("lens", [[2, 3], [70, 1, 5], [200, 64, 33, 1000]])
def test_many_tokens_and_then_one(width, blocks, taps, lens, dtype):
    """Requests of several lengths in one step (tiles of 16 tokens and of 64, that begin inside a request and before one), then a token each:
    32-bit sums of up to 192 terms and up to 1,000 steps of a recurrence that forgets, so 1e-4 of the largest output."""
    from llama_cu_amd.kernels import ops
    unit = Unit(width, blocks, taps)
    args = unit.args()
    rows = [rnd(k, 2 * width + 8, seed=30 + i).to(dtype) for i, k in enumerate(lens)]
    more = rnd(len(lens), 2 * width + 8, seed=50).to(dtype)
    state = torch.full((len(lens) + 1, taps, width), 5.0, device="cuda")
    slots = list(range(len(lens), 0, -1))
    out_type, rel = (torch.float32, 1e-4) if dtype == torch.float32 else (torch.bfloat16, 2.0 ** -7)
    got = ops.rglru(torch.cat(rows).cuda(), *args, state, hand_step(lens, lens, slots), out_type, gates=unit.gates)
    then = ops.rglru(more.cuda(), *args, state, hand_step([1] * len(lens), [k + 1 for k in lens], slots), out_type, gates=unit.gates)
    for i, (k, part) in enumerate(zip(lens, got.split(lens))):
        want, after = unit.want(torch.cat([rows[i], more[i:i + 1]]).float())
        assert_close(part, want[:k], rel, f"request {i}")
        assert_close(then[i:i + 1], want[k:], rel, f"request {i}, the token behind")
        assert_close(state[slots[i]], after, 1e-4, f"state {i}")


def both_ways(unit, args, rows, state, lens, ctx, slots, out_type):
    """The same step with the packed gates and without them: outputs and the states behind it."""
    from llama_cu_amd.kernels import ops
    got = []
    for gates in (unit.gates, None):
        after = state.clone()
        got.append((ops.rglru(rows, *args, after, hand_step(lens, ctx, slots), out_type, gates=gates), after))
    return got


@pytest.mark.parametrize("types", [(torch.float32, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("width,blocks,taps", [(64, 2, 4), (16, 1, 4), (128, 2, 3), (96, 2, 2), (96, 1, 4), (2048, 16, 4), (192, 1, 1), (320, 2, 4), (128, 2, 5)])
def test_bits_do_not_depend_on_the_kernel(width, blocks, taps, types):
    """The kernels that take the packed gates add a token's products in the order of those without: single tokens up to 64 (eight parts of the input channels) and
    beyond (one), four channels a thread and one, blocks whose parts are no whole matrix instruction; portions whose tokens come in tiles of 16."""
    ti, to = types
    for offsets in ((0, 8), (3, 5)):
        unit = Unit(width, blocks, taps, offsets=offsets)
        args = unit.args()
        for n in (1, 5, 64, 65, 130):
            rows, old = rnd(n, 2 * width + 8, seed=60).to(ti).cuda(), rnd(n, taps, width, seed=61).cuda()
            (a, sa), (b, sb) = both_ways(unit, args, rows, old, [1] * n, [1 + (3 * i) % 7 for i in range(n)], list(range(n))[::-1], to)
            assert torch.equal(a, b) and torch.equal(sa, sb), (offsets, n)
        lens = [41, 1, 2, 30, 1]
        rows, old = rnd(sum(lens), 2 * width + 8, seed=62).to(ti).cuda(), rnd(5, taps, width, seed=63).cuda()
        (a, sa), (b, sb) = both_ways(unit, args, rows, old, lens, [41, 4, 2, 90, 2], [4, 2, 0, 1, 3], to)
        assert torch.equal(a, b) and torch.equal(sa, sb), offsets


@pytest.mark.parametrize("types", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("width,blocks,taps", [(2048, 16, 4), (1280, 16, 4), (3072, 16, 3), (1024, 64, 4), (768, 16, 2), (1024, 16, 6)])
def test_bits_of_many_tokens(width, blocks, taps, types):
    """64 tokens a workgroup, whose convolution a thread walks in one run, in two and in pieces that are no whole batch of sixteen."""
    ti, to = types
    unit = Unit(width, blocks, taps, offsets=(0, 8))
    lens = [700, 1, 3, 64, 560]
    rows, old = rnd(sum(lens), 2 * width + 8, seed=64).to(ti).cuda(), rnd(5, taps, width, seed=65).cuda()
    (a, sa), (b, sb) = both_ways(unit, unit.args(), rows, old, lens, [700, 2, 40, 66, 560], [0, 3, 1, 4, 2], to)
    assert torch.equal(a, b) and torch.equal(sa, sb)


@pytest.mark.parametrize("width,blocks", [(32, 2), (96, 2), (160, 2), (224, 2), (64, 2), (128, 2), (192, 2), (256, 2)])
@pytest.mark.parametrize("n", [1, 32, 33, 130])
@pytest.mark.parametrize("taps", [1, 4])
def test_single_tokens_by_the_size_of_a_block(width, blocks, n, taps):
    """Blocks of every number of sixteens up to eight, for which a workgroup has one, two, three, four or eight waves: the bits of the kernels without packed gates."""
    unit = Unit(width, blocks, taps, offsets=(0, 0))
    args, rows, state = unit.args(), rnd(n, 2 * width + 8, seed=20).cuda(), rnd(n + 1, taps, width, seed=22).cuda()
    (got, after), (want, kept) = both_ways(unit, args, rows, state, [1] * n, [1 + (3 * i) % 7 for i in range(n)], list(range(n)), torch.float32)
    assert torch.isfinite(got).all() and torch.equal(got, want) and torch.equal(after, kept)
