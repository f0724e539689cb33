"""Retention in steps of single tokens: one kernel in the place of three, with the same bits."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import TYPES, hand_step, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,d,dv,rot,inter", [(3, 128, 128, 128, False), (2, 64, 132, 32, True), (1, 20, 4, 20, False), (2, 68, 512, 0, False),
                                                 (1, 128, 36, 64, True)])
def test_the_same_bits_as_beside_a_longer_request(dtype, heads, d, dv, rot, inter):
    """The same tokens, at a request's first position and later ones, in a step of single tokens and in one where another request feeds two: outputs and
    states bit for bit; slots that no request holds are left alone."""
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.base import BuildContext
    from llama_cu_amd.parts.position import Rotary
    tdt, n = TYPES[dtype], 5
    hk, hv = heads * d, heads * dv
    off = {"q": 3, "k": 3 + hk, "v": 3 + 2 * hk, "g": 3 + 2 * hk + hv}
    rows = rnd(n + 2, 3 + 2 * hk + 2 * hv, seed=1).cuda()
    decay = torch.tensor([0.9, 0.999, 0.5][:heads]).cuda()
    kw = {}
    if rot:
        part = Rotary(d, 1000.0, 64, interleaved=inter, rot_dim=rot)
        part.load({}, BuildContext(tdt, torch.device("cuda"), 64, 16))
        cos, sin, _, _ = part.rotary_tables()
        kw = dict(cos=cos, sin=sin, rot_dim=rot, pairing=1 if inter else 0)
    start = rnd(n + 3, heads, d, dv, seed=2).cuda()
    ctx, slots = [1, 2, 17, 64, 9], [4, 0, 6, 2, 1]
    one, two = start.clone(), start.clone()
    got = ops.retention(rows[:n], off, decay, one, hand_step([1] * n, ctx, slots), heads, d, dv, 0.3, 1e-5, tdt, **kw)
    want = ops.retention(rows, off, decay, two, hand_step([1] * n + [2], ctx + [2], slots + [7]), heads, d, dv, 0.3, 1e-5, tdt, **kw)
    assert torch.equal(got, want[:n]) and torch.isfinite(got.float()).all()
    assert torch.equal(one[:7], two[:7]) and torch.equal(one[7], start[7]) and torch.equal(one[3], start[3]) and torch.equal(one[5], start[5])
    assert not torch.equal(one[4], start[4])


def test_a_request_that_feeds_nothing():
    """A step of single tokens in which a request has none: its rows are not the requests' in order, so it goes through the kernels for any step; the others' outputs and states are
    those of a step without it, its own state stays."""
    from llama_cu_amd.kernels import ops
    heads, d, dv = 2, 64, 64
    hk, hv = heads * d, heads * dv
    off = {"q": 0, "k": hk, "v": 2 * hk, "g": 2 * hk + hv}
    rows, decay, start = rnd(2, 2 * hk + 2 * hv, seed=1).cuda(), torch.tensor([0.9, 0.999]).cuda(), rnd(3, heads, d, dv, seed=2).cuda()
    one, two = start.clone(), start.clone()
    got = ops.retention(rows, off, decay, one, hand_step([1, 0, 1], [5, 4, 1], [2, 0, 1]), heads, d, dv, 0.3, 1e-5, torch.float32)
    want = ops.retention(rows, off, decay, two, hand_step([1, 1], [5, 1], [2, 1]), heads, d, dv, 0.3, 1e-5, torch.float32)
    assert torch.equal(got, want) and torch.equal(one, two) and torch.equal(one[0], start[0])
