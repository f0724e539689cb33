"""Layer norms of rows at the edges of the kernels' sizes, four elements at a time and one at a time (rows that are not aligned for
four), with planes of deltas; and the fused kernel for single tokens with other than four taps."""
from __future__ import annotations

import pytest
import torch

import plain_divasun as P
from divasun_common import assert_close
from test_gpu_divasun import F64, TYPES, hand_step, rnd

pytestmark = pytest.mark.gpu


def shifted(t, by):
    """The same values at an address ``by`` elements further."""
    room = torch.empty(t.numel() + by, dtype=t.dtype, device="cuda")
    room[by:] = t.reshape(-1).cuda()
    return room[by:].view(t.shape)


@pytest.mark.parametrize("out_type", ["float32", "bfloat16"])
@pytest.mark.parametrize("d,by", [(3, 0), (4, 0), (100, 1), (1026, 0), (2048, 0), (2048, 2), (2052, 0), (4096, 0), (4096, 1), (4100, 0)])
def test_layer_norm_rows(d, by, out_type):
    from llama_cu_amd.kernels import ops
    n, planes, tdt = 3, 2, TYPES[out_type]
    x, delta = rnd(n, d, seed=1) + 2.0, rnd(planes, n, d, seed=2)
    ws = [rnd(d, seed=k) for k in (3, 4, 5, 6)]
    xs, out, out2 = shifted(x, by), torch.empty(n, d, dtype=tdt, device="cuda"), torch.empty(n, d, dtype=tdt, device="cuda")
    ops.layernorm(xs, ws[0].cuda(), ws[1].cuda(), 1e-5, out, delta=delta.cuda(), weight2=ws[2].cuda(), bias2=ws[3].cuda(), out2=out2)
    want = (x + delta[0] + delta[1]).to(F64)
    assert_close(xs, want, 1e-6, "sum")
    rel = 1e-5 if out_type == "float32" else 2.0 ** -8 + 1e-5        # 32-bit sums; half a unit of bfloat16's last place
    assert_close(out, P.layer_norm(want, ws[0].to(F64), ws[1].to(F64), 1e-5), rel, "first")
    assert_close(out2, P.layer_norm(want, ws[2].to(F64), ws[3].to(F64), 1e-5), rel, "second")


@pytest.mark.parametrize("d,taps,by", [(72, 1, 0), (72, 3, 0), (2048, 4, 0), (2048, 4, 1), (2044, 8, 0), (513, 4, 0)])
def test_norm_and_convolution_of_single_tokens(d, taps, by):
    """Five tokens of two requests one after the other, from slots that hold other values, against the convolution of the whole."""
    from llama_cu_amd.kernels import ops
    rows = [rnd(5, d, seed=10 + r) for r in range(2)]
    w, b = [rnd(d, seed=k).cuda() for k in (3, 4)], [rnd(d, seed=k).cuda() for k in (5, 6)]
    cw = rnd(2, d, taps, seed=7, std=0.5)
    state = torch.full((3, 2, taps - 1, d), 9.0, device="cuda")
    got = []
    for t in range(5):
        x = shifted(torch.stack([rows[0][t], rows[1][t]]), by)
        out = torch.empty(2, 2, d, device="cuda")
        ops.norm_conv_single(x, None, w, b, 1e-5, cw.cuda(), state, out, hand_step([1, 1], [t + 1, t + 1], [2, 0]))
        got.append(out)
    got = torch.stack(got)                                   # [token, set, request, d]
    for r in range(2):
        for s in range(2):
            h = P.layer_norm(rows[r].to(F64), w[s].cpu().to(F64), b[s].cpu().to(F64), 1e-5)
            assert_close(got[:, s, r], P.short_conv(h, cw[s].to(F64)), 1e-5, f"request {r}, set {s}")


@pytest.mark.parametrize("d", [8, 100, 513, 1026, 2044, 2048])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5, 8])
def test_a_token_alone_has_the_bits_of_the_token_in_a_portion(d, taps):
    """32-bit: the fused kernel for single tokens against the norm and the convolution of whole portions, which are kernels of their own."""
    from llama_cu_amd.kernels import ops
    T, planes = 9, 2
    x, delta = rnd(T, d, seed=1) + 2.0, rnd(planes, T, d, seed=2)
    w, b = [rnd(d, seed=k).cuda() for k in (3, 4)], [rnd(d, seed=k).cuda() for k in (5, 6)]
    cw = rnd(2, d, taps, seed=7, std=0.5).cuda()
    h = torch.empty(2, T, d, device="cuda")
    ops.layernorm(x.cuda(), w[0], b[0], 1e-5, h[0], delta=delta.cuda(), weight2=w[1], bias2=b[1], out2=h[1])
    whole_state = torch.full((1, 2, taps - 1, d), 9.0, device="cuda")
    whole = ops.short_conv(h, cw, whole_state, torch.empty_like(h), hand_step([T], [T], [0]))
    for by in (0, 1):                                        # (rows at any address: the bits do not depend on it)
        state = torch.full((1, 2, taps - 1, d), 9.0, device="cuda")
        for t in range(T):
            out = torch.empty(2, 1, d, device="cuda")
            ops.norm_conv_single(shifted(x[t:t + 1], by), delta[:, t:t + 1].contiguous().cuda(), w, b, 1e-5, cw, state, out, hand_step([1], [t + 1], [0]))
            assert torch.equal(out[:, 0], whole[:, t]), f"token {t}, shifted by {by}"
        assert torch.equal(state, whole_state)
