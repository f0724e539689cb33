"""The product whose waves share out K, at the edges of its tiles and of its rule, against the product in 64 bits."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, rnd

pytestmark = pytest.mark.gpu
BF16_REL = 2.0 ** -8                                     # half a unit of bfloat16's last place is 2^-9 of a value; room for the sums' order


def operands(m, n, k, seed=1):
    return rnd(m, k, seed=seed).bfloat16().cuda(), (rnd(n, k, seed=seed + 1, std=k ** -0.5)).bfloat16().cuda()


def f64(t):
    return t.cpu().to(F64)


@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (3, 48, 256), (16, 4096, 384), (17, 4112, 1152), (32, 2048, 2816), (33, 32, 128), (48, 4128, 2048),
                                   (49, 80, 1024), (64, 4096, 2176)])
def test_product(m, n, k):
    from llama_cu_amd.kernels import ops
    x, w = operands(m, n, k)
    packed, want = ops.pack_weight(w), f64(x) @ f64(w).t()
    wide = torch.zeros(m, k + 24, dtype=torch.bfloat16, device="cuda")
    wide[:, 8:8 + k] = x                                 # rows of a wider array
    assert_close(ops.gemm_wavek(wide[:, 8:8 + k], packed), want, BF16_REL, "bfloat16")
    room = torch.full((m, n + 8), 7.0, device="cuda")
    ops.gemm_wavek(x, packed, out=room[:, :n])
    assert_close(room[:, :n], want, 1e-5, "float32")     # k products of 16-bit numbers in 32-bit sums
    assert (room[:, n:] == 7.0).all()
    gate = rnd(m, n, seed=5).bfloat16().cuda()
    assert_close(ops.gemm_wavek(x, packed, gate=gate), want * torch.sigmoid(f64(gate)), BF16_REL, "gated")
    shares = rnd(m, 3, seed=6).abs().cuda()
    factor = torch.rsqrt(f64(shares).sum(1, keepdim=True) / k + 1e-5)
    assert_close(ops.gemm_wavek(x, packed, out_dtype=torch.float32, row_sumsq=shares, norm_width=k, eps=1e-5), want * factor, 1e-5, "scaled rows")


@pytest.mark.parametrize("limit", [0.0, 0.5])
@pytest.mark.parametrize("m,n,k", [(1, 32, 128), (16, 96, 2048), (31, 352, 640), (64, 5632, 1024)])
def test_swiglu(m, n, k, limit):
    from llama_cu_amd.kernels import ops
    x, w = operands(m, n, k, seed=11)
    g, u = (f64(x) @ f64(w).t()).split(n // 2, dim=1)
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        want = g * torch.sigmoid(1.7 * g) * (u + 1)
    else:
        want = g * torch.sigmoid(g) * u
    got = ops.gemm_wavek(x, ops.pack_weight(w), swiglu=True, **(dict(act_alpha=1.7, act_limit=limit) if limit else {}))
    assert_close(got, want, BF16_REL, f"{m} x {n} x {k}")


@pytest.mark.parametrize("m", [8, 64])
def test_stores_round_to_the_nearest(m):
    """What is stored in 16 bits is off by half a unit of the last place at most, evenly on both sides: a root mean square of 1 / sqrt(12) of a unit
    (cut off it would be 1 / sqrt(3)) and a mean of nothing.  The bounds above, of the largest value, would let a cut pass."""
    from llama_cu_amd.kernels import ops
    n, k = 4096, 512
    x, w = operands(m, n, k, seed=51)
    packed, product, gate = ops.pack_weight(w), f64(x) @ f64(w).t(), rnd(m, n, seed=53).bfloat16().cuda()
    g, u = product.split(n // 2, dim=1)
    for what, got, want in (("plain", ops.gemm_wavek(x, packed), product), ("gated", ops.gemm_wavek(x, packed, gate=gate), product * torch.sigmoid(f64(gate))),
                            ("swiglu", ops.gemm_wavek(x, packed, swiglu=True), g * torch.sigmoid(g) * u)):
        # (values of which a 32-bit sum's error, some 1e-7 of the largest, is no part of a unit)
        big = want.abs() > 0.01 * want.abs().mean()
        want, got = want[big], f64(got)[big]
        off = (got - want) * torch.sign(want) / torch.exp2(torch.floor(torch.log2(want.abs())) - 7)
        assert off.square().mean().sqrt() < 1.02 * 12 ** -0.5, what
        assert off.mean().abs() < 6 * (12 * off.numel()) ** -0.5 + 1e-3, what      # six deviations of the mean


@pytest.mark.parametrize("m,n,k,groups", [(2, 16, 128, 3), (33, 2048, 256, 4), (64, 112, 384, 2)])
def test_groups(m, n, k, groups):
    from llama_cu_amd.kernels import ops
    w = rnd(groups * n, k, seed=21, std=k ** -0.5).bfloat16().cuda()
    rows = rnd(m, groups * k, seed=22).bfloat16().cuda()          # a token's groups side by side
    got = ops.gemm_wavek(rows.view(m, groups, k).transpose(0, 1), ops.pack_weight(w))
    want = torch.cat([f64(rows)[:, g * k:(g + 1) * k] @ f64(w)[g * n:(g + 1) * n].t() for g in range(groups)], dim=1)
    assert_close(got, want, BF16_REL, "groups")


@pytest.mark.parametrize("m", [4, 5, 32, 33, 48, 49, 64, 65])
@pytest.mark.parametrize("n,k", [(1024, 1024), (2048, 2048), (3072, 2048), (8192, 512), (8224, 512), (496, 512), (512, 384)])
def test_the_rule_against_the_general_path(m, n, k):
    """A product on both sides of the rule's lines, the rows as they are and where they cannot be loaded 16 bytes at a time."""
    from llama_cu_amd.parts.linear import Weight, linear
    x, w = operands(m, n, k, seed=31)
    weight = Weight(w)
    want = f64(x) @ f64(w).t()
    odd = torch.zeros(m, k + 1, dtype=torch.bfloat16, device="cuda")
    odd[:, 1:] = x
    for rows in (x, odd[:, 1:], x.t().contiguous().t()):
        assert_close(linear(rows, weight, out_dtype=torch.bfloat16), want, BF16_REL, f"{rows.stride()}")
        if rows.stride(1) == 1:
            assert_close(linear(rows, weight, out_dtype=torch.float32), want, 1e-5, f"{rows.stride()}, float32")


def test_what_it_refuses():
    from llama_cu_amd.kernels import ops
    x, w = operands(4, 64, 256, seed=41)
    packed = ops.pack_weight(w)
    for bad in (lambda: ops.gemm_wavek(rnd(65, 256, seed=1).bfloat16().cuda(), packed), lambda: ops.gemm_wavek(x[:, :128], packed),
                lambda: ops.gemm_wavek(x, packed, out=torch.empty(4, 62, device="cuda")),
                lambda: ops.gemm_wavek(x, packed, swiglu=True, out_dtype=torch.float32),
                lambda: ops.gemm_wavek(x, packed, gate=torch.empty(4, 32, dtype=torch.bfloat16, device="cuda")),
                lambda: ops.gemm_wavek(x, packed, row_sumsq=torch.ones(3, 1, device="cuda"), norm_width=256)):
        with pytest.raises(ops.KernelError):
            bad()


@pytest.mark.parametrize("m", [24, 25, 32, 33, 48, 49, 64, 65])
@pytest.mark.parametrize("ff,k", [(512, 1024), (512, 2048), (1408, 2048), (2816, 2048), (512, 3072), (2816, 3072), (2832, 3072)])
def test_the_rule_of_swiglu_against_the_general_path(m, ff, k):
    """A feed-forward on both sides of the rule's lines, against 64 bits."""
    from llama_cu_amd.parts.base import BuildContext, PartSpec, make_part
    part = make_part("ffn", PartSpec("swiglu", {"hidden_size": k, "intermediate_size": ff}))
    w = {n: rnd(*s.shape, seed=60 + i, std=s.shape[-1] ** -0.5).bfloat16() for i, (n, s) in enumerate(sorted(part.tensors().items()))}
    part.load({n: t.cuda() for n, t in w.items()}, BuildContext(torch.bfloat16, torch.device("cuda"), 64, 16, pack_weights=True))
    x = rnd(m, k, seed=70).bfloat16().cuda()
    gate, up, down = (next(f64(t) for n, t in w.items() if what in n) for what in ("gate", "up", "down"))
    g, u = f64(x) @ gate.t(), f64(x) @ up.t()
    # up to four roundings, of gate, up, activation and output, each 2^-9 of a value at most; an activation's slope is below 1.1
    assert_close(part.forward(x), (g * torch.sigmoid(g) * u) @ down.t(), 2.0 ** -6, f"{m} x {ff} x {k}")
