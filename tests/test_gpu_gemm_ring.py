"""Products of packed weights with up to 128 rows whose rows reach LDS by themselves: the bits of the kernel with producer waves, at edges of the ring and of the tiles."""
from __future__ import annotations

import pytest
import torch

from test_gpu_divasun import rnd

pytestmark = pytest.mark.gpu


# fewer macro-steps of K than the ring holds, as many, one more and several turns; features that end within a workgroup; slices of unequal length; with
# 16,512 features more workgroups than compute units (the shorter ring).  The kernel that takes plain weights adds in the same order, so the bits are the same
@pytest.mark.parametrize("m", [1, 17, 32, 33, 48, 49, 64, 65, 96, 97, 127, 128])
@pytest.mark.parametrize("n,k,slices", [(16, 128, 1), (80, 256, 1), (208, 384, 1), (64, 512, 1), (208, 1408, 1), (144, 1408, 3), (80, 1152, 8), (16512, 384, 1), (4160, 640, 5)])
def test_planes_are_those_of_plain_weights(m, n, k, slices):
    from llama_cu_amd.kernels import ops
    wide = rnd(m + 1, k + 16, seed=1).bfloat16()
    wide[m:] = float("nan")
    wide[:, k + 8:] = float("nan")
    wide[:, :8] = float("nan")                             # what lies around the rows counts for nothing
    if m > 20:
        wide[20] = float("nan")                            # and a row of NaN for its own results only
    x, w = wide.cuda()[:m, 8:8 + k], rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda()
    room = torch.full((ops.mid_planes(k, slices), m, n + 4), 7.0, device="cuda")
    got = ops.gemm_mid(x, ops.pack_weight(w), out=room[:, :, :n], slices=slices, packed=True)
    want = ops.gemm_mid(x, w, slices=slices)
    good = torch.arange(m) != 20
    assert torch.equal(got[:, good], want[:, good]) and torch.isfinite(got[:, good]).all() and (room[:, :, n:] == 7).all()
    assert m <= 20 or torch.isnan(got[:, 20]).all()


@pytest.mark.parametrize("m", [32, 33, 48, 49, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("di,k", [(16, 128), (80, 384), (8256, 256), (208, 1408)])
@pytest.mark.parametrize("act", [{}, dict(act_alpha=1.7, act_limit=0.8)])
def test_swiglu_is_that_of_plain_weights(m, di, k, act):
    from llama_cu_amd.kernels import ops
    x, w = rnd(m, k, seed=1).bfloat16().cuda(), rnd(2 * di, k, seed=2, std=k ** -0.5).bfloat16().cuda()
    assert torch.equal(ops.gemm_mid(x, ops.pack_weight(w), swiglu=True, packed=True, **act), ops.gemm_mid(x, w, swiglu=True, **act))


@pytest.mark.parametrize("m,parts", [(17, 1), (33, 48), (49, 100), (64, 256)])
def test_rows_that_wait_for_their_normalisation(m, parts):
    from llama_cu_amd.kernels import ops
    n, k = 208, 1408
    x, w, shares = rnd(m, k, seed=1).bfloat16().cuda(), rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda(), rnd(m, parts, seed=3).abs().cuda()
    kw = dict(slices=4, row_sumsq=shares, norm_width=k, eps=1e-3)
    assert torch.equal(ops.gemm_mid(x, ops.pack_weight(w), packed=True, **kw), ops.gemm_mid(x, w, **kw))


# features that leave the last workgroup of 256 a tile; one round of workgroups, and two; K that leaves none, one and two steps behind the ring's turns
@pytest.mark.parametrize("m", [33, 48, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("n,k", [(49168, 2048), (49152, 2176), (120064, 2304)])
def test_many_features_uncut(m, n, k):
    from llama_cu_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(m, k, device="cuda", generator=g).bfloat16(), (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).bfloat16()
    assert ops.mid_f32_preferred(m, n, k)
    assert torch.equal(ops.gemm_mid(x, ops.pack_weight(w), slices=1, packed=True), ops.gemm_mid(x, w, slices=1))


def test_rows_that_span_more_than_a_load_reaches():
    """65 to 128 rows of 32-bit logits taken out of longer sequences, 4 GiB and more from the first to the last: ``linear`` leaves them to the library, and the kernel refuses
    them.  (A load's place in the rows is 32 bits.)"""
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.linear import Weight, linear
    m, k, n, apart = 100, 2048, 49152, (1 << 31) // 99 + 8 & ~7
    room = torch.empty((m - 1) * apart + k, dtype=torch.bfloat16, device="cuda")
    x = room.as_strided((m, k), (apart, 1))
    x.copy_(rnd(m, k, seed=1))
    w = Weight(rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda())
    assert ops.mid_f32_preferred(m, n, k) and not ops.mid_supported(x, w.plain) and ops.mid_supported(room.as_strided((m, k), (apart - 32, 1)), w.plain)
    want = x.double() @ w.plain.double().T
    assert (linear(x, w, out_dtype=torch.float32) - want).abs().max() < 1e-4
    with pytest.raises(ops.KernelError):
        ops.gemm_mid(x, w.packed, slices=1, packed=True)
