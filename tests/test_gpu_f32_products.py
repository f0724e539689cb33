"""What 32-bit products do beside the product: SwiGLU, rows that wait for their normalisation, the residual sum and the next norm's weight;
at the edges of their tiles, against the same in 64 bits, and a row alone against the row among others."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, rnd

pytestmark = pytest.mark.gpu
REL = 3e-6                                               # 32-bit sums of up to 1,408 products and 1,024 squares


@pytest.mark.parametrize("m,n,k", [(1, 16, 4), (2, 1408, 1024), (16, 17, 68), (17, 100, 512), (65, 352, 1408)])
def test_rows_that_wait_and_swiglu(m, n, k):
    from llama_cu_amd.kernels import ops
    x, w, shares = rnd(m, k, seed=1), rnd(2 * n, k, seed=2, std=k ** -0.5), rnd(m, 67, seed=3).abs() + 0.1
    y = x.to(F64) @ w.to(F64).t() * torch.rsqrt(shares.to(F64).sum(1, keepdim=True) / k + 1e-5)
    kw = dict(row_sumsq=shares.cuda(), norm_width=k, eps=1e-5)
    xg, wg = x.cuda(), w.cuda()
    assert_close(ops.gemm_skinny_f32(xg, wg, **kw), y, REL, "scaled")
    g, u = y.split(n, dim=1)
    pair = ops.gemm_skinny_f32(xg, wg, swiglu=True, **kw)
    assert_close(pair, g * torch.sigmoid(g) * u, REL, "swiglu")
    gl, ul = g.clamp(max=0.5), u.clamp(-0.5, 0.5)
    want = gl * torch.sigmoid(1.7 * gl) * (ul + 1)
    # gate and up may each be off by REL times their largest; the derivatives add up to less than 2.5 (0.5 is the largest gate, 1.5 the
    # largest u + 1), but the outputs are clamped to much smaller numbers than gate and up are
    rel = 2.5 * REL * max(1.0, float(y.abs().max() / want.abs().max()))
    assert_close(ops.gemm_skinny_f32(xg, wg, swiglu=True, act_alpha=1.7, act_limit=0.5, **kw), want, rel, "limited")
    for r in {0, m // 2, m - 1}:
        one = dict(kw, row_sumsq=kw["row_sumsq"][r:r + 1].contiguous())
        assert torch.equal(ops.gemm_skinny_f32(xg[r:r + 1], wg, swiglu=True, **one), pair[r:r + 1])


@pytest.mark.parametrize("m,n,k", [(1, 16, 4), (3, 1024, 1408), (16, 17, 68), (17, 100, 512), (70, 1028, 1024)])
def test_residual_and_the_next_norm(m, n, k):
    from llama_cu_amd.kernels import ops
    x, w, res, nw = rnd(m, k, seed=1), rnd(n, k, seed=2, std=k ** -0.5), rnd(m, n + 5, seed=3), rnd(n, seed=4)
    whole = res.cuda()
    xg, wg, ng = x.cuda(), w.cuda(), nw.cuda()
    h, sumsq = ops.gemm_skinny_f32_add_norm(xg, wg, whole[:, 2:2 + n], ng, scale=0.5)
    want = res[:, 2:2 + n].to(F64) + 0.5 * (x.to(F64) @ w.to(F64).t())
    assert_close(whole[:, 2:2 + n], want, REL, "residual")
    assert torch.equal(whole[:, :2].cpu(), res[:, :2]) and torch.equal(whole[:, 2 + n:].cpu(), res[:, 2 + n:])
    assert_close(h, want * nw.to(F64), REL, "rows")
    assert_close(sumsq.sum(1), (want * want).sum(1), REL, "squares")
    for r in {0, m // 2, m - 1}:
        alone = res[r:r + 1, 2:2 + n].contiguous().cuda()
        h1, s1 = ops.gemm_skinny_f32_add_norm(xg[r:r + 1], wg, alone, ng, scale=0.5)
        assert torch.equal(alone, whole[r:r + 1, 2:2 + n]) and torch.equal(h1, h[r:r + 1]) and torch.equal(s1, sumsq[r:r + 1])
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny_f32_add_norm(xg, wg, whole[:, 2:2 + n], ng.bfloat16())
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny_f32_add_norm(xg, wg, whole[:, :n - 1], ng)


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("m", [3, 70])
def test_every_form_of_a_plain_product(m, accumulate, scaled):
    from llama_cu_amd.kernels import ops
    n, k = 1028, 136                                          # (70 rows: 16 a workgroup; 1,000: 64)
    for rows in (m, 1000) if m == 70 else (m,):
        x, w, base, shares = rnd(rows, k, seed=1), rnd(n, k, seed=2, std=k ** -0.5), rnd(rows, n, seed=3), rnd(rows, 5, seed=4).abs()
        out = base.cuda()
        kw = dict(row_sumsq=shares.cuda(), norm_width=k, eps=1e-5) if scaled else {}
        ops.gemm_skinny_f32(x.cuda(), w.cuda(), out=out, accumulate=accumulate, **kw)
        want = x.to(F64) @ w.to(F64).t()
        if scaled:
            want = want * torch.rsqrt(shares.to(F64).sum(1, keepdim=True) / k + 1e-5)
        assert_close(out, want + base.to(F64) if accumulate else want, REL, f"{rows}")
