"""The product of many rows in tiles, against 64 bits: every shape of tile at edges of tiles, of the rings and of the rows, with each epilogue."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import rnd

pytestmark = pytest.mark.gpu

BF16_REL = 2.0 ** -8            # one rounding of the result, and the largest of the 32-bit sums' errors far below it


# fewer steps of K than a ring holds, as many, and more; one row, a tile less one and more, several tiles; features that end within a tile
@pytest.mark.parametrize("shape", [0, 1, 2])
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (127, 80, 128), (129, 208, 192), (257, 400, 256), (300, 1040, 320), (511, 16, 1088), (33, 2112, 704)])
def test_tiles(shape, m, n, k):
    from llama_cu_amd.kernels import ops
    x, w = rnd(m, k + 24, seed=1).bfloat16().cuda()[:, 8:8 + k], rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda()
    want = x.double() @ w.double().T
    assert_close(ops.gemm_tiles(x, w, shape), want, BF16_REL, "bfloat16")
    assert_close(ops.gemm_tiles(x, w, shape, out_dtype=torch.float32), want, 1e-5, "float32")
    room = torch.full((m + 1, n + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.gemm_tiles(x, w, shape, out=room[:m, :n])
    assert torch.equal(room[:m, :n], ops.gemm_tiles(x, w, shape)) and (room[m:] == 7).all() and (room[:, n:] == 7).all()
    for limit in (0.0, 0.8):
        g, u = want.chunk(2, 1)
        act = g * torch.sigmoid(g) * u
        if limit:
            g, u = torch.clamp(g, max=limit), torch.clamp(u, -limit, limit)
            act = g * torch.sigmoid(1.7 * g) * (u + 1.0)
        got = ops.gemm_tiles(x, w, shape, swiglu=True, **(dict(act_alpha=1.7, act_limit=limit) if limit else {}))
        assert_close(got, act, BF16_REL, f"swiglu, limit {limit}")


def test_rows_and_features_know_nothing_of_each_other():
    """A row of NaN and a feature of infinities reach their own row and column only; rows that hold more than the operands' K, and what lies behind the last row, are not
    looked at."""
    from llama_cu_amd.kernels import ops
    m, n, k = 200, 144, 128
    wide = rnd(m, 2 * k, seed=1).bfloat16()
    wide[:, k:] = float("nan")
    wide[70, :k] = float("nan")
    w = rnd(n, k, seed=2).bfloat16()
    w[9] = float("inf")
    for shape in range(3):
        y = ops.gemm_tiles(wide.cuda()[:, :k], w.cuda(), shape).float().cpu()
        good = torch.ones(m, n, dtype=torch.bool)
        good[70] = False
        good[:, 9] = False
        assert torch.isfinite(y[good]).all() and torch.isnan(y[70]).all() and not torch.isfinite(y[:, 9]).any()


@pytest.mark.parametrize("m,n,k", [(2014, 2560, 2048), (1100, 2048, 2048), (2014, 5632, 2048)])
def test_the_products_that_the_rule_names(m, n, k):
    """What ``linear`` computes where ``tiles_choice`` names a shape, and the choice itself at its edges."""
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.linear import linear
    swiglu = n == 5632
    shape = ops.tiles_choice(m, n, k, swiglu)
    assert shape >= 0 and ops.tiles_choice(ops.TUNING.tiles_rows, n, k, swiglu) == -1 and ops.tiles_choice(m, n, k + 8, swiglu) == -1
    x, w = rnd(m, k, seed=1).bfloat16().cuda(), rnd(n, k, seed=2, std=k ** -0.5).bfloat16().cuda()
    if swiglu:
        g, u = (x.double() @ w.double().T).chunk(2, 1)
        assert_close(ops.gemm_tiles(x, w, shape, swiglu=True), g * torch.sigmoid(g) * u, BF16_REL, "swiglu")
        return
    assert torch.equal(linear(x, w), ops.gemm_tiles(x, w, shape))
    assert_close(linear(x, w), x.double() @ w.double().T, BF16_REL, "linear")


def test_what_is_refused():
    from llama_cu_amd.kernels import ops
    x, w = rnd(40, 128, seed=1).bfloat16().cuda(), rnd(64, 128, seed=2).bfloat16().cuda()
    for bad in (lambda: ops.gemm_tiles(x, w, 3), lambda: ops.gemm_tiles(x.float(), w, 0), lambda: ops.gemm_tiles(x[:, :96], w[:, :96].contiguous(), 0),
                lambda: ops.gemm_tiles(x, w[:40], 0), lambda: ops.gemm_tiles(x[:, 1:65], w[:, :64].contiguous(), 0),
                lambda: ops.gemm_tiles(x, w, 0, out=torch.empty(40, 66, dtype=torch.bfloat16, device="cuda")[:, 1:65])):
        with pytest.raises(ops.KernelError):
            bad()


@pytest.mark.parametrize("m,n,k,shape", [(576, 4096, 4096, 0), (577, 4096, 4096, -1), (768, 4096, 4096, -1), (769, 4096, 4096, 0), (768, 4096, 4032, 0), (480, 5120, 4096, 0), (576, 5120, 4096, -1), (577, 5120, 4096, 0)])
def test_where_finer_tiles_fill_a_round(m, n, k, shape):
    """On a card of 256 compute units; on both sides of the lines between which the library's finer tiles are taken."""
    from llama_cu_amd.kernels import ops
    if ops.TUNING.compute_units != 256:
        pytest.skip("the lines are those of 256 compute units")
    assert ops.tiles_choice(m, n, k) == shape


def test_operands_on_other_devices_are_refused():
    """A weight, or an output, in host memory: the library's error from ``linear``, the kernel's own from ``gemm_tiles``, and no launch."""
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.linear import linear, tiles_swiglu_shape
    x, w = rnd(1100, 2048, seed=1).bfloat16().cuda(), rnd(2048, 2048, seed=2).bfloat16().cuda()
    assert ops.tiles_choice(1100, 2048, 2048) >= 0 and tiles_swiglu_shape(x, w) >= 0 and tiles_swiglu_shape(x, w.cpu()) == -1
    out = torch.empty(1100, 2048, dtype=torch.bfloat16)
    for bad in (lambda: linear(x, w.cpu()), lambda: linear(x, w, out=out), lambda: linear(x, w.cpu(), out_dtype=torch.float32)):
        with pytest.raises(RuntimeError):
            bad()
    for known in (False, True):
        for bad in (lambda: ops.gemm_tiles(x, w.cpu(), 0, known=known), lambda: ops.gemm_tiles(x, w, 0, out=out, known=known)):
            with pytest.raises(ops.KernelError):
                bad()


def test_rows_of_no_width():
    from llama_cu_amd.parts.linear import linear
    x, w = torch.empty(1100, 0, dtype=torch.bfloat16, device="cuda"), torch.empty(2048, 0, dtype=torch.bfloat16, device="cuda")
    for dtype in (torch.bfloat16, torch.float32):
        y = linear(x, w, out_dtype=dtype)
        assert y.shape == (1100, 2048) and y.dtype == dtype and (y == 0).all()


def test_an_output_of_another_shape():
    """The library makes it fit, with a warning; the kernel in tiles would refuse it."""
    from llama_cu_amd.parts.linear import linear
    x, w = rnd(1100, 128, seed=1).bfloat16().cuda(), rnd(2048, 128, seed=2).bfloat16().cuda()
    for shape in ((1100, 2056), (1104, 2048)):
        out = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
        with pytest.warns(UserWarning, match="resized"):
            assert linear(x, w, out=out) is out
        assert out.shape == (1100, 2048)
        assert_close(out, x.double() @ w.double().T, BF16_REL, "resized")


def test_a_product_that_is_differentiated():
    """Where a gradient is asked for, ``linear`` of many bfloat16 rows stays the library's, which has one."""
    from llama_cu_amd.parts.linear import linear
    x, w = rnd(1100, 128, seed=1).bfloat16().cuda(), rnd(2048, 128, seed=2).bfloat16().cuda()
    g = rnd(1100, 2048, seed=3).bfloat16().cuda()
    grads = torch.autograd.grad(linear(x.requires_grad_(), w.requires_grad_()), (x, w), g)
    assert_close(grads[0], g.double() @ w.double(), BF16_REL, "x")
    assert_close(grads[1], g.double().T @ x.double(), BF16_REL, "w")
    with torch.no_grad():
        assert not linear(x, w).requires_grad
