"""Products whose rows come in by quads of lanes (``quad_rows.h``), at the edges of the loads' and the tiles' row counts.  Operands are small whole numbers,
whose products and sums are whole numbers below 2^24: every result is the exact one or a row or a k is in the wrong place."""
from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def whole(shape, seed, lo=-3, hi=4):
    return torch.randint(lo, hi, shape, generator=torch.Generator().manual_seed(seed)).double()


def rows_of(x, rows_behind=0):
    """``x`` on the GPU as rows of a wider array whose other elements are NaN."""
    wide = torch.full((x.shape[0] + rows_behind, x.shape[1] + 16), float("nan"), dtype=BF16, device="cuda")
    wide[:x.shape[0], 8:8 + x.shape[1]] = x.to(BF16).cuda()
    return wide[:x.shape[0], 8:8 + x.shape[1]]


@pytest.mark.parametrize("m", [1, 3, 4, 5, 7, 8, 9, 15, 16, 17, 24, 31, 32])
def test_few_rows(m):
    from llama_cu_amd.kernels import ops
    for n, k, tiles in ((48, 256, 1), (80, 1408, 2), (64, 640, 4), (16, 6400, 1)):
        x, w = whole((m, k), 1), whole((n, k), 2)
        want, rows, wg = x @ w.t(), rows_of(x, m % 2), w.to(BF16).cuda()
        for waves in (4, 8):
            for weight, packed in ((wg, False), (ops.pack_weight(wg), True)):
                got = ops.gemm_skinny(rows, weight, out_dtype=torch.float32, tiles=tiles, waves=waves, packed=packed)
                assert torch.equal(got.cpu().double(), want), (n, k, tiles, waves, packed)
    x, w = whole((m, 200), 3), whole((40, 200), 4)           # a last macro-step that is not whole, NaN behind it
    assert torch.equal(ops.gemm_skinny(rows_of(x), w.to(BF16).cuda(), out_dtype=torch.float32).cpu().double(), x @ w.t())


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16, 17, 32, 33, 48, 49, 63, 64])
def test_waves_that_share_out_k(m):
    from llama_cu_amd.kernels import ops
    for n, k in ((48, 128), (4112, 256), (80, 1152), (32, 2176), (16, 6400)):
        x, w = whole((m, k), 5), whole((n, k), 6)
        got = ops.gemm_wavek(rows_of(x, m % 2), ops.pack_weight(w.to(BF16).cuda()), out_dtype=torch.float32)
        assert torch.equal(got.cpu().double(), x @ w.t()), (n, k)
    x, w = whole((m, 3 * 128), 7), whole((3 * 16, 128), 8)
    got = ops.gemm_wavek(rows_of(x).unflatten(1, (3, 128)).transpose(0, 1), ops.pack_weight(w.to(BF16).cuda()), out_dtype=torch.float32)
    assert torch.equal(got.cpu().double(), torch.cat([x[:, 128 * g:128 * g + 128] @ w[16 * g:16 * g + 16].t() for g in range(3)], 1))


@pytest.mark.parametrize("m", [2, 5, 16, 33, 48, 49, 64])
@pytest.mark.parametrize("heads,kv_heads,dim,k", [(4, 1, 64, 256), (3, 2, 128, 1152), (2, 2, 32, 128)])
def test_q_k_v_as_the_row_sharing_kernel_makes_them(m, heads, kv_heads, dim, k):
    """Exact sums, so both kernels round, rotate and store the same numbers; positions beyond the table and tokens without a place among them."""
    from llama_cu_amd.kernels import ops
    x = rows_of(whole((m, k), 9))
    w = ops.pack_weight(whole(((heads + 2 * kv_heads) * dim, k), 10).to(BF16).cuda())
    pos = torch.arange(m, dtype=torch.int32) * 3 % 50
    slots = torch.randperm(80, generator=torch.Generator().manual_seed(11))[:m].to(torch.int32)
    pos[m // 2], slots[m - 1] = 70, -1
    ang = torch.arange(64)[:, None] * torch.linspace(0.1, 1.0, dim // 2)[None]
    tables = torch.cos(ang).cuda().contiguous(), torch.sin(ang).cuda().contiguous()
    caches = [torch.zeros(5, 2, kv_heads * dim * 16, dtype=BF16, device="cuda") for _ in range(2)]
    a = ops.gemm_wavek_qkv_rope(x, w, pos.cuda(), slots.cuda(), *tables, caches[0], heads, kv_heads, dim, 16)
    b = ops.gemm_mid_qkv_rope(x, w, pos.cuda(), slots.cuda(), *tables, caches[1], heads, kv_heads, dim, 16, packed=True)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and torch.equal(caches[0].view(torch.int16), caches[1].view(torch.int16))


def test_rows_far_apart():
    from llama_cu_amd.kernels import ops
    x, w = whole((2, 128), 12), whole((32, 128), 13)
    far = torch.empty(2, 1 << 24, dtype=BF16, device="cuda")[:, :128]
    far.copy_(x.to(BF16))
    packed = ops.pack_weight(w.to(BF16).cuda())
    for got in (ops.gemm_skinny(far, packed, out_dtype=torch.float32, packed=True), ops.gemm_wavek(far, packed, out_dtype=torch.float32)):
        assert torch.equal(got.cpu().double(), x @ w.t())


@pytest.mark.parametrize("m", [1, 2, 3])
def test_rows_far_apart_in_every_form(m):
    """One row among them, whose stride says nothing: 2^24 elements and more are no reason to refuse it."""
    from llama_cu_amd.kernels import ops
    x, w = whole((m, 128), 18), whole((192, 128), 19)
    want = x @ w.t()

    def far(dtype):
        rows = torch.empty(m, (1 << 24) + 8, dtype=dtype, device="cuda")[:, :128]
        rows.copy_(x.to(dtype))
        return rows

    xb, xf, wb, wf = far(BF16), far(torch.float32), w.to(BF16).cuda(), w.float().cuda()
    packed = ops.pack_weight(wb)
    same = lambda got: torch.equal(got.double().cpu(), want)
    assert same(ops.gemm_skinny(xb, wb, out_dtype=torch.float32)) and same(ops.gemm_skinny(xb, packed, out_dtype=torch.float32, packed=True))
    assert same(ops.gemm_wavek(xb, packed, out_dtype=torch.float32)) and same(ops.gemm_skinny_f32(xf, wf))
    one = x[:1] @ w[:192].t()                           # two groups of the same row, a view whose groups and rows are all far apart
    pair = xb[:1].unsqueeze(0).expand(2, 1, 128)
    for got in (ops.gemm_wavek(pair, packed, out_dtype=torch.float32),
                ops.gemm_skinny_grouped(pair, packed, torch.empty(1, 192, dtype=torch.float32, device="cuda"), packed=True)):
        assert torch.equal(got.double().cpu(), one)
    for add_norm, rows, weight in ((ops.gemm_skinny_add_norm, xb, wb), (ops.gemm_skinny_f32_add_norm, xf, wf)):
        residual = torch.zeros(m, 192, device="cuda")
        add_norm(rows, weight, residual, torch.ones(192, device="cuda"))
        assert same(residual)
    pos = torch.zeros(m, dtype=torch.int32, device="cuda")
    tables = torch.ones(8, 16, device="cuda"), torch.zeros(8, 16, device="cuda")
    cache = torch.zeros(1, 2, 32 * 16, dtype=BF16, device="cuda")
    for got in (ops.gemm_wavek_qkv_rope(xb, packed, pos, pos - 1, *tables, cache, 4, 1, 32, 16),
                ops.gemm_skinny_qkv_rope(xb, packed, pos, pos - 1, *tables, cache, 4, 1, 32, 16, packed=True)):
        assert torch.equal(got.double().cpu(), want[:, :128].to(BF16).double())


@pytest.mark.parametrize("m", [33, 64])
def test_which_kernel_makes_q_k_v(m, monkeypatch):
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.linear import Weight, linear_qkv_rope
    calls = []
    real = ops.gemm_wavek_qkv_rope
    monkeypatch.setattr(ops, "gemm_wavek_qkv_rope", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    x, z = rows_of(whole((m, 256), 14)), torch.zeros(m, dtype=torch.int32, device="cuda")
    weight = Weight(whole((6 * 64, 256), 15).to(BF16).cuda())
    table, cache = torch.ones(8, 32, device="cuda"), torch.zeros(1, 2, 64 * 16, dtype=BF16, device="cuda")
    got = linear_qkv_rope(x, weight, z, z - 1, table, torch.zeros_like(table), cache, 4, 1, 64, 16)
    assert calls and torch.equal(got.double().cpu(), (x.double().cpu() @ weight.plain[:256].double().cpu().t()).to(BF16).double())


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16, 17, 63, 64, 65, 900])
def test_32_bit_rows(m):
    from llama_cu_amd.kernels import ops
    for n, k in ((16, 64), (72, 1088), (40, 68), (1024, 132), (32, 4160)):
        x, w = whole((m, k), 16), whole((n, k), 17)
        wide = torch.full((m, k + 8), float("nan"), device="cuda")
        wide[:, 4:4 + k] = x.cuda()
        assert torch.equal(ops.gemm_skinny_f32(wide[:, 4:4 + k], w.float().cuda()).cpu().double(), x @ w.t()), (n, k)


@pytest.mark.parametrize("m", [17, 20, 21, 24, 25, 32])
def test_four_tiles_and_a_last_one_of_few_rows(m):
    """The loads of the second sixteen rows: one, two and four, several macro-steps a wave; sums below 2^24, and SwiGLU's bfloat16 rounding of its 32-bit functions."""
    from llama_cu_amd.kernels import ops
    for n, k in ((64, 3200), (128, 5120)):
        x, w = whole((m, k), 20), whole((n, k), 21)
        packed, rows = ops.pack_weight(w.to(BF16).cuda()), rows_of(x, m % 2)
        assert torch.equal(ops.gemm_skinny(rows, packed, out_dtype=torch.float32, tiles=4, waves=8, packed=True).cpu().double(), x @ w.t())
        sums = (x @ w.t()) / 64                              # (a gate that does not saturate: the rows in 64ths)
        want = torch.nn.functional.silu(sums[:, :n // 2]) * sums[:, n // 2:]
        got = ops.gemm_skinny(rows_of(x / 64, m % 2), packed, swiglu=True, tiles=4, waves=8, packed=True).cpu().double()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-30).all()


@pytest.mark.parametrize("m,n,k", [(16, 6144, 4096), (17, 6144, 4096), (9, 4096, 1408), (48, 1152, 2816), (49, 1152, 2816), (63, 1152, 2816), (64, 1152, 2816)])
def test_products_on_both_sides_of_a_line(m, n, k):
    """The kernels and the library's product between which ``linear`` chooses: exact sums, rounded once."""
    from llama_cu_amd.parts.linear import Weight, linear
    x, w = whole((m, k), 22), whole((n, k), 23)
    got = linear(rows_of(x, m % 2), Weight(w.to(BF16).cuda()))
    assert torch.equal(got.double().cpu(), (x @ w.t()).to(BF16).double())


@pytest.mark.parametrize("m", [3, 7, 16, 70])
@pytest.mark.parametrize("k", [4, 272, 512, 1000, 1536, 1796, 2564])
def test_macro_steps_of_a_wave_in_32_bits(m, k):
    """None to six macro-steps of 64 a wave, the last one whole and not; a grid of fewer and of more workgroups than compute units; NaN behind the rows' ends, infinity in the
    matrix' last column.  Whole numbers: the sums are exact."""
    from llama_cu_amd.kernels import ops
    for n in (40, 4112):
        x, w = whole((m, k), 24), whole((n, k), 25)
        wide = torch.full((m, k + 20), float("nan"), device="cuda")
        wide[:, 4:4 + k] = x.float().cuda()
        rows = torch.full((n, k + 20), float("nan"), device="cuda")
        rows[:, 8:8 + k] = w.float().cuda()
        want, add = x @ w.t(), whole((m, n), 26).float().cuda()
        assert torch.equal(ops.gemm_skinny_f32(wide[:, 4:4 + k], rows[:, 8:8 + k]).double().cpu(), want)
        got = ops.gemm_skinny_f32(wide[:, 4:4 + k], rows[:, 8:8 + k], out=add.clone(), accumulate=True)
        assert torch.equal(got.double().cpu(), want + add.double().cpu())
        rows[5, 8 + k - 1] = float("inf")                    # a row of its own: no other feature sees it, and of its sums those whose token is not zero there are infinite
        got = ops.gemm_skinny_f32(wide[:, 4:4 + k], rows[:, 8:8 + k]).double().cpu()
        last = x[:, -1]
        assert torch.equal(got[:, :5], want[:, :5]) and torch.equal(got[:, 6:], want[:, 6:])
        assert torch.equal(torch.isnan(got[:, 5]), last == 0) and torch.equal(got[last != 0, 5], last[last != 0] * math.inf)
