"""The decode kernel's merge of its waves: outputs that cannot be stored four at a time are the same bits as those that can, and both are
the generic kernel's numbers up to rounding, with and without a window (whose first keys lie anywhere)."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,dh", [(4, 4, 32), (16, 4, 128), (20, 1, 64), (34, 2, 96)])
@pytest.mark.parametrize("window,splits", [(0, 1), (0, 3), (50, 1)])
def test_stores(nh, nkv, dh, window, splits):
    from llama_cu_amd.kernels import ops
    ctx, page = [1, 31, 33, 128, 129, 290], 16
    n, most = len(ctx), -(-max(ctx) // page)
    cache = rnd(n * most + 1, 2, nkv * dh * page, seed=1).bfloat16().cuda()
    table = (torch.randperm(n * most, generator=torch.Generator().manual_seed(2)) + 1).to(torch.int32).view(n, most).contiguous().cuda()
    q = rnd(n, nh * dh, seed=3).bfloat16().cuda()
    starts, of, lens = torch.arange(n + 1, dtype=torch.int32).cuda(), torch.arange(n, dtype=torch.int32).cuda(), torch.tensor(ctx, dtype=torch.int32).cuda()
    scale = dh ** -0.5
    even, odd = torch.empty(n, nh * dh, dtype=torch.bfloat16, device="cuda"), torch.zeros(n, nh * dh + 4, dtype=torch.bfloat16, device="cuda")
    wanted = torch.empty_like(even)
    ops.paged_attention_generic(q, wanted, cache, table, starts, lens, of, nh, nkv, dh, page, scale, window)
    ops.attention_decode(q, even, cache, table, starts, lens, n, nh, nkv, dh, page, scale, window, splits)
    assert_close(even, wanted, 3 * 2.0 ** -8, "against the generic kernel")        # the weights and both outputs rounded to bfloat16
    if splits == 1:                                                                # (the kernel that adds parts stores four at a time only)
        ops.attention_decode(q, odd[:, 2:2 + nh * dh], cache, table, starts, lens, n, nh, nkv, dh, page, scale, window, splits)
        assert torch.equal(odd[:, 2:2 + nh * dh], even)
        assert (odd[:, :2] == 0).all() and (odd[:, 2 + nh * dh:] == 0).all()


@pytest.mark.parametrize("nh,nkv,dh", [(15, 1, 128), (16, 1, 128), (17, 1, 32)])
@pytest.mark.parametrize("page", [16, 48, 64])
@pytest.mark.parametrize("splits", [1, 8])
def test_rows_waves_and_pages(nh, nkv, dh, page, splits):
    """Fifteen rows a workgroup are the most that eight waves share, sixteen go to four; pages of 16 tokens and of several times as many; lengths at the
    edges of a step of 32 keys, of a round of the waves and of the parts."""
    from llama_cu_amd.kernels import ops
    ctx = [1, 16, 17, 32, 128, 129, 256, 257, 513]
    n, most = len(ctx), -(-max(ctx) // page)
    cache = rnd(n * most + 1, 2, nkv * dh * page, seed=4).bfloat16().cuda()
    table = (torch.randperm(n * most, generator=torch.Generator().manual_seed(5)) + 1).to(torch.int32).view(n, most).contiguous().cuda()
    q = rnd(n, nh * dh, seed=6).bfloat16().cuda()
    starts, of, lens = torch.arange(n + 1, dtype=torch.int32).cuda(), torch.arange(n, dtype=torch.int32).cuda(), torch.tensor(ctx, dtype=torch.int32).cuda()
    got, wanted = torch.empty(n, nh * dh, dtype=torch.bfloat16, device="cuda"), torch.empty(n, nh * dh, dtype=torch.bfloat16, device="cuda")
    ops.paged_attention_generic(q, wanted, cache, table, starts, lens, of, nh, nkv, dh, page, dh ** -0.5, 0)
    ops.attention_decode(q, got, cache, table, starts, lens, n, nh, nkv, dh, page, dh ** -0.5, 0, splits)
    assert_close(got, wanted, 3 * 2.0 ** -8, "against the generic kernel")        # the weights and both outputs rounded to bfloat16
    ops.attention_decode(q, got.fill_(float("nan")), cache, table, starts, lens, n, nh, nkv, dh, page, dh ** -0.5, 0, splits, few_keys=True)
    assert_close(got, wanted, 3 * 2.0 ** -8, "four waves, however many keys")


@pytest.mark.parametrize("nh,nkv,dh,n,splits", [(4, 4, 64, 80, 1), (2, 2, 128, 30, 4)])
def test_requests_whose_longest_has_many_keys(nh, nkv, dh, n, splits):
    """More workgroups than compute units with eight waves, and parts of heads of 128 with four: what the caller's word for many keys changes is the number of waves."""
    from llama_cu_amd.kernels import build, ops
    units, waves = torch.cuda.get_device_properties(0).multi_processor_count, build.load("attention_mfma").lcu_attention_decode_waves
    if units == 256:
        assert waves(n, nh, nkv, dh, splits, units, 0) != waves(n, nh, nkv, dh, splits, units, 2)
    page, ctx = 16, [1 + (37 * i) % 300 for i in range(n - 1)] + [1100]
    most = -(-max(ctx) // page)
    cache = rnd(n * most + 1, 2, nkv * dh * page, seed=4).bfloat16().cuda()
    table = (torch.randperm(n * most, generator=torch.Generator().manual_seed(5)) + 1).to(torch.int32).view(n, most).contiguous().cuda()
    q = rnd(n, nh * dh, seed=6).bfloat16().cuda()
    starts, of, lens = torch.arange(n + 1, dtype=torch.int32).cuda(), torch.arange(n, dtype=torch.int32).cuda(), torch.tensor(ctx, dtype=torch.int32).cuda()
    got, wanted = torch.empty(n, nh * dh, dtype=torch.bfloat16, device="cuda"), torch.empty(n, nh * dh, dtype=torch.bfloat16, device="cuda")
    ops.paged_attention_generic(q, wanted, cache, table, starts, lens, of, nh, nkv, dh, page, dh ** -0.5, 0)
    for many in (False, True):
        ops.attention_decode(q, got.fill_(float("nan")), cache, table, starts, lens, n, nh, nkv, dh, page, dh ** -0.5, 0, splits, many_keys=many)
        assert_close(got, wanted, 3 * 2.0 ** -8, f"many keys: {many}")        # the weights and both outputs rounded to bfloat16
