"""The norm over whole projections on its way into the pages, four columns at a time and one (rows that are not aligned for four), below, at and
beyond what a workgroup keeps in registers."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, TYPES, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["float32", "bfloat16"])
@pytest.mark.parametrize("nh,nkv,dh,dv,page,by", [(1, 1, 8, 1, 8, 0), (16, 4, 128, 128, 16, 0), (16, 4, 128, 128, 16, 1), (33, 33, 128, 7, 24, 0),
                                                  (9, 3, 120, 36, 8, 4)])
def test_norm_factor_and_store(nh, nkv, dh, dv, page, by, kind):
    from llama_cu_amd.kernels import ops
    tdt, n, eps, coef, every = TYPES[kind], 5, 1e-5, 0.25, 3
    nq, nk, nv = nh * dh, nkv * dh, nkv * dv
    rows = rnd(n, nq + nk + nv, seed=1).to(tdt)
    wide = torch.zeros(n, nq + nk + nv + by + (-(nq + nk + nv + by)) % 4, dtype=tdt, device="cuda")
    qkv = wide[:, by:by + nq + nk + nv]
    qkv.copy_(rows)
    qw, kw = rnd(nq, seed=2), rnd(nk, seed=3)
    cache = torch.zeros(3, 1, nkv * (dh + dv) * page, dtype=tdt, device="cuda")
    slots = torch.tensor([0, 2 * page + 1, page + page - 1, -1, page], dtype=torch.int32).cuda()          # (one row is stored nowhere)
    positions = torch.tensor([0, 5, 2, 900, 7], dtype=torch.int32).cuda()
    ops.qk_norm_store(qkv, positions, nh, nkv, dh, dv, qw.cuda(), kw.cuda(), eps, coef, every, cache, slots, page)
    x = rows.to(F64)
    q, k = x[:, :nq], x[:, nq:nq + nk]
    factor = 1 + coef * torch.log(torch.floor((positions.cpu().to(F64) + 1) / every) + 1)
    rel = 1e-5 if kind == "float32" else 2.0 ** -8 + 1e-5                          # 32-bit sums; half a unit of bfloat16's last place
    assert_close(qkv[:, :nq], q * torch.rsqrt((q * q).mean(1, keepdim=True) + eps) * qw.to(F64) * factor[:, None], rel, "queries")
    assert torch.equal(qkv[:, nq:].cpu(), rows[:, nq:])
    keys = k * torch.rsqrt((k * k).mean(1, keepdim=True) + eps) * kw.to(F64)
    held = torch.zeros(3, page, dtype=torch.bool)
    ks = cache[:, 0, :nk * page].view(3, nkv, dh // 8, page, 8).permute(0, 3, 1, 2, 4).reshape(3, page, nk).cpu()
    vs = cache[:, 0, nk * page:].view(3, nv, page).transpose(1, 2).cpu()
    for t in (0, 1, 2, 4):
        at, tok = divmod(int(slots[t]), page)
        held[at, tok] = True
        assert_close(ks[at, tok], keys[t], rel, f"keys of row {t}")
        assert torch.equal(vs[at, tok], rows[t, nq + nk:])
    assert (ks[~held] == 0).all() and (vs[~held] == 0).all()


@pytest.mark.parametrize("kind", ["float32", "bfloat16"])
@pytest.mark.parametrize("nh,nkv,dh,dv", [(1, 1, 8, 3), (16, 4, 128, 128), (33, 5, 120, 20), (80, 40, 128, 8)])
def test_a_rows_bits_do_not_depend_on_the_number_of_rows(nh, nkv, dh, dv, kind):
    """On both sides of the line between a workgroup a part and one for all three; one to forty stretches of a sum."""
    from llama_cu_amd.kernels import ops
    tdt, page, n = TYPES[kind], 16, 300
    qkv = rnd(n, nh * dh + nkv * (dh + dv), seed=1).to(tdt).cuda()
    qw, kw = rnd(nh * dh, seed=2).cuda(), rnd(nkv * dh, seed=3).cuda()
    positions, slots = torch.arange(n, dtype=torch.int32).cuda(), torch.randperm(n, generator=torch.Generator().manual_seed(4)).to(torch.int32).cuda()
    outs = []
    for cut in (n, 128, 7):
        rows, cache = qkv.clone(), torch.zeros(-(-n // page), 1, nkv * (dh + dv) * page, dtype=tdt, device="cuda")
        for a in range(0, n, cut):
            b = min(n, a + cut)
            ops.qk_norm_store(rows[a:b], positions[a:b].contiguous(), nh, nkv, dh, dv, qw, kw, 1e-5, 0.3, 5, cache, slots[a:b].contiguous(), page)
        outs.append((rows, cache))
    for rows, cache in outs[1:]:
        assert torch.equal(rows, outs[0][0]) and torch.equal(cache, outs[0][1])
