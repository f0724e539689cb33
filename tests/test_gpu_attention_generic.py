"""The attention kernel for every shape, where a request's keys meet the edges of a wave's sixteen and a workgroup's 128, against the
same sums in 64 bits; what the cache holds beyond a request's keys, and table entries that no key needs, are not looked at."""
from __future__ import annotations

import pytest
import torch

from divasun_common import assert_close
from test_gpu_divasun import F64, TYPES, rnd

pytestmark = pytest.mark.gpu


def attend(q, k, v, scale, lo, slope, sink, cap):
    """One query of one head over keys lo .. the last, in 64 bits."""
    s = k @ q * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    s = s + slope * (torch.arange(len(s), dtype=F64) - (len(s) - 1))
    e = torch.exp(s[lo:] - s[lo:].max())
    total = e.sum() + (torch.exp(sink - s[lo:].max()) if sink is not None else 0.0)
    return (e / total) @ v[lo:]


@pytest.mark.parametrize("kind", ["float32", "bfloat16"])
@pytest.mark.parametrize("dh,dv,page,window,chunk,extras", [
    (128, 128, 16, 0, 0, False), (64, 64, 8, 20, 0, False), (8, 1, 8, 0, 48, True), (96, 40, 24, 0, 0, True), (136, 136, 16, 130, 0, False),
    (128, 129, 64, 0, 0, True), (576, 512, 16, 0, 0, False), (640, 640, 8, 1, 0, False)])
def test_edges(kind, dh, dv, page, window, chunk, extras):
    from llama_cu_amd.kernels import ops
    tdt, nh, nkv, scale, cap = TYPES[kind], 4, 2, dh ** -0.5, 20.0 if extras else 0.0
    ctx, fed = [1, 16, 17, 50, 128, 129, 300, 45], [1, 1, 1, 1, 1, 2, 1, 9]
    most = -(-max(ctx) // page)
    pages = sum(-(-c // page) for c in ctx) + 1
    cache = torch.full((pages, 1, nkv * (dh + dv) * page), float("nan"))
    table = torch.zeros(len(ctx), most + 2, dtype=torch.int32)                    # entries that no key needs: page 0, which holds NaN only
    ids = iter((torch.randperm(pages - 1, generator=torch.Generator().manual_seed(3)) + 1).tolist())
    ks, vs = [rnd(c, nkv, dh, seed=r).to(tdt) for r, c in enumerate(ctx)], [rnd(c, nkv, dv, seed=50 + r).to(tdt) for r, c in enumerate(ctx)]
    for r, c in enumerate(ctx):
        seen = 0 if not (window or chunk) else min((c - f - 1) // chunk * chunk if chunk else c - f - window for f in range(fed[r]))
        for first in range(0, c, page):
            if first + page <= seen:
                continue                                                           # passed by: the table still says page 0
            at = table[r, first // page] = next(ids)
            n = min(page, c - first)
            for g in range(nkv):
                keys = cache[at, 0, g * dh * page:(g + 1) * dh * page].view(dh // 8, page, 8)
                keys[:, :n] = ks[r][first:first + n, g].view(n, dh // 8, 8).transpose(0, 1).float()
                cache[at, 0, nkv * dh * page + g * dv * page:][:dv * page].view(dv, page)[:, :n] = vs[r][first:first + n, g].t().float()
    n = sum(fed)
    q = rnd(n, nh * dh + 3, seed=99).to(tdt)[:, 3:]                                # rows at any element
    starts = torch.tensor([0] + fed, dtype=torch.int32).cumsum(0).to(torch.int32)
    of = torch.repeat_interleave(torch.arange(len(ctx)), torch.tensor(fed)).to(torch.int32)
    slopes, sinks = (rnd(nh, seed=7).abs() * 0.1, rnd(nh, seed=8)) if extras else (None, None)
    out = torch.empty(n, nh * dv, dtype=tdt, device="cuda")
    wide = torch.zeros(n, nh * dh + 3, dtype=tdt, device="cuda")
    wide[:, 3:] = q.cuda()
    ops.paged_attention_generic(wide[:, 3:], out, cache.to(tdt).cuda(), table.cuda(), starts.cuda(), torch.tensor(ctx, dtype=torch.int32).cuda(), of.cuda(),
                                nh, nkv, dh, page, scale, window, slopes.cuda() if extras else None, dv, chunk, sinks.cuda() if extras else None, cap)
    want = torch.empty(n, nh, dv, dtype=F64)
    for t in range(n):
        r = int(of[t])
        p = ctx[r] - (int(starts[r + 1]) - t)
        lo = p - p % chunk if chunk else max(0, p - window + 1) if window else 0
        for h in range(nh):
            g = h // (nh // nkv)
            want[t, h] = attend(q[t, h * dh:(h + 1) * dh].to(F64), ks[r][:p + 1, g].to(F64), vs[r][:p + 1, g].to(F64), scale, lo,
                                float(slopes[h]) if extras else 0.0, sinks[h].to(F64) if extras else None, cap)
    assert_close(out, want.view(n, -1), 2e-6 if kind == "float32" else 2.0 ** -8, f"{dh} {dv}")     # 32-bit sums of up to 640 terms; one rounding


@pytest.mark.parametrize("kind,dh,dv", [("float32", 64, 64), ("float32", 128, 96), ("float32", 96, 40), ("bfloat16", 128, 128), ("float32", 256, 200), ("bfloat16", 576, 512)])
@pytest.mark.parametrize("window", [0, 70])
def test_a_token_among_few_and_among_many(kind, dh, dv, window):
    """Single tokens of 1 to 300 keys, so many (token, head) pairs that workgroups have eight, four or two waves: the same bits."""
    from llama_cu_amd.kernels import ops
    tdt, nh, nkv, page, n = TYPES[kind], 8, 2, 16, 280
    ctx = [1 + (37 * r) % 300 for r in range(n)]
    ctx[:8] = [1, 16, 17, 112, 113, 128, 129, 300]
    most = -(-max(ctx) // page)
    table = torch.stack([torch.randperm(64, generator=torch.Generator().manual_seed(r))[:most] for r in range(n)]).to(torch.int32).cuda()
    cache = torch.randn(64, 1, nkv * (dh + dv) * page, generator=torch.Generator().manual_seed(1)).to(tdt).cuda()
    q = rnd(n, nh * dh, seed=2).to(tdt).cuda()
    lengths = torch.tensor(ctx, dtype=torch.int32).cuda()

    def run(first, count):
        out = torch.empty(count, nh * dv, dtype=tdt, device="cuda")
        each = torch.arange(count + 1, dtype=torch.int32, device="cuda")
        return ops.paged_attention_generic(q[first:first + count], out, cache, table[first:first + count].contiguous(), each, lengths[first:first + count].contiguous(),
                                           each[:count].contiguous(), nh, nkv, dh, page, dh ** -0.5, window, None, dv)
    whole = run(0, n)                                        # 2,240 pairs
    for first, count in ((0, 255), (0, 256), (150, 128), (8, 127), (0, 8), (77, 1)):
        assert torch.equal(run(first, count), whole[first:first + count]), (first, count)
    for r in range(8):                                       # ... and the right ones
        pages = table[r].long().cpu()
        keys = cache[pages, 0, :nkv * dh * page].cpu().view(most, nkv, dh // 8, page, 8).permute(1, 0, 3, 2, 4).reshape(nkv, most * page, dh)[:, :ctx[r]].to(F64)
        values = cache[pages, 0, nkv * dh * page:].cpu().view(most, nkv, dv, page).permute(1, 0, 3, 2).reshape(nkv, most * page, dv)[:, :ctx[r]].to(F64)
        want = torch.cat([attend(q[r, h * dh:(h + 1) * dh].cpu().to(F64), keys[h // 4], values[h // 4], dh ** -0.5, max(0, ctx[r] - window) if window else 0, 0.0, None, 0.0)
                          for h in range(nh)])
        assert_close(whole[r], want, 2e-6 if kind == "float32" else 2.0 ** -8, f"{r}")
