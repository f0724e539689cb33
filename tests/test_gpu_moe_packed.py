"""Experts' matrices in the kernels' own order (``ops.pack_experts``) against the matrices as they are, and the kernel for few rows
an expert at the edges of its lists, tiles and quarters of K."""
from __future__ import annotations

import pytest
import torch

import plain_divasun as P
from divasun_common import assert_close
from test_gpu_divasun import F64, TYPES, rnd

pytestmark = pytest.mark.gpu


# one pair; an expert with 17 rows (two tiles) and K of less than a step; K that ends within a step, and rows that end within a tile;
# more pairs than a list holds; the kernel for many rows; every quarter of K of another length
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("experts,top,d,ff,n", [(4, 1, 72, 24, 1), (2, 1, 16, 8, 31), (5, 2, 200, 88, 33), (160, 8, 72, 16, 300), (4, 2, 264, 136, 300),
                                                (8, 3, 1032, 40, 40)])
def test_packed_experts(dtype, experts, top, d, ff, n):
    from llama_cu_amd.kernels import ops
    tdt = TYPES[dtype]
    h, router = rnd(n, d, seed=1).to(tdt).cuda(), rnd(experts, d, seed=2, std=0.5).cuda()
    up, down = rnd(experts, ff, d, seed=3, std=d ** -0.5).to(tdt).cuda(), rnd(experts, d, ff, seed=4, std=ff ** -0.5).to(tdt).cuda()
    base = rnd(n, d, seed=5)
    ids, wts = ops.moe_route(h, router, top)
    outs = []
    for u, w in ((up, down), (ops.pack_experts(up), ops.pack_experts(down)), (up, ops.pack_experts(down))):
        out = base.clone().cuda()
        ops.moe_experts(h, ids, wts, u, w, out)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    plain = {"router": router.cpu().to(F64)}
    for e in range(experts):
        plain[f"e{e}.up"], plain[f"e{e}.down"] = up[e].cpu().to(F64), down[e].cpu().to(F64)
    want = base.to(F64) + P.moe(h.cpu().to(F64), plain, experts, top)
    assert_close(outs[0], want, 1e-4 if dtype == "float32" else 3e-2, "output")      # (the bounds of the unpacked experts' test)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,ff", [(1, 16), (20, 48), (200, 112)])
def test_packed_gated_experts(dtype, n, ff):
    from llama_cu_amd.kernels import ops
    experts, top, d, tdt = 6, 2, 104, TYPES[dtype]
    h, router = rnd(n, d, seed=1).to(tdt).cuda(), rnd(experts + 1, d, seed=2).cuda()
    gate, up = (rnd(experts, ff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (3, 4))
    down = rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda()
    ids, wts = ops.moe_route(h, router, top, softmax_chosen=True)        # (the last of the router's rows is an identity expert)
    rows, outs = ops.gated_rows(gate, up), []
    assert torch.equal(ops.pack_gated_experts(gate, up).data, ops.pack_experts(rows).data)
    for u, w in ((rows, down), (ops.pack_experts(rows), ops.pack_experts(down))):
        out = torch.empty(n, d, device="cuda")
        ops.moe_experts(h, ids, wts, u, w, out, gated=True, fresh=True, identity=1, act_alpha=1.702, act_limit=2.0)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    x, want = h.cpu().to(F64), torch.zeros(n, d, dtype=F64)
    for t in range(n):
        for e, w in zip(ids[t].tolist(), wts[t].cpu().to(F64)):
            if e == experts:
                want[t] += w * x[t]
                continue
            g = torch.clamp(gate[e].cpu().to(F64) @ x[t], max=2.0)
            v = torch.clamp(up[e].cpu().to(F64) @ x[t], -2.0, 2.0)
            want[t] += w * (down[e].cpu().to(F64) @ (g * torch.sigmoid(1.702 * g) * (v + 1.0)))
    assert_close(outs[0], want, 1e-4 if dtype == "float32" else 3e-2, "output")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,ff,sff,gate", [(1, 16, 48, True), (17, 112, 16, False), (32, 32, 208, True)])
def test_a_shared_expert_beside_the_others(dtype, n, ff, sff, gate):
    """The shared expert smaller and larger than the others, at one and two tiles of rows, against the sum in 64 bits."""
    from llama_cu_amd.kernels import ops
    experts, top, d, tdt = 5, 2, 88, TYPES[dtype]
    pack = ops.pack_experts
    h, router = rnd(n, d, seed=1).to(tdt).cuda(), rnd(experts + 1, d, seed=2).cuda()
    gates, ups = (rnd(experts, ff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (3, 4))
    down = rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda()
    sg, su = (rnd(1, sff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (6, 7))
    sd = rnd(1, d, sff, seed=8, std=sff ** -0.5).to(tdt).cuda()
    up_p, down_p = pack(ops.gated_rows(gates, ups)), pack(down)
    assert ops.moe_shared_beside(n, top, experts, up_p, down_p) == (n * top <= 16 * experts)
    ids, wts, g = ops.moe_route(h, router, top, softmax_chosen=True, extra=1)
    out = torch.full((n, d), 3.0, device="cuda")
    ops.moe_experts(h, ids, wts, up_p, down_p, out, gated=True, shared_expert=(pack(ops.gated_rows(sg, su)), pack(sd)),
                    shared_gate=g if gate else None, act_alpha=1.702, act_limit=2.0)
    x, want = h.cpu().to(F64), torch.full((n, d), 3.0, dtype=F64)
    f = lambda t: t.cpu().to(F64)
    z = f(sg[0]) @ x.T
    shared = (f(sd[0]) @ (z * torch.sigmoid(z) * (f(su[0]) @ x.T))).T
    want += shared * (torch.sigmoid(x @ f(router[experts]))[:, None] if gate else 1.0)
    for t in range(n):
        for e, w in zip(ids[t].tolist(), f(wts[t])):
            a, b = torch.clamp(f(gates[e]) @ x[t], max=2.0), torch.clamp(f(ups[e]) @ x[t], -2.0, 2.0)
            want[t] += w * (f(down[e]) @ (a * torch.sigmoid(1.702 * a) * (b + 1.0)))
    assert_close(out, want, 1e-4 if dtype == "float32" else 3e-2, "output")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("experts,top,n,all_of", [(16, 1, 64, 49), (16, 1, 65, 65), (16, 1, 128, 97), (17, 1, 129, 129), (70, 4, 200, 33), (1024, 3, 100, 100)])
def test_an_expert_that_many_tokens_name(dtype, experts, top, n, all_of):
    """Experts of few rows on average, one of which ``all_of`` of the tokens name: on both sides of the number of pairs from which on they come
    sorted, in tiles; every row has the bits that it has alone."""
    from llama_cu_amd.kernels import ops
    d, ff, tdt = 72, 32, TYPES[dtype]
    h = rnd(n, d, seed=1).to(tdt).cuda()
    up, down = rnd(experts, 2 * ff, d, seed=2, std=d ** -0.5).to(tdt).cuda(), rnd(experts, d, ff, seed=3, std=ff ** -0.5).to(tdt).cuda()
    g = torch.Generator().manual_seed(4)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(n)])
    for t in range(all_of):
        if not (ids[t] == experts - 1).any():
            ids[t, t % top] = experts - 1
    ids, wts = ids.to(torch.int32).cuda(), torch.rand(n, top, generator=g).cuda()
    packed = ops.pack_experts(up), ops.pack_experts(down)
    outs = []
    for u, w in ((up, down), packed):
        out = torch.empty(n, d, device="cuda")
        ops.moe_experts(h, ids, wts, u, w, out, gated=True, fresh=True)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    for t in range(0, n, 7):
        one = torch.empty(1, d, device="cuda")
        ops.moe_experts(h[t:t + 1], ids[t:t + 1].contiguous(), wts[t:t + 1].contiguous(), *packed, one, gated=True, fresh=True)
        assert torch.equal(one[0], outs[1][t]), f"token {t}"
    x, want = h.cpu().to(F64), torch.zeros(n, d, dtype=F64)
    u, w = up.cpu().to(F64).view(experts, ff // 16, 2, 16, d), down.cpu().to(F64)
    for t in range(n):
        for e, weight in zip(ids[t].tolist(), wts[t].cpu().to(F64)):
            a, b = (u[e, :, k].reshape(ff, d) @ x[t] for k in (0, 1))
            want[t] += weight * (w[e] @ (a * torch.sigmoid(a) * b))
    assert_close(outs[0], want, 1e-5 if dtype == "float32" else 2.0 ** -8, "output")      # (one rounding to bfloat16, of the activations, under sums over ff)


def test_a_shared_expert_beside_sorted_pairs():
    """32 tokens of nine experts each: the pairs come in tiles, the shared expert rides along all the same."""
    from llama_cu_amd.kernels import ops
    experts, top, n, d, ff, sff = 40, 9, 32, 64, 16, 48
    h = rnd(n, d, seed=1).cuda()
    up, down = rnd(experts, 2 * ff, d, seed=2, std=d ** -0.5).cuda(), rnd(experts, d, ff, seed=3, std=ff ** -0.5).cuda()
    sg, su, sd = rnd(1, sff, d, seed=4, std=d ** -0.5).cuda(), rnd(1, sff, d, seed=5, std=d ** -0.5).cuda(), rnd(1, d, sff, seed=6, std=sff ** -0.5).cuda()
    g = torch.Generator().manual_seed(7)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(n)]).to(torch.int32).cuda()
    wts = torch.rand(n, top, generator=g).cuda()
    packed = ops.pack_experts(up), ops.pack_experts(down)
    assert ops.moe_shared_beside(n, top, experts, *packed)
    both, alone = torch.empty(n, d, device="cuda"), torch.empty(n, d, device="cuda")
    ops.moe_experts(h, ids, wts, *packed, both, gated=True, fresh=True, shared_expert=(ops.pack_gated_experts(sg, su), ops.pack_experts(sd)))
    ops.moe_experts(h, ids, wts, *packed, alone, gated=True, fresh=True)
    z = h.cpu().to(F64) @ sg[0].cpu().to(F64).T
    want = alone.cpu().to(F64) + (z * torch.sigmoid(z) * (h.cpu().to(F64) @ su[0].cpu().to(F64).T)) @ sd[0].cpu().to(F64).T
    assert_close(both, want, 1e-5, "output")


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_token_with_few_and_with_more_others(dtype, gated):
    """A mixture with a shared expert whose matrices are packed, on both sides of the number of tokens up to which the shared expert is computed
    beside the others: in 32 bits a token has the same bits, in bfloat16 the two are one rounding of the shared row and one of its
    activations apart."""
    from llama_cu_amd.kernels import ops
    from llama_cu_amd.parts.base import BuildContext
    from llama_cu_amd.parts.moe import GatedMoE
    d, ff, sff, experts, top, tdt = 520, 48, 528, 12, 2, TYPES[dtype]      # (K beyond 256: the two paths cut their sums at other places)
    part = GatedMoE(d, ff, experts, top, shared_size=sff, shared_gated=gated)
    tensors = {n: rnd(*t.shape, seed=k, std=t.shape[-1] ** -0.5).to(tdt).cuda() for k, (n, t) in enumerate(part.tensors().items())}
    part.load(tensors, BuildContext(tdt, torch.device("cuda"), 64, 16, pack_weights=True))
    h, few = rnd(3 * ops.MOE_SHARED_ROWS, d, seed=99).to(tdt).cuda(), ops.MOE_SHARED_ROWS
    whole = part.forward(h)
    for n in (1, few - 1, few, few + 1):
        for first in (0, h.shape[0] - n):
            got = part.forward(h[first:first + n].contiguous())
            if dtype == "float32":
                assert torch.equal(got, whole[first:first + n]), n
            else:
                # a rounding is at most 2^-9 of a value: one of sff activations under weights of sff ** -0.5 each (2^-9 of the largest together, and
                # the other path's as much), one of the shared row
                assert_close(got, whole[first:first + n].cpu().to(F64), 3 * 2.0 ** -9, f"{n}")


# an expert's tiles at their edges (of 32 to 128 rows, by the sizes), beside experts with few rows and with none;
# K of less than a step, of whole steps, and one that ends within a unit of the last; features that end within a block, fewer blocks than dies
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("counts,d,ff", [((17, 96, 97, 0, 33, 193), 264, 48), ((128, 129, 81, 95, 0, 100), 1096, 272), ((1, 600, 31, 65), 40, 1040),
                                         ((32, 64, 127, 96, 1, 288), 64, 16)])
@pytest.mark.parametrize("gated,pack", [(True, True), (True, False), (False, True), (False, False)])
def test_tiles_of_many_rows(dtype, counts, d, ff, gated, pack):
    from llama_cu_amd.kernels import ops
    experts, n, tdt = len(counts), sum(counts), TYPES[dtype]
    order = torch.randperm(n, generator=torch.Generator().manual_seed(0))
    ids = torch.repeat_interleave(torch.arange(experts, dtype=torch.int32), torch.tensor(counts))[order].view(n, 1).cuda()
    h, wts = rnd(n, d, seed=1).to(tdt).cuda(), torch.rand(n, 1, generator=torch.Generator().manual_seed(2)).cuda()
    gate, up = (rnd(experts, ff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (3, 4))
    down = rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda()
    u, w = ops.gated_rows(gate, up) if gated else up, down
    if pack:
        u, w = ops.pack_experts(u), ops.pack_experts(w)

    def run(part):
        out = torch.zeros(part.stop - part.start, d, device="cuda")
        return ops.moe_experts(h[part].contiguous(), ids[part].contiguous(), wts[part].contiguous(), u, w, out, **({"gated": True, "fresh": True} if gated else {}))
    got = run(slice(0, n))
    few = 16 * experts                     # steps of so few take the kernel for few rows: a token has the same bits
    assert torch.equal(got, torch.cat([run(slice(a, min(n, a + few))) for a in range(0, n, few)]))
    e, x, s = ids[:, 0].long().cpu(), h.cpu().to(F64), wts.cpu().to(F64)
    g, v, y = gate.cpu().to(F64)[e], up.cpu().to(F64)[e], down.cpu().to(F64)[e]
    if gated:
        a = torch.einsum("nfd,nd->nf", g, x)
        want = s * torch.einsum("ndf,nf->nd", y, a * torch.sigmoid(a) * torch.einsum("nfd,nd->nf", v, x))
    else:
        want = torch.einsum("ndf,nf->nd", y, torch.nn.functional.gelu(torch.einsum("nfd,nd->nf", v, x * s)))
    assert_close(got, want, 1e-4 if dtype == "float32" else 3e-2, "output")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("counts,d,ff", [((17, 96, 97, 0, 33, 193), 264, 48), ((128, 129, 81, 95, 0, 100), 1096, 272), ((1, 600, 31, 65), 40, 1040)])
@pytest.mark.parametrize("gated,pack", [(True, True), (False, False)])
def test_tiles_of_every_size(dtype, counts, d, ff, gated, pack, monkeypatch):
    """Which rows share a tile changes no bit."""
    from llama_cu_amd.kernels import ops
    experts, n, tdt = len(counts), sum(counts), TYPES[dtype]
    order = torch.randperm(n, generator=torch.Generator().manual_seed(0))
    ids = torch.repeat_interleave(torch.arange(experts, dtype=torch.int32), torch.tensor(counts))[order].view(n, 1).cuda()
    h, wts = rnd(n, d, seed=1).to(tdt).cuda(), torch.rand(n, 1, generator=torch.Generator().manual_seed(2)).cuda()
    gate, up = (rnd(experts, ff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (3, 4))
    u, w = ops.gated_rows(gate, up) if gated else up, rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda()
    if pack:
        u, w = ops.pack_experts(u), ops.pack_experts(w)
    got = []
    for tile in (16, 32, 48, 64, 96, 112, 128):
        monkeypatch.setattr(ops, "moe_tile_rows", lambda *sizes: tile)
        got.append(ops.moe_experts(h, ids, wts, u, w, torch.zeros(n, d, device="cuda"), **({"gated": True, "fresh": True} if gated else {})))
    for g in got[1:]:
        assert torch.equal(g, got[0])


def test_tiles_that_leave_no_compute_unit_idle():
    """Small products in small tiles, large ones in tiles that fill the compute units in whole turns; (type: 1 bfloat16, 0 32 bits)."""
    from llama_cu_amd.kernels import ops
    for sizes, rows in [((1, 400, 16, 1024, 1024, 512), 32), ((1, 1400, 16, 1024, 1024, 512), 64), ((1, 2200, 16, 1024, 1024, 512), 96), ((1, 3400, 16, 1024, 1024, 512), 128),
                        ((0, 700, 8, 1024, 1024, 1024), 32), ((0, 280, 4, 544, 520, 272), 32), ((1, 4028, 16, 2048, 2048, 2048), 96), ((1, 1400, 16, 2048, 2048, 1024), 128),
                        ((1, 256, 16, 2048, 2048, 1024), 16), ((1, 16, 16, 2048, 2048, 1024), 0)]:
        assert ops.moe_tile_rows(*sizes) == rows, sizes


@pytest.mark.parametrize("gated", [True, False])
def test_memory_that_nobody_reads_is_not_asked_for(gated):
    """One expert a token that is not gated adds its rows where they belong; a sum that begins afresh and is left to others has no rows of its own."""
    from llama_cu_amd.kernels import ops
    n, d, ff, experts = 512, 2048, 64, 4
    h = rnd(n, d, seed=1).to(torch.bfloat16).cuda()
    ids, wts = (torch.arange(n, dtype=torch.int32)[:, None] % experts).cuda(), torch.ones(n, 1, device="cuda")
    up, down = (torch.zeros(experts, r, k, dtype=torch.bfloat16, device="cuda") for r, k in (((2 if gated else 1) * ff, d), (d, ff)))
    out = torch.zeros(n, d, device="cuda") if not gated else None
    with pytest.raises(ops.KernelError):
        ops.moe_experts(h, ids, wts, up, down, None, gated=gated)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    kept = ops.moe_experts(h, ids, wts, up, down, out, gated=gated, fresh=gated, defer=gated)
    more = torch.cuda.max_memory_allocated() - before
    assert more <= 4 * n * d * gated + 2 * n * ff + (1 << 16), more            # (the pairs' rows, the activations, the lists)
    if gated:
        assert torch.equal(kept.rows(), torch.zeros(n, d, device="cuda"))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,top,experts,identity", [(1, 1, 3, 0), (1, 4, 8, 2), (3, 2, 2, 0), (16, 4, 5, 3), (16, 2, 40, 0), (17, 1, 4, 0)])
@pytest.mark.parametrize("d,ff", [(72, 32), (520, 144)])
def test_the_experts_that_any_pair_names(dtype, n, top, experts, identity, d, ff):
    """The kernel of the least pairs at its edges (one pair; every expert named; 64 pairs; 16 tokens, and 17 of which it takes none): the same bits as from tiles of 16
    sorted rows, with and without identity experts and a shared one."""
    from llama_cu_amd.kernels import build, ops
    tdt = TYPES[dtype]
    h = rnd(n, d, seed=1).to(tdt).cuda()
    gen = torch.Generator().manual_seed(2)
    ids = torch.stack([torch.randperm(experts + identity, generator=gen)[:top] for _ in range(n)]).to(torch.int32).cuda()
    wts = torch.rand(n, top, generator=gen).cuda()
    rows = ops.gated_rows(*(rnd(experts, ff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (3, 4)))
    up, down = ops.pack_experts(rows), ops.pack_experts(rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda())
    sff = 48
    shared = (ops.pack_experts(ops.gated_rows(*(rnd(1, sff, d, seed=k, std=d ** -0.5).to(tdt).cuda() for k in (6, 7)))),
              ops.pack_experts(rnd(1, d, sff, seed=8, std=sff ** -0.5).to(tdt).cuda()))
    kw = dict(gated=True, fresh=True, identity=identity, shared_expert=shared if ops.moe_shared_beside(n, top, experts, up, down) else None)
    got, want = torch.empty(n, d, device="cuda"), torch.empty(n, d, device="cuda")
    ops.moe_experts(h, ids, wts, up, down, got, **kw)
    lib = build.load("moe")
    real, lib.lcu_moe_tile_rows = lib.lcu_moe_tile_rows, lambda *a: 16
    try:
        ops.moe_experts(h, ids, wts, up, down, want, **kw)
    finally:
        lib.lcu_moe_tile_rows = real
    assert torch.equal(got, want)


def experts_of(experts, d, ff, tdt, gated):
    """Packed matrices of ``experts`` experts, and those of a shared one."""
    from llama_cu_amd.kernels import ops
    sff = 48
    rows = lambda e, f, seed: rnd(e, f, d, seed=seed, std=d ** -0.5).to(tdt).cuda()
    first = ops.gated_rows(rows(experts, ff, 3), rows(experts, ff, 4)) if gated else rows(experts, ff, 3)
    up, down = ops.pack_experts(first), ops.pack_experts(rnd(experts, d, ff, seed=5, std=ff ** -0.5).to(tdt).cuda())
    return up, down, (ops.pack_experts(ops.gated_rows(rows(1, sff, 6), rows(1, sff, 7))), ops.pack_experts(rnd(1, d, sff, seed=8, std=sff ** -0.5).to(tdt).cuda()))


def beside_tiles(h, ids, wts, up, down, monkeypatch, **kw):
    """``moe_experts`` as it chooses and from tiles of 16 sorted rows, whatever memory they are given full of NaN beforehand."""
    from llama_cu_amd.kernels import build, ops
    empty = torch.empty

    def poisoned(*a, **k):
        t = empty(*a, **k)
        return t.fill_(float("nan")) if t.is_floating_point() else t
    lib = build.load("moe")
    outs = []
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", poisoned)
        for tiles in (lib.lcu_moe_tile_rows, lambda *a: 16):
            m.setattr(lib, "lcu_moe_tile_rows", tiles)
            outs.append(torch.zeros(h.shape, device="cuda"))
            ops.moe_experts(h, ids, wts, up, down, outs[-1], **kw)
    return outs


# 9 tokens of two, all on one expert (18 pairs); 16 of four on two experts (32 each), on one (64; of 4 experts they go to the other kernel) and with a last turn of a single pair (17)
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("n,top,experts,named", [(9, 2, 2, [[0, 0]] * 9), (16, 4, 8, [[3, 5, 5, 3]] * 16), (16, 4, 4, [[1] * 4] * 16), (16, 4, 6, [[1] * 4] * 16),
                                                 (16, 2, 40, [[7, 7]] + [[7, 8]] * 15)])
@pytest.mark.parametrize("d,ff", [(72, 32), (520, 144)])
def test_an_expert_that_a_token_names_more_than_once(dtype, gated, n, top, experts, named, d, ff, monkeypatch):
    """An expert's pairs may be more than the step's tokens: every one of them is multiplied, with the bits of tiles of 16 sorted rows."""
    from llama_cu_amd.kernels import ops
    tdt = TYPES[dtype]
    up, down, shared = experts_of(experts, d, ff, tdt, gated)
    h, wts = rnd(n, d, seed=1).to(tdt).cuda(), torch.rand(n, top, generator=torch.Generator().manual_seed(2)).cuda()
    kw = dict(gated=True, fresh=True, shared_expert=shared if ops.moe_shared_beside(n, top, experts, up, down) else None) if gated else {}
    assert ops.moe_tile_rows(ops._type(h, "rows"), n * top, experts, up.shape[1], d, ff) == 0
    got, want = beside_tiles(h, torch.tensor(named, dtype=torch.int32).cuda(), wts, up, down, monkeypatch, **kw)
    assert torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_row_of_nan_among_rows_that_share_an_expert(dtype, monkeypatch):
    """The router gives a row of NaN its first expert in every place; what the other rows, which name that expert too, get from it does not change."""
    from llama_cu_amd.kernels import ops
    tdt, n, top, experts, d, ff = TYPES[dtype], 16, 4, 8, 72, 32
    up, down, shared = experts_of(experts, d, ff, tdt, True)
    h, router = rnd(n, d, seed=1).to(tdt).cuda(), rnd(experts, d, seed=2).cuda()
    bias = torch.zeros(experts, device="cuda")
    bias[0] = 100.0                                          # every row names expert 0
    healthy = ops.moe_route(h, router, top, bias)
    h[0] = float("nan")
    ids, wts = ops.moe_route(h, router, top, bias)
    assert (ids[1:] == healthy[0][1:]).all() and (ids == 0).sum() == n + top - 1
    got, want = beside_tiles(h, ids, wts, up, down, monkeypatch, gated=True, fresh=True, shared_expert=shared)
    assert torch.isnan(got[0]).all() and torch.isfinite(got[1:]).all() and torch.equal(got[1:], want[1:])
