"""The sum of a token's experts inside the norm that adds it to the residual stream, against the sum made first: the same bits; and the sum against 64 bits."""
import pytest
import torch

from test_gpu_divasun import F64, TYPES, hand_step, rnd

pytestmark = pytest.mark.gpu


def pair_sum(n, d, dtype, top, base, wts, shared, identity, seed=0):
    """``(sum, its value in 64 bits)``; rows of y that belong to identity experts hold NaN: nobody may use them."""
    from llama_cu_amd.kernels import ops
    real, tdt = 5, TYPES[dtype]
    y, h = rnd(n * top, d, seed=seed), rnd(n, d, seed=seed + 1).to(tdt)
    w = rnd(n, top, seed=seed + 2) if wts else None
    b = rnd(n, d, seed=seed + 3) if base else None
    s, s32 = (rnd(n, d, seed=seed + 4).to(tdt) if shared == "rows" else None), (rnd(n, d, seed=seed + 4) if shared == "32" else None)
    gate = rnd(n, seed=seed + 5) if shared else None
    ids = torch.randint(0, real + 3, (n, top), generator=torch.Generator().manual_seed(seed), dtype=torch.int32) if identity else None
    want = b.to(F64) if base else torch.zeros(n, d, dtype=F64)
    for k in range(top):
        rows = y.view(n, top, d)[:, k].to(F64)
        if identity:
            rows = torch.where((ids[:, k] >= real)[:, None], h.to(F64), rows)
        want = want + rows * (w[:, k:k + 1].to(F64) if wts else 1.0)
    if shared:
        want = want + gate[:, None].to(F64) * (s if s is not None else s32).to(F64)
    if identity:
        y.view(n, top, d)[ids >= real] = float("nan")
    c = lambda t: t.cuda() if t is not None else None
    return ops.PairSum(n, d, tdt, top, c(y), c(w), c(b), c(s), c(s32), c(gate), c(ids), c(h), real), want


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("base", [True, False])
@pytest.mark.parametrize("shared", [None, "rows", "32"])
@pytest.mark.parametrize("top", [1, 2, 3])
def test_roundings_of_its_terms(dtype, base, shared, top):
    """Bit for bit: an expert's product is rounded, then added; the shared expert's is added in one rounding."""
    n, d = 7, 1028
    p, _ = pair_sum(n, d, dtype, top, base, True, shared, True, seed=3)
    c = lambda t: t.cpu() if t is not None else None
    y, w, ids, h, own, gate = c(p.y).view(n, top, d), c(p.wts), c(p.ids), c(p.h).float(), c(p.shared if p.shared is not None else p.shared32), c(p.gate)
    want = c(p.base).clone() if base else torch.zeros(n, d)
    for k in range(top):
        want = want + w[:, k:k + 1] * torch.where((ids[:, k] >= p.real)[:, None], h, y[:, k])
    if shared:
        want = (want.to(F64) + gate[:, None].to(F64) * own.to(F64)).float()          # (the product of two 32-bit numbers is exact in 64 bits)
    assert torch.equal(p.rows().cpu(), want)


# widths of one and of two pieces a thread at both numbers of threads, with rests; beyond and beside what the norms' kernels add up
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,d,top,base,wts,shared,identity", [
    (1, 4, 1, True, False, None, False), (3, 1024, 2, True, True, "32", True), (5, 1028, 3, False, True, "rows", False), (2, 2048, 2, True, False, None, False),
    (70, 2052, 5, False, True, "32", True), (2, 4096, 4, True, True, "rows", True), (2, 4100, 2, False, True, None, False)])
def test_the_norms_add_it_up(dtype, n, d, top, base, wts, shared, identity):
    from llama_cu_amd.kernels import ops
    tdt = TYPES[dtype]
    made = lambda: pair_sum(n, d, dtype, top, base, wts, shared, identity)
    p, want = made()
    rows = p.rows()
    # top + 2 terms of about one each, a rounding of 2^-24 of the partial sum behind each
    assert (rows.cpu().to(F64) - want).abs().max() <= (top + 2) * 2.0 ** -22 * want.abs().max()
    vec = lambda k: (rnd(d, seed=k) + 1).cuda()
    x = rnd(n, d, seed=50).cuda()
    for out_dtype in {tdt, torch.float32}:
        got, ref = [], []
        for delta, to in ((made()[0], got), (rows, ref)):
            a, o1, o2 = x.clone(), torch.empty(n, d, dtype=out_dtype, device="cuda"), torch.empty(n, d, dtype=out_dtype, device="cuda")
            ops.layernorm(a, vec(1), vec(2), 1e-5, o1, delta=delta, weight2=vec(3), bias2=vec(4), out2=o2)
            to += [a, o1, o2]
            b = x.clone()
            to += [b, ops.norm_post(b, delta if to is ref else made()[0], vec(5), 1e-5, vec(6), 1e-6, out_dtype=out_dtype)]
            c = x.clone()
            to += [c, ops.norm_post(c, delta if to is ref else made()[0], vec(5), 1e-5) or c, ops.norm_post(c, delta if to is ref else made()[0], vec(5), 1e-5, out_dtype=out_dtype)]
        for k, (g, r) in enumerate(zip(got, ref)):
            assert torch.equal(g, r), k


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("d,taps,sets", [(4, 1, 1), (1024, 2, 2), (1028, 3, 2), (2048, 4, 2), (2048, 8, 1), (600, 5, 2)])
def test_the_norms_with_their_convolutions_add_it_up(dtype, d, taps, sets):
    from llama_cu_amd.kernels import ops
    n, tdt = 3, TYPES[dtype]
    vec = lambda k: (rnd(d, seed=k) + 1).cuda()
    cw, x = rnd(sets, d, taps, seed=60).cuda(), rnd(n, d, seed=50).cuda()
    got, ref = [], []
    for to in (got, ref):
        p, _ = pair_sum(n, d, dtype, 2, True, True, None, False)
        a, state = x.clone(), rnd(n, sets, max(taps - 1, 1), d, seed=61).cuda()[:, :, :taps - 1].contiguous()
        out = ops.norm_conv_single(a, p if to is got else p.rows(), [vec(k) for k in range(sets)], [vec(3 + k) for k in range(sets)], 1e-5, cw, state,
                                   torch.empty(sets, n, d, dtype=tdt, device="cuda"), hand_step([1] * n, [1, 3, 9], [2, 0, 1]))
        to += [a, state, out]
    for k, (g, r) in enumerate(zip(got, ref)):
        assert torch.equal(g, r), k


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rows_that_begin_at_any_element(dtype):
    """Contiguous rows within a larger tensor, one element past its start: taken by the experts as they are, and by the norms."""
    from llama_cu_amd.kernels import ops
    n, d, ff, experts, tdt = 5, 64, 32, 4, TYPES[dtype]

    def past(t):
        whole = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        part = whole[1:].view(t.shape)
        part.copy_(t)
        return part
    gate, up, down = (rnd(experts, *s, seed=k, std=0.1).to(tdt).cuda() for k, s in enumerate(((ff, d), (ff, d), (d, ff))))
    w = ops.gated_rows(gate, up)
    ids = torch.randint(0, experts + 2, (n, 2), generator=torch.Generator().manual_seed(1), dtype=torch.int32).cuda()
    h, shared, out, wts = rnd(n, d, seed=5).to(tdt).cuda(), rnd(n, d, seed=6).to(tdt).cuda(), rnd(n, d, seed=7).cuda(), rnd(n, 2, seed=8).cuda()
    run = lambda h, shared, out, **kw: ops.moe_experts(h, ids, wts, w, down, out, gated=True, shared=shared, identity=2, **kw)
    want = run(h, shared, out.clone())
    assert torch.equal(run(past(h), past(shared), past(out)), want)
    vec = lambda k: (rnd(d, seed=k) + 1).cuda()
    x, a, b = rnd(n, d, seed=9).cuda(), torch.empty(n, d, dtype=tdt, device="cuda"), torch.empty(n, d, dtype=tdt, device="cuda")
    x2 = x.clone()
    ops.layernorm(x, vec(1), vec(2), 1e-5, a, delta=want)
    ops.layernorm(x2, vec(1), vec(2), 1e-5, b, delta=run(past(h), past(shared), past(out), defer=True))
    assert torch.equal(x, x2) and torch.equal(a, b)


def test_a_sum_is_added_up_once():
    """A second time would add the terms twice where the sum lies in one of them; and they are let go of."""
    from llama_cu_amd.kernels import ops
    vec = (rnd(64, seed=1) + 1).cuda()
    uses = [lambda p: p.rows(), lambda p: ops.norm_post(rnd(3, 64).cuda(), p, vec, 1e-5),
            lambda p: ops.layernorm(rnd(3, 64).cuda(), vec, vec, 1e-5, torch.empty(3, 64, device="cuda"), delta=p),
            lambda p: ops.norm_conv_single(rnd(3, 64).cuda(), p, [vec], [vec], 1e-5, torch.ones(1, 64, 1, device="cuda"), torch.empty(3, 1, 0, 64, device="cuda"),
                                           torch.empty(1, 3, 64, device="cuda"), hand_step([1] * 3, [1, 2, 3], [0, 1, 2]))]
    for use in uses:
        p, _ = pair_sum(3, 64, "float32", 2, True, True, None, False)
        use(p)
        assert p.y is None and p.base is None
        for again in uses:
            with pytest.raises(ops.KernelError):
                again(p)
