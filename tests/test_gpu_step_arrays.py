"""What a step brings to the device in one launch, against the host's own arrays."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pieces", [[(0, 4, 1, 0, 4)], [(8, 0, 3, 8, 4)], [(0, 1020, 1, 0, 1024), (1024, 4, 7, 12, 8), (2000, 2096, 1, 0, 2096)],
                                    [(8 * i, 4, 1, 0, 4 + 4 * (i % 2)) for i in range(61)], [(0, 262140, 1, 0, 262140)], []])
def test_pieces_come_over_and_nothing_else_changes(pieces):
    from llama_cu_amd.kernels import ops
    n = 262144
    host = torch.arange(1, n + 1, dtype=torch.int32).pin_memory()
    dev = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    at = ops.host_on_device(host)
    for turn in range(3):                   # the host's values change between launches: nothing old may be read
        host += turn
        want = dev.cpu()
        for a, cols, rows, stride, width in pieces:
            for r in range(rows):
                want[a + r * stride:a + r * stride + cols] = host[a + r * stride:a + r * stride + cols]
                want[a + r * stride + cols:a + r * stride + width] = 0
        ops.step_arrays(at, dev, pieces)
        torch.cuda.synchronize()
        assert torch.equal(dev.cpu(), want)


def test_pieces_outside_the_array_are_refused():
    from llama_cu_amd.kernels import ops
    host = torch.zeros(64, dtype=torch.int32).pin_memory()
    dev = torch.zeros(64, dtype=torch.int32, device="cuda")
    at = ops.host_on_device(host)
    for piece in [(-4, 4, 1, 0, 4), (2, 4, 1, 0, 4), (60, 8, 1, 0, 8), (0, 8, 1, 0, 4), (0, 8, 9, 8, 8), (0, 8, 2, 4, 8)]:
        with pytest.raises(ops.KernelError):
            ops.step_arrays(at, dev, [piece])
    with pytest.raises(ops.KernelError):
        ops.host_on_device(torch.zeros(4, dtype=torch.int32))


@pytest.mark.parametrize("positions", [96, 90])
def test_steps_in_turn_bring_their_own_arrays(positions):
    """More steps than the builder has host buffers, on two streams in turn, without a wait between them: each step's device arrays are its own."""
    import llama_cu_amd  # noqa: F401
    from llama_cu_amd.cache import CacheGroup, CacheManager
    from llama_cu_amd.engine.batch import BatchBuilder
    groups = [CacheGroup(40, 8, 0), CacheGroup(20, 16, 0)]
    cache = CacheManager(groups, 4)
    max_pages = [-(-positions // g.page_size) for g in groups]
    device = torch.device("cuda:0")
    builder = BatchBuilder(cache, 32, 4, max_pages, device)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    seen = []
    lengths = {0: 0, 1: 0, 2: 0}
    for k in range(3 * builder.RING + 1):
        ids = [0, 1, 2] if k % 3 else [2, 0]
        toks = [[(7 * k + i) % 50] * (1 + (k + i) % 3) for i in ids]
        for i, t in zip(ids, toks):
            if lengths[i] + len(t) > positions:
                cache.release(i)
                lengths[i] = 0
            if not cache.has(i):
                cache.add(i)
            assert cache.reserve(i, lengths[i] + len(t))
        stream = streams[k // 2 % 2]
        streams[1 - k // 2 % 2].synchronize()     # one device buffer: a stream's step begins when the other's has ended
        with torch.cuda.stream(stream):
            step = builder.build(ids, toks, [[0]] * len(ids), 50, upload=False)
            host, dev = step.extra("mine", 6)
            host[:6] = torch.arange(6, dtype=torch.int32) + 10 * k
            builder_host = [t.clone() for t in (builder._h("positions")[:step.n], builder._h("block_table0")[:len(ids) * max_pages[0]],
                                                builder._h("block_table1")[:len(ids) * max_pages[1]], builder._h("slots1")[:step.n], builder._h("ctx_len")[:len(ids)])]
            builder.upload()
            seen.append((builder_host + [torch.tensor([t for ts in toks for t in ts], dtype=torch.int32), torch.arange(6, dtype=torch.int32) + 10 * k],
                         [t.clone() for t in (step.positions, step.block_tables[0].reshape(-1), step.block_tables[1].reshape(-1), step.slot_maps[1], step.ctx_len,
                                              step.tokens, dev)]))
        for i, t in zip(ids, toks):
            cache.commit(i)
            lengths[i] += len(t)
    torch.cuda.synchronize()
    for k, (want, got) in enumerate(seen):
        for w, g in zip(want, got):
            assert torch.equal(w, g.cpu()), k
