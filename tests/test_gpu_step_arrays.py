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


@pytest.mark.parametrize("pieces", [[(0, 4, 1, 0, 4)], [(0, 1020, 1, 0, 1024), (1024, 4, 7, 12, 8), (1200, 0, 2, 8, 8), (2000, 2096, 1, 0, 2096)],
                                    [(8 * i, 4, 1, 0, 4 + 4 * (i % 2)) for i in range(61)], [(0, 262140, 1, 0, 262140)], []])
def test_pieces_of_ordinary_memory_come_over_packed(pieces):
    """What stands in pinned memory is the pieces, one behind the other, and no more."""
    from llama_cu_amd.kernels import ops
    n = 262144
    size = sum(cols * rows for _, cols, rows, _, _ in pieces)
    host = torch.arange(1, n + 1, dtype=torch.int32)
    pinned = torch.zeros(n + 8, dtype=torch.int32).pin_memory()
    dev = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    at = ops.host_on_device(pinned)
    for turn in range(3):
        host += turn
        want = dev.cpu()
        for a, cols, rows, stride, width in pieces:
            for r in range(rows):
                want[a + r * stride:a + r * stride + cols] = host[a + r * stride:a + r * stride + cols]
                want[a + r * stride + cols:a + r * stride + width] = 0
        ops.step_arrays(at + 16, dev, pieces, arrays=host, packed=pinned[4:4 + size])
        torch.cuda.synchronize()
        assert torch.equal(dev.cpu(), want)
        assert not pinned[:4].any() and not pinned[4 + size:].any()
    if size:
        with pytest.raises(ops.KernelError):
            ops.step_arrays(at + 16, dev, pieces, arrays=host, packed=pinned[4:size])


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


def test_marks_say_that_everything_has_been_read():
    """Of one launch and of the several that many pieces take; places of 24 pieces a launch, 64 workgroups."""
    from llama_cu_amd.engine.host_reads import MARKS
    from llama_cu_amd.kernels import ops
    n = 1 << 20
    host = torch.zeros(MARKS + n, dtype=torch.int32).pin_memory()
    dev = torch.zeros(n, dtype=torch.int32, device="cuda")
    at = ops.host_on_device(host)
    whole = lambda a, c: (a, c, 1, 0, c)
    for ticket, (pieces, marks) in enumerate([([whole(0, 4)], 1), ([whole(0, 1024)], 1), ([whole(0, 1028)], 2), ([whole(0, n)], 64), ([], 0), ([whole(0, 0)], 0),
                                              ([whole(4 * i, 4) for i in range(25)], 1), ([whole(0, n // 2)] + [whole(n // 2 + 4 * i, 4) for i in range(47)] + [whole(0, 0)] * 3, 1)], 5):
        left = ops.step_arrays(at + 4 * MARKS, dev, pieces, at, ticket)
        torch.cuda.synchronize()
        assert left == marks
        assert host[:marks].tolist() == [ticket] * marks and not (host[marks:MARKS] == ticket).any()


def builder_of(positions, max_tokens=32):
    import llama_cu_amd  # noqa: F401
    from llama_cu_amd.cache import CacheGroup, CacheManager
    from llama_cu_amd.engine.batch import BatchBuilder
    groups = [CacheGroup(40, 8, 0), CacheGroup(20, 16, 0)]
    cache = CacheManager(groups, 4)
    builder = BatchBuilder(cache, max_tokens, 4, [-(-positions // g.page_size) for g in groups], torch.device("cuda:0"))
    torch.cuda.synchronize()                # (its device buffer is cleared on this stream; the steps may come on others)
    return cache, builder


def busy(a, times=200):
    """Some tens of milliseconds of ordinary work on the current stream."""
    for _ in range(times):
        a = (a @ a).clamp_(-1, 1)
    return a


def test_a_builder_that_goes_has_its_queued_step_read_first():
    """The step stands behind other work when its builder goes; who asks for pinned memory then must not get what the step will read."""
    import gc
    from llama_cu_amd.engine import host_reads
    a = torch.eye(4096, device="cuda")
    host_reads._sweep()
    assert not host_reads._left
    cache, builder = builder_of(96)
    cache.add(0)
    assert cache.reserve(0, 20)
    entries = builder._reads.memory.numel()
    torch.cuda.synchronize()
    busy(a)
    step = builder.build([0], [list(range(1, 21))], [[3, 19]], 50, upload=False)
    names = ["tokens", "positions", "logit_rows", "slots0", "block_table1"]
    want = [builder._h(name)[:t.numel()].clone() for name, t in zip(names, (step.tokens, step.positions, step.logit_rows, step.slot_maps[0], step.block_tables[1]))]
    builder.upload()
    got = [t.clone() for t in (step.tokens, step.positions, step.logit_rows, step.slot_maps[0], step.block_tables[1])]
    del builder, step
    gc.collect()
    assert len(host_reads._left) == 1                # (the work in front takes longer than the lines between)
    fresh = [torch.full((entries,), -7, dtype=torch.int32).pin_memory() for _ in range(4)]
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert torch.equal(g.flatten().cpu(), w)
    builder_of(96)
    assert not host_reads._left and all((f == -7).all() for f in fresh)


@pytest.mark.parametrize("ordered", ["one stream", "two streams"])
def test_steps_that_queue_up_bring_their_own_arrays(ordered):
    """More steps than the builder has room for are built while the GPU is busy with other work: it waits for the reads of the oldest, and each step's arrays are its own."""
    a = torch.eye(4096, device="cuda")
    cache, builder = builder_of(96)
    cache.add(0)
    waits, length = [], 0
    wait = builder._reads.wait
    builder._reads.wait = lambda place: (waits.append(not builder._reads.done(place)), wait(place))[1]
    streams = [torch.cuda.Stream() for _ in range(2)] if ordered == "two streams" else [torch.cuda.current_stream()] * 2
    torch.cuda.synchronize()
    seen = []
    steps = 3 * builder.RING + 1
    with torch.cuda.stream(streams[0]):
        busy(a)
    for k in range(steps):
        length += 1 + k % 3
        assert cache.reserve(0, length)
        stream = streams[k // 2 % 2]
        if ordered == "two streams":
            stream.wait_stream(streams[1 - k // 2 % 2])      # (one device buffer: on the GPU a stream's step stands behind the other's; the host does not wait)
        with torch.cuda.stream(stream):
            step = builder.build([0], [[(5 * k + j) % 50 for j in range(1 + k % 3)]], [[0]], 50)
            seen.append((step.tokens.clone(), step.ctx_len.clone()))
        cache.commit(0)
    torch.cuda.synchronize()
    assert any(waits)
    length = 0
    for k, (tokens, ctx) in enumerate(seen):
        length += 1 + k % 3
        assert tokens.tolist() == [(5 * k + j) % 50 for j in range(1 + k % 3)] and ctx.tolist() == [length], k


def test_a_step_may_go_to_the_device_again():
    """With what was added to its arrays after the first time, and with its other arrays as they were; the next step's come behind it."""
    cache, builder = builder_of(96)
    cache.add(0)
    length = 0
    for k in range(2 * builder.RING + 1):
        tokens = [(11 * k + j) % 50 for j in range(1 + k % 2)]
        length += len(tokens)
        assert cache.reserve(0, length)
        step = builder.build([0], [tokens], [[0]], 50)
        cache.commit(0)
        host, dev = step.extra("late", 8)
        host[:8] = torch.arange(8, dtype=torch.int32) + 100 * k
        step.tokens.zero_()                          # (what the second launch brings is not what the first one left)
        builder.upload()
        assert step.tokens.tolist() == tokens and step.ctx_len.tolist() == [length] and step.q_start.tolist() == [0, len(tokens)]
        assert dev.tolist() == [100 * k + j for j in range(8)]


@pytest.mark.parametrize("positions", [96, 90])
def test_steps_in_turn_bring_their_own_arrays(positions):
    """More steps than the builder has room for, on two streams in turn, the host waiting for one when it goes on with the other: all arrays of each step are its own."""
    cache, builder = builder_of(positions)
    max_pages = builder.max_pages
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
