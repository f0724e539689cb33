"""When memory that queued kernels read may be written or given back; the marks are written by hand here."""
import gc
import threading
import time

import pytest
import torch

import llama_cu_amd  # noqa: F401
from llama_cu_amd.engine import host_reads
from llama_cu_amd.engine.host_reads import MARKS, HostReads


class Owner:
    pass


class Stream:
    def __init__(self, run=lambda: None):
        self.run = run

    def synchronize(self):
        self.run()


def reads_of(places, data=8):
    return HostReads(torch.zeros(HostReads.entries(places, data), dtype=torch.int32), places)


def mark(reads, place, marks, ticket):
    reads.memory[place * MARKS:place * MARKS + marks] = ticket


def test_a_place_is_read_when_every_workgroup_of_its_own_launch_says_so():
    r = reads_of(3)
    assert r.data.numel() == 8 and all(r.done(k) for k in range(3))
    t = r.next_ticket()
    r.launched(1, 3, t, None)
    assert r.done(0) and r.done(2) and not r.done(1)
    mark(r, 0, 3, t)                                  # another place's
    mark(r, 1, 2, t)
    assert not r.done(1)
    mark(r, 1, 3, t)
    assert r.done(1)
    u = r.next_ticket()
    r.launched(1, 3, u, None)                         # what the launch before left counts for nothing
    assert u != t and not r.done(1)
    mark(r, 1, 3, u)
    assert r.done(1)
    r.launched(1, 0, r.next_ticket(), None)           # nothing was launched
    assert r.done(1)


def test_tickets_stay_positive():
    r = reads_of(1)
    r._ticket = 0x7ffffffe
    assert [r.next_ticket() for _ in range(3)] == [0x7fffffff, 1, 2]


def test_waiting(monkeypatch):
    r = reads_of(2)
    t = r.next_ticket()
    r.launched(0, 2, t, None)
    later = threading.Thread(target=lambda: (time.sleep(0.05), mark(r, 0, 2, t)))
    later.start()
    r.wait(0)
    assert r.done(0)
    later.join()
    # beyond its patience it waits for the stream
    monkeypatch.setattr(host_reads, "PATIENCE", 0.0)
    u = r.next_ticket()
    r.launched(1, 1, u, Stream(lambda: mark(r, 1, 1, u)))
    r.wait(1)
    r.launched(1, 1, r.next_ticket(), Stream())
    with pytest.raises(RuntimeError):
        r.wait(1)


def test_room_is_given_again_when_it_has_been_read():
    """Parts of all sizes in turn: none overlaps one that is still to be read, and nobody waits who need not."""
    gen = torch.Generator().manual_seed(5)
    r = reads_of(4, 64)
    waited, queued = [], []                           # queued: (place, start, end, ticket), read from the front on

    def wait(place):
        if not r.done(place):
            waited.append(place)
            while not r.done(place):
                p, _, _, t = queued.pop(0)
                mark(r, p, 1, t)
    r.wait = wait
    for turn in range(400):
        size = int(torch.randint(1, 65 if turn % 7 == 0 else 20, (1,), generator=gen))
        before = list(queued)
        del waited[:]
        place, start = r.room(size)
        assert start % 4 == 0 and start + size <= 64
        assert all(place != p and (end <= start or start + size <= a) for p, a, end, _ in queued)
        assert not waited or len(before) == 4 or any(a < start + size and start < end for _, a, end, _ in before)
        t = r.next_ticket()
        r.launched(place, 1, t, None)
        queued.append((place, start, start + size, t))
        if turn % 3 == 0:                             # the oldest is read
            p, _, _, t = queued.pop(0)
            mark(r, p, 1, t)
    with pytest.raises(ValueError):
        r.room(65)
    assert reads_of(2, 64).room(64) == (0, 0)


def test_memory_stays_until_it_has_been_read():
    host_reads._sweep()
    before = len(host_reads._left)
    owner, r = Owner(), reads_of(2)
    memory, t = r.memory, r.next_ticket()
    r.belongs_to(owner)
    r.launched(1, 2, t, None)
    del r
    assert len(host_reads._left) == before            # its owner is there
    del owner
    gc.collect()
    assert len(host_reads._left) == before + 1 and host_reads._left[-1].memory is memory
    other, idle = Owner(), reads_of(1)                # another owner comes and goes with nothing queued
    idle.belongs_to(other)
    del other, idle
    gc.collect()
    assert len(host_reads._left) == before + 1
    memory[MARKS:MARKS + 2] = t
    reads_of(1)
    assert len(host_reads._left) == before
