"""Pinned host memory that kernels of this package read by its address, and when it may be written or given back.

Torch's allocator of pinned memory waits for the copies that torch itself makes from a block before it gives the block to
somebody else.  Of a kernel that reads the block by its address it knows nothing: a block that is dropped while such a
kernel waits in a queue is the next owner's at once.  Here the kernels say themselves that they have read: each of their
workgroups leaves a ticket in the block's own first entries (``ops.step_arrays``), which costs the queue nothing and
holds whatever streams they ran on.
"""
from __future__ import annotations

import collections
import ctypes
import time
import weakref
from typing import List, Optional, Tuple

import torch

MARKS = 64                  # the most workgroups of a launch that reads (step_arrays.hip)
PATIENCE = 1.0              # seconds for which a wait looks at the marks; then it waits for the whole stream

# Memory whose owner is gone while kernels still have to read it.  Each entry goes when its marks are there; looked through whenever
# an owner comes or goes.  (A deque: appending and taking from its ends need no lock, and an owner may go at any time, within a
# collection of garbage too.)
_left: collections.deque = collections.deque()


def _sweep() -> None:
    for _ in range(len(_left)):
        try:
            reads = _left.popleft()
        except IndexError:
            return
        if not all(reads.done(k) for k in range(reads.places)):
            _left.append(reads)


def _leave(reads: "HostReads") -> None:
    _sweep()
    if not all(reads.done(k) for k in range(reads.places)):
        _left.append(reads)


class HostReads:
    """The int32 tensor ``memory`` (pinned): marks for ``places`` launches, and ``data`` behind them, of which each launch reads a part (``room``)."""

    def __init__(self, memory: torch.Tensor, places: int):
        _sweep()
        self.memory, self.places = memory, int(places)
        self.data = memory[self.places * MARKS:]
        self._marks = (ctypes.c_int * (self.places * MARKS)).from_address(memory.data_ptr())
        self._ticket = 0
        self._rooms: collections.deque = collections.deque()      # (place, start, end) of the parts that were given out last, the oldest first
        self._next = self._head = 0
        self._awaited: List[Optional[Tuple[int, int, object]]] = [None] * self.places     # (marks, ticket, stream) of the launch that reads the place

    @staticmethod
    def entries(places: int, data: int) -> int:
        """Entries of a ``memory`` whose ``data`` are so many."""
        return places * MARKS + data

    def belongs_to(self, owner) -> None:
        """The memory stays until the launches that are queued when ``owner`` goes have read it.  (Nothing is asked of the GPU then: an owner may go while
        a graph is captured, and nobody waits for it.)"""
        weakref.finalize(owner, _leave, self).atexit = False

    def room(self, size: int) -> Tuple[int, int]:
        """``(place, start)``: so many entries of ``data`` (16-byte pieces) for the next launch, behind the last ones or at the beginning again.  Waits for the launches that read there
        before, oldest first, and for the oldest of all if as many as there are places are still to read."""
        size = (size + 3) // 4 * 4
        if size > self.data.numel():
            raise ValueError(f"{size} entries do not fit in the {self.data.numel()} that there are")
        start = self._head if self._head + size <= self.data.numel() else 0
        while len(self._rooms) == self.places or any(a < start + size and start < b for _, a, b in self._rooms):
            self.wait(self._rooms.popleft()[0])
        place = self._next
        self._rooms.append((place, start, start + size))
        self._next, self._head = (place + 1) % self.places, start + size
        return place, start

    def next_ticket(self) -> int:
        self._ticket = self._ticket % 0x7fffffff + 1
        return self._ticket

    def launched(self, place: int, marks: int, ticket: int, stream) -> None:
        """A launch that reads ``place`` stands in ``stream`` and will leave ``ticket`` in the place's first ``marks`` marks."""
        self._awaited[place] = (marks, ticket, stream) if marks else None

    def done(self, place: int) -> bool:
        """Whether what was launched last has read ``place``."""
        awaited = self._awaited[place]
        if awaited is None:
            return True
        marks, ticket, _ = awaited
        at = place * MARKS
        if any(self._marks[k] != ticket for k in range(at, at + marks)):
            return False
        self._awaited[place] = None
        return True

    def wait(self, place: int) -> None:
        """Wait until what was launched last has read ``place``."""
        if self.done(place):
            return
        end = time.perf_counter() + PATIENCE
        while not self.done(place):
            if time.perf_counter() < end:
                time.sleep(0)                # (other threads run)
                continue
            self._awaited[place][2].synchronize()        # a step of more than a second, or one that failed
            if not self.done(place):
                self._awaited[place] = None
                raise RuntimeError("a step's arrays were never read: its launch was recorded and not run, or failed")
