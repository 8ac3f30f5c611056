"""The pool of pinned result blocks, with host memory in the library's place."""

import ctypes as C
import mmap
import os
import threading

import numpy as np
import pytest

from pygpukit_amd.core import pinned


class _HostMemory:
    def __init__(self):
        self.blocks = {}

    def pgk_host_alloc(self, p, nbytes):
        block = C.create_string_buffer(nbytes)
        p._obj.value = C.addressof(block)
        self.blocks[p._obj.value] = block
        return 0

    def pgk_host_free(self, p):
        del self.blocks[p.value]
        return 0


@pytest.fixture
def memory(monkeypatch):
    m = _HostMemory()
    monkeypatch.setattr(pinned._hip, "load", lambda: m)
    monkeypatch.setattr(pinned, "_free", {})
    monkeypatch.setattr(pinned, "_free_bytes", 0)
    return m


def test_a_block_that_ends_while_its_own_thread_holds_the_pool(memory):
    """As when a collection of cyclic garbage runs under the pool's lock: the thread goes on."""
    held = [pinned.empty((100,))]

    def end_it():
        with pinned._lock:
            held.clear()

    t = threading.Thread(target=end_it, daemon=True)
    t.start()
    t.join(10)
    assert not t.is_alive()
    assert len(pinned._free[400]) == 1


@pytest.mark.parametrize("over", [0, 1])
def test_arrays_beyond_the_pool_are_ordinary_ones(memory, monkeypatch, over):
    monkeypatch.setattr(pinned, "POOL_BYTES", 4000)
    a = pinned.empty((1000 + over,))
    a[:] = 1
    assert len(memory.blocks) == 1 - over and a.dtype == np.float32
    del a
    assert pinned._free_bytes == (0 if over else 4000)


def _count(memory):
    calls = []
    alloc, free = memory.pgk_host_alloc, memory.pgk_host_free
    memory.pgk_host_alloc = lambda p, n: (calls.append(n), alloc(p, n))[1]
    memory.pgk_host_free = lambda p: (calls.append(-1), free(p))[1]
    return calls


def test_results_of_varying_size_share_blocks(memory):
    """1 to 24 rows of 15194 values, each result dropped when the next is there: two blocks are in use at a time, of the six sizes from 64 KiB to 2 MiB."""
    calls = _count(memory)
    rng = np.random.default_rng(0)
    for rows in rng.integers(1, 25, 400):
        out = pinned.empty((int(rows), 15194))
        out[:] = rows
        assert (out == rows).all()
    del out
    assert len(calls) <= 12 and -1 not in calls
    assert pinned._free_bytes == sum(calls) and pinned._held_bytes == 0


def test_a_full_pool_makes_room_for_another_size(memory, monkeypatch):
    monkeypatch.setattr(pinned, "POOL_BYTES", 1 << 20)
    held = [pinned.empty((16384,)) for _ in range(16)]
    del held
    assert pinned._free_bytes == 1 << 20
    calls = _count(memory)
    for _ in range(20):
        out = pinned.empty((1 << 17,))
        del out
    assert calls == [-1] * 8 + [1 << 19]
    assert sum(len(b) for b in memory.blocks.values()) == 1 << 20


def test_what_arrays_hold_is_bounded_too(memory, monkeypatch):
    """Results that are kept: pinned up to the pool's size, ordinary from then on, and pinned again once they are gone."""
    monkeypatch.setattr(pinned, "POOL_BYTES", 1 << 20)
    held = [pinned.empty((16384,)) for _ in range(20)]
    for i, a in enumerate(held):
        a[:] = i
    assert [a.base is not None for a in held] == [True] * 16 + [False] * 4
    assert all((a == i).all() for i, a in enumerate(held))
    assert pinned.empty((5,)).base is None
    del held, a
    assert pinned.empty((16384,)).base is not None and len(memory.blocks) == 16


def test_the_end_of_a_block_calls_nothing_of_the_device(memory, monkeypatch):
    """It may come in any thread, and inside a stream capture."""
    held = [pinned.empty((100000,)) for _ in range(8)]
    monkeypatch.setattr(pinned, "POOL_BYTES", 1 << 19)
    calls = _count(memory)
    del held
    assert calls == []


def test_a_refused_allocation_leaves_an_ordinary_array_and_the_counts(memory):
    memory.pgk_host_alloc = lambda p, n: 2
    held = pinned._held_bytes
    assert pinned.empty((100000,)).base is None and pinned._held_bytes == held


def test_a_forked_process_reads_the_arrays_that_were_there(memory, monkeypatch):
    """With memory that is not inherited, as the driver's: blocks of their own and two that share a page."""
    maps = []

    def alloc(p, nbytes):
        if nbytes > 4096 or not maps:
            maps.append(mmap.mmap(-1, max(nbytes, 4096)))
            maps[-1].madvise(mmap.MADV_DONTFORK)
            at = 0
        else:
            at = 1024
        p._obj.value = C.addressof(C.c_char.from_buffer(maps[-1])) + at
        return 0

    memory.pgk_host_alloc = alloc
    held = [pinned.empty((n,)) for n in (100, 200, 30000, 200000)]
    gone = pinned.empty((300000,))
    del gone
    for i, a in enumerate(held):
        a[:] = np.arange(a.size) + i
    part = held[3][777:]
    child = os.fork()
    if child == 0:
        status = 1
        try:
            ok = all((a == np.arange(a.size) + i).all() for i, a in enumerate(held)) and part[0] == 780
            held[2][:] = 0
            ok = ok and pinned.empty((300000,)).base is None
            held.clear()
            status = 0 if ok else 2
        finally:
            os._exit(status)
    assert os.waitpid(child, 0)[1] == 0
    assert all((a == np.arange(a.size) + i).all() for i, a in enumerate(held))
    assert not pinned._at_fork and pinned.empty((300000,)).base is not None
