"""The pool of pinned result blocks, with host memory in the library's place."""

import ctypes as C
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
