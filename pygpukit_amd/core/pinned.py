"""NumPy arrays on pinned host memory, for results that a call copies back from the device.

Into pageable memory the runtime copies by way of its own pinned buffers and touches every fresh page of the result: a prompt of 93 tokens with its
151936 fp32 logits took 1.23 ms that way, 1.15 into a pinned array, sixteen prompts in one call 5.4 and 5.0.  A block returns to the pool with the last view
of its array.  Blocks that arrays hold and free ones together are at most POOL_BYTES: beyond, arrays are ordinary ones, so a caller that keeps its results pays for
64 MiB of allocations (0.03 to 0.4 ms a MiB) and from then on what pageable memory costs.  Results of varying size share blocks: from CLASS_BYTES on a block is a
power of two and serves whatever fits (400 calls of 1 to 24 rows of logits, each result dropped at the next call: at most ten allocations; 242 where a block only
served its own size).

Pinned pages are not inherited by a forked process (the driver maps them so), where an ordinary array's are: the arrays that are alive at a fork get pages with
their values at the same addresses in the child, and the child's own results are ordinary arrays."""

from __future__ import annotations

import ctypes as C
import math
import mmap
import os
import sys
import threading

import numpy as np

from pygpukit_amd import _hip

POOL_BYTES = 64 << 20
CLASS_BYTES = 32 << 10
_lock = threading.RLock()   # a garbage collection under it may end another block in the same thread
_free: dict[int, list[int]] = {}
_free_bytes = 0
_held_bytes = 0
_held: dict[int, int] = {}   # address -> bytes that its array uses
_forked = False


class _Block:
    """Owner of one pinned allocation; the array made from it keeps it alive.  Its end calls nothing of the device's: memory is given back in empty()."""

    def __init__(self, address: int, nbytes: int, used: int, shape: tuple, typestr: str):
        self.address, self.nbytes = address, nbytes
        _held[address] = used
        self.__array_interface__ = {"data": (address, False), "shape": shape, "typestr": typestr, "version": 3}

    def __del__(self):
        global _free_bytes, _held_bytes
        if sys is None or sys.is_finalizing() or _forked:   # the process's memory goes with it; a child has no pool
            return
        with _lock:
            _held.pop(self.address, None)
            _free.setdefault(self.nbytes, []).append(self.address)
            _free_bytes += self.nbytes
            _held_bytes -= self.nbytes


def _take(size: int):
    """(address, size) of the smallest free block that serves `size` bytes, or None; under the lock"""
    if _free.get(size):
        return _free[size].pop(), size
    fits = [n for n in list(_free) if _free[n] and n >= size >= CLASS_BYTES]
    return (_free[min(fits)].pop(), min(fits)) if fits else None


def empty(shape: tuple, dtype=np.float32) -> np.ndarray:
    """np.empty on pinned memory; on ordinary memory for what the pool has no room for and where no pinned memory is to be had."""
    global _free_bytes, _held_bytes
    dtype, shape = np.dtype(dtype), tuple(int(n) for n in shape)
    size = nbytes = math.prod(shape) * dtype.itemsize
    if nbytes >= CLASS_BYTES:
        size = 1 << (nbytes - 1).bit_length()
    if nbytes == 0 or size > POOL_BYTES or _forked:
        return np.empty(shape, dtype)
    address, evicted = None, []
    with _lock:
        found = _take(size)
        if found:
            address, size = found
            _free_bytes -= size
        else:
            if _held_bytes + size > POOL_BYTES:
                return np.empty(shape, dtype)
            while _held_bytes + _free_bytes + size > POOL_BYTES and any(_free.values()):
                n = max(n for n in list(_free) if _free[n])
                evicted.append(_free[n].pop())
                _free_bytes -= n
        _held_bytes += size
    for a in evicted:
        _hip.load().pgk_host_free(C.c_void_p(a))
    if address is None:
        p = C.c_void_p()
        if _hip.load().pgk_host_alloc(C.byref(p), size) != 0 or not p.value:
            with _lock:
                _held_bytes -= size
            return np.empty(shape, dtype)
        address = p.value
    return np.asarray(_Block(address, size, nbytes, shape, dtype.str))


_at_fork: list[tuple[int, bytes]] = []


def _before_fork():
    _lock.acquire()
    _at_fork.extend((a, C.string_at(a, n)) for a, n in list(_held.items()))


def _after_fork_in_parent():
    _at_fork.clear()
    _lock.release()


def _after_fork_in_child():
    global _forked
    libc_mmap = C.CDLL(None).mmap
    libc_mmap.restype, libc_mmap.argtypes = C.c_void_p, [C.c_void_p, C.c_size_t, C.c_int, C.c_int, C.c_int, C.c_long]
    fixed_noreplace = 0x100000           # pages that the child has are left to it

    def mapped(first, nbytes):
        return libc_mmap(first, nbytes, mmap.PROT_READ | mmap.PROT_WRITE, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | fixed_noreplace, -1, 0) == first

    for address, values in _at_fork:
        first, end = address & -mmap.PAGESIZE, address + len(values)
        if not mapped(first, end - first):           # a neighbour has mapped a page of it, or nothing is missing
            for page in range(first, end, mmap.PAGESIZE):
                mapped(page, mmap.PAGESIZE)
        C.memmove(address, values, len(values))
    _at_fork.clear()
    _free.clear()
    _forked = True
    _lock.release()


os.register_at_fork(before=_before_fork, after_in_parent=_after_fork_in_parent, after_in_child=_after_fork_in_child)
