"""The pool of memory that a step's logits stand on (krasis_amd.serve_store._RowPool), on the CPU: a stand-in for the library hands out ordinary pages."""
import gc
import mmap
import os
import subprocess
import sys

import numpy as np
import pytest

from krasis_amd import serve_store as S


class Lib:
    """kr_serve_rows_alloc / kr_serve_rows_free over anonymous pages that, as a device's, a forked child does not get; `refuse`: allocations fail"""
    def __init__(self):
        self.live, self.asked, self.refuse = {}, 0, False

    def kr_serve_rows_alloc(self, handle, nbytes, out):
        self.asked += 1
        if self.refuse:
            return -3
        m = mmap.mmap(-1, nbytes)
        m.madvise(mmap.MADV_DONTFORK)
        at = np.frombuffer(m, np.uint8).ctypes.data
        self.live[at] = m
        out._obj.value = at
        return 0

    def kr_serve_rows_free(self, ptr):
        return 0 if self.live.pop(ptr.value, None) is not None else -1

    def pinned(self):
        return sum(len(m) for m in self.live.values())


def test_refused_memory_means_the_copy():
    lib = Lib(); pool = S._RowPool(lib)
    a = pool.take(None, 3, 20000)
    a[:] = 7
    lib.refuse = True
    held = [pool.take(None, 1, 20000) for _ in range(40)]       # another size of block: nothing of it is there
    assert held == [None] * 40
    assert lib.asked <= 1 + 1 + 40 // pool.RETRY                 # refused memory is not asked for at every step
    assert pool.take(None, 3, 20000) is not None                 # blocks that are there still serve
    assert (a == 7).all()
    lib.refuse = False
    got = [pool.take(None, 1, 20000) for _ in range(pool.RETRY + 1)]
    assert got[-1] is not None and got[-1].shape == (1, 20000)


def test_growing_batches_are_not_shut_out():
    """one row of 151936 logits to sixteen, every size for a while: blocks of sizes that are no longer used make room"""
    lib = Lib(); pool = S._RowPool(lib); V = 151936
    for rows in (1, 2, 5, 13, 16, 27, 1):
        for _ in range(pool.RETRY + 2):
            last = pool.take(None, rows, V)
            if last is not None:
                last[0, 0] = last[-1, -1] = rows
        assert last is not None and last.shape == (rows, V), rows
        assert pool._bytes == lib.pinned() <= pool.MOST


def test_room_is_not_made_of_what_is_held_and_not_at_every_step():
    lib = Lib(); pool = S._RowPool(lib); V = 151936
    held = [pool.take(None, 5, V) for _ in range(32)]            # 32 blocks of 4 MB
    for i, h in enumerate(held):
        h[:] = i
    asked = lib.asked
    assert all(pool.take(None, 13, V) is None for _ in range(3 * pool.RETRY)) and lib.asked == asked
    assert all((h == i).all() for i, h in enumerate(held))
    held = held[:1]                                              # the first slab keeps one block
    for _ in range(2 * pool.RETRY + 2):                          # sizes in turn
        a, b = pool.take(None, 13, V), pool.take(None, 5, V)
    assert a is not None and b is not None and lib.asked - asked <= 4
    assert (held[0] == 0).all()


def test_the_interpreter_ends_quietly():
    """a store, its pool and arrays that nobody closed: nothing is said at the end, and nothing is called into a library that may be down"""
    code = ("import sys; sys.path.insert(0, '.')\n"
            "from tests.test_serve_rows_pool import Lib, S\n"
            "lib = Lib(); pool = S._RowPool(lib); keep = pool.take(None, 3, 20000)\n"
            "sys.modules['anchor'] = S; S.anchor = (pool, keep)\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stderr == "", r.stderr


def test_arrays_live_on_in_a_forked_child():
    lib = Lib(); pool = S._RowPool(lib)
    a, b, gone = pool.take(None, 3, 20001), pool.take(None, 3, 20001), pool.take(None, 3, 20001)
    a[:] = np.arange(a.size).reshape(a.shape); b[:] = -1
    view = b[2, 5:]
    del gone, b
    want = a.copy()
    pid = os.fork()
    if pid == 0:
        ok = np.array_equal(a, want) and bool((view == -1).all())
        a[:] = 5; view[:] = 6                                    # the child's own from here on
        del a, view; gc.collect()
        os._exit(0 if ok and len(lib.live) == 1 and pool.take(None, 3, 20001) is not None else 1)      # (a stand-in's new slab; the parent's blocks are not the child's)
    assert os.waitpid(pid, 0)[1] == 0
    assert np.array_equal(a, want) and (view == -1).all()
    del a, view; gc.collect()
    assert pool._bytes == lib.pinned()
    for _ in range(40):
        assert pool.take(None, 3, 20001) is not None             # the parent's blocks still come round
    assert pool._bytes == lib.pinned()
