"""The pool of memory that a step's logits stand on (krasis_amd.serve_store._RowPool), on the CPU: a stand-in for the library hands out ordinary pages."""
import mmap

import numpy as np
import pytest

from krasis_amd import serve_store as S


class Lib:
    """kr_serve_rows_alloc / kr_serve_rows_free over anonymous pages; `refuse`: allocations fail"""
    def __init__(self):
        self.live, self.asked, self.refuse = {}, 0, False

    def kr_serve_rows_alloc(self, handle, nbytes, out):
        self.asked += 1
        if self.refuse:
            return -3
        m = mmap.mmap(-1, nbytes)
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
