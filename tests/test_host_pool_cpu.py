"""HostPool over a device library that counts: when pinned memory is allocated and freed, and by whom."""
import ctypes as C

import numpy as np
import pytest

from gpreempt_amd import capi


class CountingLib:
    def __init__(self):
        self.blocks, self.allocated, self.freed = {}, 0, 0

    def gp_host_alloc_coherent(self, host, dev, n):
        block = (C.c_char * n.value)()
        address = C.addressof(block)
        self.blocks[address] = block
        self.allocated += 1
        host._obj.value = dev._obj.value = address
        return 0

    def gp_host_free(self, p):
        del self.blocks[p.value]
        self.freed += 1
        return 0


@pytest.fixture
def counting(monkeypatch):
    lib = CountingLib()
    monkeypatch.setattr(capi, "lib", lambda: lib)
    return lib


@pytest.mark.parametrize("n", [1, 4000, 100000, 5 << 20, 84 << 20])
def test_a_caller_that_keeps_its_outputs_pays_for_a_few_allocations(counting, n):
    pool, kept = capi.HostPool(), []
    for _ in range(100 if n < 1 << 20 else 12):
        kept.append(pool.empty(n))
    room = -(-n // 4096) * 4096
    assert counting.allocated <= max(4, min(64, (1 << 20) // room))
    assert counting.allocated * n <= capi.HostPool.LIMIT
    assert all(a.nbytes == n and (ptr is None or ptr == a.ctypes.data) for a, ptr in kept)
    assert kept[-1][1] is None and kept[0][1] is not None


@pytest.mark.parametrize("n", [4000, 84 << 20])
def test_a_loop_allocates_twice_and_the_garbage_collector_frees_nothing(counting, n):
    pool = capi.HostPool()
    out = None
    for _ in range(50):
        out, ptr = pool.empty(n)
        assert ptr is not None
    assert counting.allocated == 2 and counting.freed == 0
    many = [pool.empty(n) for _ in range(4)]
    del out, many
    assert counting.freed == 0  # freeing waits for the GPU; an array may die anywhere
    pool.trim(0)
    assert counting.freed == counting.allocated and not counting.blocks
    a, ptr = pool.empty(n)
    assert ptr is not None  # what has been given back may be allocated again
    a[:] = 7
    assert (a == 7).all()


def test_a_new_executor_finds_the_blocks_of_the_last_one(counting):
    pool = capi.HostPool()
    out = pool.empty(84 << 20)
    out = pool.empty(84 << 20)
    pool.trim()  # (the executor goes first, its last output afterwards)
    del out
    pool.trim()
    for _ in range(3):
        assert pool.empty(84 << 20)[1] is not None
        pool.trim()
    assert counting.allocated == 2 and counting.freed == 0


def test_trim_keeps_the_small_blocks(counting):
    pool = capi.HostPool()
    arrays = [pool.empty(n) for n in (4096, 4096, 1 << 20, 100 << 20, 200 << 20)]
    pool.trim(0)
    assert counting.freed == 0  # all of them are in use
    del arrays
    pool.trim()
    assert counting.freed == 1 and pool._idle <= pool.KEEP
    pool.trim()
    assert counting.freed == 1
