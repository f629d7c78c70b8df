"""The pool of blocks that results lie in: what it keeps, gives back and refuses, over a stand-in for the allocator."""
import gc
import threading

import numpy as np

from axonml_amd.quant import _HostBlocks


class Lib:
    """Ordinary memory by address."""

    def __init__(self):
        self.blocks, self.refuse = {}, False

    def axq_host_alloc(self, handle, size, p):
        if self.refuse:
            return -21
        a = np.zeros(size, np.uint8)
        p._obj.value = a.ctypes.data
        self.blocks[a.ctypes.data] = a
        return 0

    def axq_host_free(self, ptr):
        del self.blocks[ptr]


class Ctx:
    def __init__(self):
        self.lib, self.handle = Lib(), 1


def test_blocks_live_as_long_as_their_arrays():
    ctx = Ctx()
    pool = _HostBlocks(ctx)
    a = pool.array((3, 1000))
    assert a.shape == (3, 1000) and a.dtype == np.float32 and a.flags.writeable and a.flags.c_contiguous
    row, at = a[1], a.ctypes.data
    row[:] = 7
    del a
    assert pool.kept == 0 and pool.array((3, 1000)).ctypes.data != at  # a view still lies in it
    assert (row == 7).all()
    del row
    gc.collect()
    assert pool.kept == 2 * 12288 and {pool.take(12288), pool.take(12288)} == set(ctx.lib.blocks)


def test_what_is_kept_and_handed_out_is_bounded():
    ctx = Ctx()
    pool = _HostBlocks(ctx)
    pool.KEEP, pool.MOST = 3 * 4096, 5 * 4096
    held = [pool.array((1024,)) for _ in range(7)]
    assert len(ctx.lib.blocks) == 5 and pool.total == 5 * 4096
    del held
    gc.collect()
    assert len(ctx.lib.blocks) == 3 and pool.kept == pool.total == 3 * 4096
    big = pool.array((4, 1024))  # needs what is kept to go
    assert len(ctx.lib.blocks) == 1 and pool.total == 4 * 4096
    pool.close()
    del big
    gc.collect()
    assert not ctx.lib.blocks and pool.total == 0
    assert pool.array((5,)).shape == (5,) and not ctx.lib.blocks
    assert pool.array((0, 5)).shape == (0, 5)


def test_a_block_that_comes_back_while_others_go():
    """The collector may run anywhere, here in the middle of giving blocks back."""
    ctx = Ctx()
    pool = _HostBlocks(ctx)
    other = [pool.array((3000,))]
    held = [pool.array((1000,)), pool.array((2000,))]
    free = ctx.lib.axq_host_free

    def free_and_collect(ptr):
        free(ptr)
        other.clear()
    del held
    ctx.lib.axq_host_free = free_and_collect
    pool.MOST = pool.total
    big = pool.array((1024,) * 2)  # more than there may be: what is idle goes
    assert big.shape == (1024, 1024) and pool.total == pool.kept == 12288
    ctx.lib.axq_host_free = free
    pool.close()
    assert not ctx.lib.blocks and pool.total == pool.kept == 0


def test_no_page_locked_memory():
    ctx = Ctx()
    ctx.lib.refuse = True
    assert _HostBlocks(ctx).array((2, 3)).shape == (2, 3)


def test_threads():
    ctx = Ctx()
    pool = _HostBlocks(ctx)
    pool.KEEP = 4 * 4096

    def work(seed):
        rng = np.random.default_rng(seed)
        held = []
        for i in range(300):
            a = pool.array((int(rng.integers(1, 3000)),))
            a[:] = seed * 1000 + i
            held.append((a, seed * 1000 + i))
            if len(held) > 5:
                b, v = held.pop(int(rng.integers(0, 6)))
                assert (b == v).all()
    threads = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gc.collect()
    assert pool.total == pool.kept <= 4 * 4096 and len(ctx.lib.blocks) == sum(map(len, pool.idle.values()))
