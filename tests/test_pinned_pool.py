"""The binding's pool of pinned result memory, with an allocator in ordinary
memory: blocks are reused only after their last array is gone, the two limits
hold, and threads may take and drop arrays at once."""
import ctypes as C
import gc
import threading

import numpy as np
import pytest


class FakeLib:
    """nes_host_alloc / nes_host_free on ctypes buffers."""

    def __init__(self, fail=False):
        self.live, self.freed, self.fail = {}, 0, fail

    def nes_host_alloc(self, n, out):
        if self.fail:
            return -12
        b = (C.c_uint8 * n)()
        self.live[C.addressof(b)] = b
        out._obj.value = C.addressof(b)
        return 0

    def nes_host_free(self, p):
        del self.live[p]
        self.freed += 1
        return 0


@pytest.fixture
def pool(monkeypatch):
    import nes_amd as N
    fake = FakeLib()
    monkeypatch.setattr(N, "_lib", fake)
    p = N._PinnedPool()
    monkeypatch.setattr(N, "_pinned", p)
    yield N, p, fake
    gc.collect()


def test_blocks_return_with_their_last_array(pool):
    N, p, fake = pool
    a = N._out_array((100, 50), np.float32)
    addr = a.ctypes.data
    a[:] = 3.0
    part = a[10:20, ::7]          # a view keeps the block
    del a
    gc.collect()
    b = N._out_array((100, 50), np.float32)
    assert b.ctypes.data != addr and (part == 3.0).all()
    del part
    gc.collect()
    c = N._out_array((99, 50), np.float32)  # same size class
    assert c.ctypes.data == addr and len(fake.live) == 2
    assert b.flags.writeable and b.flags.c_contiguous


def test_limits(pool):
    N, p, fake = pool
    p.LIMIT, p.KEEP = 4 * 4096, 4096
    held = [N._out_array((4096,), np.uint8) for _ in range(6)]
    assert p.allocated == 4 * 4096 and len(fake.live) == 4  # the others are ordinary arrays
    del held
    gc.collect()
    assert p.allocated == p.unused == 4096 and fake.freed == 3
    fake.fail = True
    assert N._out_array((10000,), np.uint8).shape == (10000,)  # no pinned memory: an ordinary array
    assert p.allocated == 4096
    assert N._out_array((0, 3), np.uint8).size == 0


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 307200 * 3, 12197850 * 4])
def test_size_classes(pool, n):
    N, p, _ = pool
    s = p.size_class(n)
    assert s >= n and s % 4096 == 0 and s <= max(4096, n + max(4096, n // 4))
    assert p.size_class(s) == s


def test_threads(pool):
    N, p, fake = pool
    bad = []

    def work(k):
        for i in range(200):
            a = N._out_array((500 + i,), np.int32)
            a[:] = k
            b = N._out_array((500 + i,), np.int32)
            b[:] = -k
            if not (a == k).all():
                bad.append((k, i))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(1, 7)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    gc.collect()
    assert not bad and p.unused == p.allocated <= p.KEEP


class DontForkLib(FakeLib):
    """Memory that a forked child does not inherit, as pinned memory is."""

    def nes_host_alloc(self, n, out):
        import mmap
        m = mmap.mmap(-1, n)
        m.madvise(mmap.MADV_DONTFORK)
        out._obj.value = C.addressof(C.c_char.from_buffer(m))
        self.live[out._obj.value] = m
        return 0


def in_child(f):
    """Exit code (or minus the signal) of a forked child that runs f."""
    import os
    pid = os.fork()
    if pid == 0:
        code = 1
        try:
            code = 0 if f() else 2
        finally:
            os._exit(code)
    return os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1])


def test_forked_children_keep_their_arrays(pool, monkeypatch):
    """A child forked between calls reads the values that arrays had at the
    fork, may write and drop them and take more, and forks in turn; nothing of
    it reaches the parent's arrays or its pool."""
    N, p, _ = pool
    monkeypatch.setattr(N, "_lib", DontForkLib())
    arrays = [N._out_array((n, 3), np.float32) for n in (1, 1000, 70000)]
    for i, a in enumerate(arrays):
        a[:] = i + 1.5
    part = arrays[1][5:9]
    dropped = N._out_array((50,), np.int32)
    del dropped                       # a free block stays the parent's
    gc.collect()

    def child():
        ok = all((a == i + 1.5).all() for i, a in enumerate(arrays))
        arrays[0][:] = 9.0
        more = N._out_array((50,), np.int32)
        more[:] = 7
        ok = ok and in_child(lambda: (arrays[0] == 9.0).all() and (arrays[2] == 3.5).all()) == 0
        arrays.clear()
        gc.collect()
        return ok and (part == 2.5).all() and (more == 7).all()

    allocated = p.allocated
    for _ in range(2):
        assert in_child(child) == 0
    assert all((a == i + 1.5).all() for i, a in enumerate(arrays)) and (part == 2.5).all()
    assert p.allocated == allocated and p.unused == 4096 and len(p.live) == 3
    again = N._out_array((50,), np.int32)
    assert p.unused == 0 and len(p.live) == 4
    del again
