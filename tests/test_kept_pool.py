"""The workspace the library keeps between static queries (kept_pool.h), over a
small memory on the CPU: a kept buffer never makes an allocation fail that
would fit without it, a call that could be served once can be served again,
and nothing stays without a holder (a mesh)."""
import ctypes as C
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MB = 1 << 20


@pytest.fixture()
def pool():
    L = C.CDLL(os.environ.get("CCD_EMU", os.path.join(HERE, "emu", "libccd_emu.so")))
    i64, vp = C.c_int64, C.c_void_p
    L.emu_pool_reset.argtypes = [i64]
    L.emu_pool_used.restype = i64
    L.emu_pool_kept.restype = i64
    L.emu_pool_alloc.argtypes = [i64, C.POINTER(vp)]
    L.emu_pool_free.argtypes = [vp]
    L.emu_pool_take.argtypes = [C.c_int, i64, C.POINTER(vp), C.POINTER(i64)]
    L.emu_pool_give.argtypes = [C.c_int, vp, i64, C.c_int]
    L.emu_pool_reset(1000 * MB)
    L.emu_pool_hold()
    yield L
    L.emu_pool_release()
    assert L.emu_pool_used() == 0


def call(L, n, idle=1, dev=0):
    """One static query: takes n MB of workspace and hands it back."""
    p, b = C.c_void_p(), C.c_int64()
    rc = L.emu_pool_take(dev, n * MB, C.byref(p), C.byref(b))
    if rc == 0:
        assert p.value and b.value >= n * MB
        L.emu_pool_give(dev, p, b, idle)
    return rc


def kept(L, dev=0):
    return L.emu_pool_kept(dev) // MB


def test_buffer_is_kept_and_reused(pool):
    assert call(pool, 200) == 0 and kept(pool) == 200
    assert call(pool, 50) == 0 and kept(pool) == 200
    assert call(pool, 300) == 0 and kept(pool) == 300
    assert pool.emu_pool_used() == 300 * MB
    assert call(pool, 100, idle=0) == 0 and kept(pool) == 0   # work in flight: not kept
    assert call(pool, 600) == 0 and kept(pool) == 0           # larger than what is kept


def test_larger_workspace_replaces_the_kept_one(pool):
    """400 MB are kept and 600 free: a call for 700 MB fits only without them."""
    assert call(pool, 400) == 0 and kept(pool) == 400
    assert call(pool, 700) == 0
    assert kept(pool) == 0 and pool.emu_pool_used() == 0


def test_other_allocations_get_the_kept_memory(pool):
    """400 MB are kept on one device and 100 on another, 500 are free."""
    assert call(pool, 400) == 0 and call(pool, 100, dev=3) == 0
    p = C.c_void_p()
    assert pool.emu_pool_alloc(450 * MB, C.byref(p)) == 0
    pool.emu_pool_free(p)
    assert kept(pool) == 400 and kept(pool, 3) == 100   # it fitted beside them
    assert pool.emu_pool_alloc(900 * MB, C.byref(p)) == 0
    assert kept(pool) == 0 and kept(pool, 3) == 0
    q = C.c_void_p()
    assert pool.emu_pool_alloc(200 * MB, C.byref(q)) != 0   # more than there is
    pool.emu_pool_free(p)


def test_kept_memory_counts_as_free(pool):
    """A quarter of what is free, asked for twice: the kept buffer is part of it."""
    total = 1000 * MB
    for _ in range(3):
        free = total - pool.emu_pool_used() + pool.emu_pool_kept(0)
        assert free == total
        assert call(pool, free // 4 // MB) == 0
        assert kept(pool) == 250


def test_nothing_is_kept_without_a_mesh(pool):
    assert call(pool, 300) == 0 and kept(pool) == 300
    pool.emu_pool_hold()
    pool.emu_pool_release()
    assert kept(pool) == 300
    pool.emu_pool_release()
    assert kept(pool) == 0 and pool.emu_pool_used() == 0
    assert call(pool, 300) == 0 and kept(pool) == 0
    pool.emu_pool_hold()


@pytest.mark.parametrize("copies", [0, 1, 2, 3, 100])
def test_host_task_runs_once_and_throws_nothing(copies):
    """The task beside a device build runs in place when its thread cannot be
    made, also for want of memory: nothing is thrown at the C entry."""
    L = C.CDLL(os.environ.get("CCD_EMU", os.path.join(HERE, "emu", "libccd_emu.so")))
    assert L.emu_host_task(copies) == 1
