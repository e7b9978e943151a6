"""Who waits for the last users of a released block: the streams and the host that are handed its
memory, and nobody for later work."""
import ctypes

import numpy as np
import pytest

from compute import Tensors
from compute import _capi as capi

pytestmark = pytest.mark.gpu
lib = capi.lib
N = 1 << 24


def new_stream(T):
    st = ctypes.c_void_p()
    capi.check(lib.cs_stream_create(T.device, ctypes.byref(st)))
    return st.value


def block_at(where, allocate):
    """Allocates N floats until they lie at `where` (allocations take the lowest free block)."""
    handles = []
    for _ in range(8):
        h, p = ctypes.c_void_p(), ctypes.c_void_p()
        capi.check(allocate(N * 4, ctypes.byref(h)))
        capi.check(lib.cs_buffer_device_ptr(h.value, ctypes.byref(p)))
        handles.append(h)
        if p.value == where:
            return handles
    raise AssertionError("the released block was not handed out")


def queue_copies(T, dst, src, count):
    for _ in range(count):
        capi.check(lib.cs_memcpy_dtod(T.stream, dst, src, N * 4))


def recorded(T):
    ev = ctypes.c_void_p()
    capi.check(lib.cs_event_record(T.stream, ctypes.byref(ev)))
    return ev


def complete(ev):
    done = ctypes.c_int()
    capi.check(lib.cs_event_query(ev, ctypes.byref(done)))
    return done.value


@pytest.mark.parametrize("others", [0, 1, 2])  # streams created between the release and the one that gets the block
def test_any_new_stream_waits(others):
    with Tensors(0) as T:
        src = T.Tensor.random((N,), seed=3).doBuffer()
        want, kept, where = src.to_numpy(N), T._alloc(N * 4), src.ptr
        queue_copies(T, kept.ptr, where, 20)
        src.release()
        streams = [new_stream(T) for _ in range(others + 1)]
        handles = block_at(where, lambda n, h: lib.cs_buffer_alloc_on(streams[-1], n, h))
        capi.check(lib.cs_fill_uniform(streams[-1], where, N, 1, 5.0, 6.0))
        capi.check(lib.cs_stream_synchronize(streams[-1]))
        assert np.array_equal(kept.to_numpy(N), want)
        for h in handles:
            capi.check(lib.cs_buffer_release(h.value))
        kept.release()
        for st in streams:
            capi.check(lib.cs_stream_destroy(st))


def test_host_allocation_waits_for_the_last_users():
    """cs_buffer_alloc returns a block only when it is free for any stream, also where a stream-ordered
    allocation has handed the block back before."""
    with Tensors(0) as T:
        src, kept = T._alloc(N * 4), T._alloc(N * 4)
        where = src.ptr
        queue_copies(T, kept.ptr, where, 100)
        used = recorded(T)
        src.release()
        T._alloc(256).release()  # hands the block back
        handles = block_at(where, lambda n, h: lib.cs_buffer_alloc(T.device, n, h))
        assert complete(used)
        for h in handles:
            capi.check(lib.cs_buffer_release(h.value))
        capi.check(lib.cs_event_release(used))
        kept.release()


def test_host_allocation_does_not_wait_for_later_work():
    with Tensors(0) as T:
        src, kept, free = T._alloc(N * 4), T._alloc(N * 4), T._alloc(N * 4)
        where = free.ptr
        T.synchronize()
        free.release()
        queue_copies(T, kept.ptr, src.ptr, 2000)
        later = recorded(T)
        handles = block_at(where, lambda n, h: lib.cs_buffer_alloc(T.device, n, h))
        assert not complete(later)
        T.synchronize()
        for h in handles:
            capi.check(lib.cs_buffer_release(h.value))
        capi.check(lib.cs_event_release(later))
        src.release()
        kept.release()


def test_finished_releases_leave_the_bytes_in_use():
    """A block whose users are done no longer counts as in use at the next release."""
    with Tensors(0) as T:
        big, small = T._alloc(N * 4), T._alloc(256)
        before = T.info(capi.INFO_ARENA_IN_USE_BYTES)
        big.release()
        T.synchronize()
        small.release()
        assert T.info(capi.INFO_ARENA_IN_USE_BYTES) <= before - N * 4
