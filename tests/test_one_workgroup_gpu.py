"""Reductions around the sizes that one workgroup takes and finishes alone, and blocks of memory that
change hands without an event."""
import ctypes

import numpy as np
import pytest

from compute import Tensors, _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 1023, 1024, 1025, 4095, 4096, 4097, 4100, 8193])
def test_sums_and_maxima(n):
    x = inputs.heavy_tails(inputs.normal(n, 51), 52) if n else np.zeros(0, np.float32)
    exact, bound = x.astype(np.float64).sum(), fp64.sum_bound(x)
    with Tensors(0) as T:
        t = T.Tensor(x)
        b = upload(T, x)
        out, out64 = alloc(T, 2), alloc(T, 2, np.float64)
        capi.check(capi.lib.cs_reduce_sum(T.stream, b.ptr, n, out.ptr, None))
        capi.check(capi.lib.cs_reduce_sum(T.stream, b.ptr, n, None, out64.ptr))
        inline = t + T.Tensor.fill(0.0, (n,))
        f, _ = T.compile_sum(inline.closure, inline.shape)
        leaves = (ctypes.c_void_p * 1)(b.ptr)
        capi.check(capi.lib.cs_fused_sum(T.stream, f, leaves, 1, out.ptr + 4, None))
        capi.check(capi.lib.cs_fused_sum(T.stream, f, leaves, 1, None, out64.ptr + 8))
        s, s64 = download(T, out, 2), download(T, out64, 2, np.float64)
        assert np.all(np.abs(s - exact) <= bound + abs(exact) * 2.0 ** -24)
        assert abs(s64[0] - exact) <= 1e-12 * max(np.abs(x).sum(), 1.0) and abs(s64[1] - exact) <= bound
        assert s[0] == np.float32(s64[0]) and s[1] == np.float32(s64[1])
        if n:
            assert t.maxValue().flatArray()[0] == x.max()
        capi.lib.cs_fused_release(f)
        for h in (b, out, out64):
            h.release()


@pytest.mark.parametrize("shape", [(1, 5000), (1, 30), (3, 20), (128, 8), (129, 8), (4, 1000), (5, 1000)])
def test_row_totals(gpu_tensors, shape):
    T = gpu_tensors
    a = inputs.normal(shape[0] * shape[1], 61).reshape(shape)
    b, tot, tot64 = upload(T, a), alloc(T, 1), alloc(T, 1, np.float64)
    for f in (capi.lib.cs_reduce_rows, capi.lib.cs_reduce_rows_noalloc):
        capi.check(f(T.stream, b.ptr, shape[0], shape[1], None, None, tot.ptr, tot64.ptr))
        exact = a.astype(np.float64).sum()
        assert abs(download(T, tot64, 1, np.float64)[0] - exact) <= 1e-12 * np.abs(a).sum()
        assert download(T, tot, 1)[0] == np.float32(download(T, tot64, 1, np.float64)[0])
    for h in (b, tot, tot64):
        h.release()


def test_released_block_on_a_new_stream():
    """A block released with one stream alive, its work still queued, goes to a stream that is created
    afterwards: the new stream's writes come after that work."""
    n = 1 << 24
    with Tensors(0) as T:
        for k in range(3):
            e = T.Tensor.exp(T.Tensor.random((n,), seed=k)) * T.Tensor.random((n,), seed=k + 9)
            want = e.flatArray()
            src = e.doBuffer()
            kept = T._alloc(n * 4)
            capi.check(capi.lib.cs_memcpy_dtod(T.stream, kept.ptr, src.ptr, n * 4))
            where = src.ptr
            src.release()  # the copy out of it is still queued
            st, handles, ptrs = ctypes.c_void_p(), [], []
            capi.check(capi.lib.cs_stream_create(T.device, ctypes.byref(st)))
            while where not in ptrs and len(ptrs) < 8:  # allocations take the lowest free block
                h, p = ctypes.c_void_p(), ctypes.c_void_p()
                capi.check(capi.lib.cs_buffer_alloc_on(st.value, n * 4, ctypes.byref(h)))
                capi.check(capi.lib.cs_buffer_device_ptr(h.value, ctypes.byref(p)))
                handles.append(h)
                ptrs.append(p.value)
            assert where in ptrs
            capi.check(capi.lib.cs_fill_uniform(st.value, where, n, 1, 5.0, 6.0))
            capi.check(capi.lib.cs_stream_synchronize(st.value))
            assert np.array_equal(kept.to_numpy(n), want)
            for h in handles:
                capi.check(capi.lib.cs_buffer_release(h.value))
            kept.release()
            capi.check(capi.lib.cs_stream_destroy(st.value))
