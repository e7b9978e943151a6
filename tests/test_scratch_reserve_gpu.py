"""A product that needs no scratch itself sizes the stream's for later calls, where memory is left for it:
without room the product still runs, and the scratch that was there stays."""
import ctypes

import numpy as np
import pytest

from compute import _capi as capi
from compute import Tensors
from gpu_util import alloc, download

pytestmark = pytest.mark.gpu
lib = capi.lib


def test_a_product_without_room_for_scratch():
    n = 1 << 26  # its operand copies would take 8 GiB
    with Tensors(0) as T:
        a, b, c = alloc(T, n), alloc(T, 1), alloc(T, n)
        capi.check(lib.cs_fill_uniform(T.stream, a.ptr, n, 5, -1.0, 1.0))
        capi.check(lib.cs_fill_uniform(T.stream, b.ptr, 1, 6, -1.0, 1.0))
        product = lambda m: capi.check(lib.cs_gemm(T.stream, capi.GEMM_FP32, m, 1, 1, a.ptr, 1, b.ptr, 1, c.ptr, 1))  # noqa: E731
        product(1000)  # scratch for small calls
        filler = []
        for size in (64 << 30, 16 << 30, 4 << 30):  # until less than 4 GiB are left
            while True:
                h = ctypes.c_void_p()
                if lib.cs_buffer_alloc(T.device, size, ctypes.byref(h)):
                    break
                filler.append(h)
        try:
            product(n)
            want = download(T, a, n) * download(T, b, 1)
            assert np.array_equal(download(T, c, n), want)
            # the small scratch is still there under capture
            out, g = alloc(T, 1), ctypes.c_void_p()
            capi.check(lib.cs_graph_begin_capture(T.stream))
            capi.check(lib.cs_reduce_sum(T.stream, a.ptr, 1 << 20, out.ptr, None))
            capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
            lib.cs_graph_release(g)
        finally:
            for h in filler:
                capi.check(lib.cs_buffer_release(h.value))
            capi.check(lib.cs_arena_trim(T.device))
        for h in (a, b, c, out):
            h.release()
