"""An eager call sizes the stream's scratch for captured calls of up to its size, whichever kernels they take."""
import ctypes

import numpy as np
import pytest

from compute import Tensors
from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu
lib = capi.lib


def replay(T, call):
    g = ctypes.c_void_p()
    capi.check(lib.cs_graph_begin_capture(T.stream))
    try:
        call()
    finally:
        capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
    for _ in range(3):
        capi.check(lib.cs_graph_launch(T.stream, g))
    T.synchronize()
    lib.cs_graph_release(g)


def test_fewer_but_longer_rows():
    """Short rows share partials, long ones have one each."""
    with Tensors(0) as T:
        many, few, cols = 400000, 300000, 2052
        x, total = alloc(T, few * cols), alloc(T, 1, np.float64)
        capi.check(lib.cs_fill_uniform(T.stream, x.ptr, few * cols, 3, -1.0, 1.0))
        rows = lambda r, c: capi.check(lib.cs_reduce_rows(T.stream, x.ptr, r, c, None, None, None, total.ptr))  # noqa: E731
        rows(many, 8)
        replay(T, lambda: rows(few, cols))
        got = download(T, total, 1, np.float64)[0]
        rows(few, cols)
        assert got == download(T, total, 1, np.float64)[0]
        x.release()
        total.release()


@pytest.mark.parametrize("variant", [capi.GEMM_FP32, capi.GEMM_BF16, capi.GEMM_BF16X3, capi.GEMM_FP8])
@pytest.mark.parametrize("eager,captured", [((300, 300, 300), (257, 257, 300)), ((1100, 1100, 1000), (1030, 1025, 1000)),
                                            ((2100, 2100, 900), (2049, 2049, 900)), ((3000, 300, 500), (2000, 300, 500))])
def test_result_over_an_operand(variant, eager, captured):
    """A product into its own operand copies both, also where the eager one needed no copies."""
    with Tensors(0) as T:
        m, n, k = eager
        a, b, c = (upload(T, inputs.uniform(s, 80 + i)) for i, s in enumerate((m * k, k * n, m * n)))
        capi.check(lib.cs_gemm(T.stream, variant, m, n, k, a.ptr, k, b.ptr, n, c.ptr, n))
        m, n, k = captured
        ld = max(n, k)
        x = inputs.uniform(m * ld, 90)
        over = upload(T, x)
        replay_input = lambda: capi.check(lib.cs_memcpy_htod(T.stream, ctypes.c_void_p(over.ptr),  # noqa: E731
                                                             x.ctypes.data_as(ctypes.c_void_p), x.nbytes))
        product = lambda: capi.check(lib.cs_gemm(T.stream, variant, m, n, k, over.ptr, ld, b.ptr, n, over.ptr, ld))  # noqa: E731
        g = ctypes.c_void_p()
        capi.check(lib.cs_graph_begin_capture(T.stream))
        try:
            product()
        finally:
            capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
        results = []
        for launch in (lambda: capi.check(lib.cs_graph_launch(T.stream, g)), product) * 2:
            replay_input()
            launch()
            results.append(download(T, over, m * ld))
        for r in results[1:]:
            assert np.array_equal(r.view(np.uint32), results[0].view(np.uint32))
        lib.cs_graph_release(g)
        for h in (a, b, c, over):
            h.release()
