"""Column sums of matrices with about as many groups of columns as CUs, cut into a few slices of rows or a
number of columns to a workgroup that no power of two gives, and of fewer than four columns."""
import ctypes

import numpy as np
import pytest

from compute import Tensors
from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu
lib = capi.lib


def column_sums(T, x, rows, cols, out):
    capi.check(lib.cs_reduce_cols(T.stream, x.ptr, rows, cols, out.ptr))


@pytest.mark.parametrize("shape", [(1025, 32768), (1025, 32769), (1030, 33001), (1100, 44003), (1027, 66000), (1026, 102401),
                                   (1022, 19058), (515, 19661), (1024, 9601),
                                   (1, 3), (84, 3), (85, 3), (86, 3), (5462, 3), (5461, 3), (8192, 2), (8193, 2),
                                   (255, 1), (257, 1), (16384, 1), (16385, 1), (300007, 3)])
def test_slices(gpu_tensors, shape):
    T, (rows, cols) = gpu_tensors, shape
    a = inputs.uniform(rows * cols, 31).reshape(shape)
    x, out = upload(T, a), alloc(T, cols)
    column_sums(T, x, rows, cols, out)
    exact, magnitude = a.sum(0, dtype=np.float64), np.abs(a).sum(0, dtype=np.float64)
    assert np.all(np.abs(download(T, out, cols) - exact) <= 2.0 ** -23 * magnitude)
    x.release()
    out.release()


def test_captured_after_a_wider_one():
    """A wider matrix without slices sizes the scratch for one with slices under capture."""
    with Tensors(0) as T:
        rows, wide, narrow = 1100, 60000, 44000
        x, out = alloc(T, rows * wide), alloc(T, wide)
        capi.check(lib.cs_fill_uniform(T.stream, x.ptr, rows * wide, 3, -1.0, 1.0))
        column_sums(T, x, rows, wide, out)
        g = ctypes.c_void_p()
        capi.check(lib.cs_graph_begin_capture(T.stream))
        try:
            column_sums(T, x, rows, narrow, out)
        finally:
            capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
        capi.check(lib.cs_graph_launch(T.stream, g))
        got = download(T, out, narrow)
        column_sums(T, x, rows, narrow, out)
        assert np.array_equal(got.view(np.uint32), download(T, out, narrow).view(np.uint32))
        lib.cs_graph_release(g)
        x.release()
        out.release()
