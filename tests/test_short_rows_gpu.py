"""Row reductions at the edges of their launch plan: lanes per row, rows per workgroup, the vector
that overlaps the end of a row, and wide rows of few."""
import numpy as np
import pytest

import oracle
from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])  # floats between the buffer's start and the matrix
@pytest.mark.parametrize("shape", [(1, 1), (300, 3), (257, 4), (1000, 7), (129, 32), (129, 33), (65, 77), (64, 129),
                                   (33, 258), (17, 515), (9, 1023), (5, 1025), (4, 2048), (3, 2049), (256, 8192),
                                   (257, 8195), (1100000, 2)])
def test_rows_plan_edges(gpu_tensors, shape, shift):
    T = gpu_tensors
    rows, cols = shape
    a = inputs.heavy_tails(inputs.normal(rows * cols, 31), 32).reshape(shape)
    b = upload(T, np.concatenate([np.zeros(shift, np.float32), a.ravel()]))
    rs, rm, tot, tot64 = alloc(T, rows), alloc(T, rows), alloc(T, 1), alloc(T, 1, np.float64)
    capi.check(capi.lib.cs_reduce_rows(T.stream, b.ptr + 4 * shift, rows, cols, rs.ptr, rm.ptr, tot.ptr, tot64.ptr))
    s64, m64, sa, total = oracle.row_stats64(a)
    assert np.all(np.abs(download(T, rs, rows) - s64) <= 4 * fp64.EPS32 * sa)
    assert np.array_equal(download(T, rm, rows), m64)
    assert abs(float(download(T, tot, 1)[0]) - total) <= 4 * fp64.EPS32 * sa.sum()
    assert abs(float(download(T, tot64, 1, np.float64)[0]) - total) <= 1e-12 * sa.sum()
    for h in (b, rs, rm, tot, tot64):
        h.release()


@pytest.mark.parametrize("cols", [3, 5, 77, 1026])
def test_short_rows_of_special_values(gpu_tensors, cols):
    """NaN is ignored by the maximum and makes the sum NaN; infinities stay; a row of the lowest
    finite value has it as its maximum."""
    T = gpu_tensors
    a = np.ones((5, cols), np.float32)
    a[0, -1] = np.nan
    a[1, :] = np.nan
    a[2, cols // 2] = np.inf
    a[3, 0] = -np.inf
    a[4, :] = np.finfo(np.float32).min
    t = T.Tensor(a)
    with np.errstate(over="ignore"):
        want = a.sum(1, dtype=np.float32)
    assert np.array_equal(t.rowSum().flatArray(), want, equal_nan=True)
    want_max = np.array([1.0, np.nan, np.inf, 1.0, np.finfo(np.float32).min], np.float32)
    assert np.array_equal(t.rowMax().flatArray(), want_max, equal_nan=True)
