"""Column sums at the edges of their launch plan: threads across, row lanes, slices and the group of
columns that overlaps the one before."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])  # floats between the buffer's start and the matrix
@pytest.mark.parametrize("shape", [(1, 1), (9000, 1), (70000, 2), (513, 3), (7, 4), (4097, 5), (65, 63), (129, 64),
                                   (1025, 66), (8200, 77), (1024, 255), (1025, 257), (33, 1027), (300, 16386),
                                   (2, 70001), (20011, 131)])
def test_cols_plan_edges(gpu_tensors, shape, shift):
    T = gpu_tensors
    rows, cols = shape
    a = inputs.heavy_tails(inputs.normal(rows * cols, 41), 42).reshape(shape)
    b = upload(T, np.concatenate([np.zeros(shift, np.float32), a.ravel()]))
    guard = 3  # floats after the result that must stay
    out = upload(T, np.full(cols + guard, 7.0, np.float32))
    capi.check(capi.lib.cs_reduce_cols(T.stream, b.ptr + 4 * shift, rows, cols, out.ptr))
    got = download(T, out, cols + guard)
    exact = a.astype(np.float64).sum(axis=0)
    assert np.all(np.abs(got[:cols] - exact) <= 4 * fp64.EPS32 * np.abs(a).astype(np.float64).sum(axis=0))
    assert np.all(got[cols:] == 7.0)
    for h in (b, out):
        h.release()


@pytest.mark.parametrize("shape", [(5, 3), (300, 6), (9000, 10)])
def test_cols_of_special_values(gpu_tensors, shape):
    T = gpu_tensors
    a = np.ones(shape, np.float32)
    a[-1, -1] = np.nan
    a[0, 0] = np.inf
    a[shape[0] // 2, 1] = -np.inf
    with np.errstate(over="ignore"):
        want = a.sum(0, dtype=np.float32)
    assert np.array_equal(T.Tensor(a).colSum().flatArray(), want, equal_nan=True)
