"""Column sums of fewer rows than a workgroup has row lanes: up to 1024 columns per workgroup."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("cols", [3, 1023, 1026, 65536 * 8 + 5, 1 << 20, (1 << 20) + 1])
def test_few_rows(gpu_tensors, rows, cols):
    T = gpu_tensors
    x = inputs.uniform(rows * cols, 4091).reshape(rows, cols)
    xb, out = upload(T, x), upload(T, np.full(cols + 8, 7.0, np.float32))
    capi.check(capi.lib.cs_reduce_cols(T.stream, xb.ptr, rows, cols, out.ptr))
    got = download(T, out, cols + 8)
    assert np.all(got[cols:] == 7.0)
    want = x.astype(np.float64).sum(axis=0)
    assert np.all(np.abs(got[:cols] - want) <= 4 * np.finfo(np.float32).eps * np.abs(x.astype(np.float64)).sum(axis=0))
    xb.release()
    out.release()
