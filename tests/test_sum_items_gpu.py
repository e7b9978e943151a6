"""Vectors per thread of fused sums: one workgroup where four make it, two from 2^22 elements whatever the
functions, and sums within the reductions' bound."""
import ctypes
import re

import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu
lib = capi.lib


@pytest.mark.parametrize("n,items", [(1024, 1), (1028, 2), (4096, 4), (4100, 1), (1 << 22, 2), ((1 << 22) + 3, 2)])
@pytest.mark.parametrize("function", ["exp", "abs"])
def test_items_of_sums(gpu_tensors, n, items, function):
    T = gpu_tensors
    t = T.Tensor.fill(0.0, (n,)).nonInline
    h, leaves = T.compile_sum(getattr(T.Tensor, function)(t).closure, (n,))
    src = ctypes.c_char_p()
    capi.check(lib.cs_fused_source(h, ctypes.byref(src)))
    assert re.search(r"unsigned q\[%d\]" % items, src.value.decode())
    a = inputs.uniform(n, 17)
    x, out, out64 = upload(T, a), alloc(T, 1), alloc(T, 1, np.float64)
    ptrs = (ctypes.c_void_p * 1)(x.ptr)
    capi.check(lib.cs_fused_sum(T.stream, h, ptrs, 1, out.ptr, out64.ptr))
    values = np.exp(a.astype(np.float64)) if function == "exp" else np.abs(a.astype(np.float64))
    # each value within 2 ulp, the compensated sum within one rounding of each block's partial
    assert abs(download(T, out64, 1, np.float64)[0] - values.sum()) <= 3 * 2.0 ** -23 * values.sum()
    lib.cs_fused_release(h)
    for b in (x, out, out64):
        b.release()
