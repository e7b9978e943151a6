"""Products with an edge of hundreds of millions, more than one launch holds: every variant, checked where
the pieces end."""
import ctypes

import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download

pytestmark = pytest.mark.gpu

LONG = (1 << 28) + 5
# the variant and its error relative to sum |a||b|: roundings of 2^-24, 2^-9 (twice), 2^-17 (twice), 2^-4 (twice)
VARIANTS = [(capi.GEMM_FP32, 2.0 ** -22), (capi.GEMM_BF16, 2.0 ** -7), (capi.GEMM_BF16X3, 2.0 ** -15), (capi.GEMM_FP8, 2.0 ** -2)]


def window(T, buf, at, n):
    out = np.empty(n, np.float32)
    capi.check(capi.lib.cs_memcpy_dtoh(T.stream, out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(buf.ptr + 4 * at),
                                       out.nbytes))
    return out


@pytest.mark.parametrize("variant,bound", VARIANTS)
@pytest.mark.parametrize("tall", [False, True])
def test_long_edge(gpu_tensors, variant, bound, tall):
    T = gpu_tensors
    short, K, n = 2, 2, LONG
    big, small, c = alloc(T, n * K), alloc(T, short * K), alloc(T, n * short)
    for buf, count, seed in ((big, n * K, 1), (small, short * K, 2)):
        capi.check(capi.lib.cs_fill_uniform(T.stream, buf.ptr, count, seed, 0.5, 1.0))
    s = download(T, small, short * K).astype(np.float64)
    if tall:
        args = (n, short, K, big.ptr, K, small.ptr, short, c.ptr, short)
    else:
        args = (short, n, K, small.ptr, K, big.ptr, n, c.ptr, n)
    capi.check(capi.lib.cs_gemm(T.stream, variant, *args))
    w = 4096
    for at in [0, n - w] + [p * (1 << 26) - w // 2 for p in (1, 2, 3, 4)]:
        at = min(at, n - w)
        if tall:
            want = window(T, big, at * K, w * K).astype(np.float64).reshape(w, K) @ s.reshape(K, short)
            got = window(T, c, at * short, w * short).reshape(w, short)
        else:
            want = s.reshape(short, K) @ np.stack([window(T, big, k * n + at, w) for k in range(K)]).astype(np.float64)
            got = np.stack([window(T, c, r * n + at, w) for r in range(short)])
        assert np.all(np.abs(got - want) <= bound * want)
    for b in (big, small, c):
        b.release()
