"""FP32 products on the three-part path of the values that lose most by the products of parts it leaves out,
and of values whose products FP32 holds exactly."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload

pytestmark = pytest.mark.gpu

WORST = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)  # parts 1, 2^-8 and -2^-17


def product(T, a, b):
    (M, K), N = a.shape, b.shape[1]
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    c = download(T, bc, M * N).reshape(M, N)
    for h in (ba, bb, bc):
        h.release()
    return c


@pytest.mark.parametrize("mnk", [(4096, 4096, 64), (2048, 2048, 1000), (1024, 1024, 4096)])
@pytest.mark.parametrize("scaled", [False, True])
def test_most_left_out(gpu_tensors, mnk, scaled):
    M, N, K = mnk
    rng = np.random.default_rng(K)
    powers = (lambda *s: np.exp2(rng.integers(-3, 4, s))) if scaled else (lambda *s: np.ones(s))
    a, b = (WORST * powers(M, K)).astype(np.float32), (WORST * powers(K, N)).astype(np.float32)
    rows = np.arange(0, M, 53)
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    # the products left out, and six roundings to a partial sum of at most |C| for each 16 of K, half of
    # |C| on the way
    bound = (1 + 6 * K / 16 / 2) * 2.0 ** -24
    assert np.all(np.abs(product(gpu_tensors, a, b)[rows] - want) <= bound * want)


def test_whole_numbers_are_exact(gpu_tensors):
    """Products of 17-bit by 5-bit whole numbers, and their sums, are whole numbers below 2^24."""
    M, N, K = 3000, 3000, 48
    rng = np.random.default_rng(5)
    a = np.zeros((M, K), np.float32)
    a[:, :7] = rng.integers(1, 1 << 17, (M, 7))
    a[:, 7:] = rng.integers(-8, 9, (M, K - 7))
    b = rng.integers(-15, 16, (K, N)).astype(np.float32)
    assert np.array_equal(product(gpu_tensors, a, b), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))
