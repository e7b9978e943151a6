"""FP32 products large enough for the three-part BF16 path: accuracy over K and scales, remainders, and
the values that its split cannot hold."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs

pytestmark = pytest.mark.gpu


def _gemm(T, a, b, lda=None, ldb=None, ldc=None):
    M, K = a.shape
    N = b.shape[1]
    lda, ldb, ldc = lda or K, ldb or N, ldc or N
    pa, pb = np.zeros((M, lda), np.float32), np.zeros((K, ldb), np.float32)
    pa[:, :K], pb[:, :N] = a, b
    ba, bb, bc = upload(T, pa), upload(T, pb), upload(T, np.full(M * ldc, 7.0, np.float32))
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, lda, bb.ptr, ldb, bc.ptr, ldc))
    c = download(T, bc, M * ldc).reshape(M, ldc)
    for h in (ba, bb, bc):
        h.release()
    assert np.all(c[:, N:] == 7.0)
    return c[:, :N].copy()


@pytest.mark.parametrize("mnk", [(3000, 3001, 300), (4096, 4096, 129), (3841, 2905, 1024), (2817, 4000, 271), (9000, 1200, 500)])
def test_shapes(gpu_tensors, mnk):
    """The bound of the FP32 variant, K tails and tiles that end in the matrix among them; rows spread
    over the matrix are checked in full."""
    M, N, K = mnk
    a, b = inputs.uniform(M * K, 4041).reshape(M, K), inputs.uniform(K * N, 4042).reshape(K, N)
    c = _gemm(gpu_tensors, a, b, K + 1, N + 2, N + 3)
    rows = np.unique(np.concatenate([np.arange(0, M, 37), [M - 1]]))
    err = fp64.gemm_normalized_error(c[rows], a[rows], b)
    print("%s normalized error %.3g" % (mnk, err))
    assert err <= 1e-6
    full = np.abs(c.astype(np.float64) - a.astype(np.float64) @ b.astype(np.float64)).max()
    assert full <= 1e-6 * K  # |a|, |b| <= 1


def test_scales(gpu_tensors):
    """Rows and columns scaled over 60 orders of magnitude: relative to the magnitudes of its own row
    and column, every element is as accurate as without scales."""
    M, N, K = 3000, 3000, 320
    a, b = inputs.uniform(M * K, 4043).reshape(M, K), inputs.uniform(K * N, 4044).reshape(K, N)
    sa = np.float32(10.0) ** np.linspace(-15, 15, M).astype(np.float32)
    sb = np.float32(10.0) ** np.linspace(15, -15, N).astype(np.float32)
    a, b = (a * sa[:, None]).astype(np.float32), (b * sb[None, :]).astype(np.float32)
    c = _gemm(gpu_tensors, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(c - a64 @ b64) <= 1e-6 * (np.abs(a64) @ np.abs(b64)))


def test_values_out_of_the_split_range(gpu_tensors):
    """Infinities, NaN, values above BF16's largest, parts below its smallest and products near FP32's:
    what FP32 products and sums give, in their tiles, and the others as before."""
    M, N, K = 3000, 3100, 290
    a, b = inputs.uniform(M * K, 4045).reshape(M, K), inputs.uniform(K * N, 4046).reshape(K, N)
    a[5, 3] = np.inf
    a[600, K - 1] = np.nan
    b[7, 1000] = -np.inf
    a[1300, :] = np.float32(3.0e-36) * a[1300, :]        # parts below BF16's range
    b[:, 2000] = np.float32(1.0e30) * b[:, 2000]
    a[2000, :] = 0.0
    a[2000, 17] = np.float32(3.4e38)                     # rounds to an infinite BF16
    a[2600, :] *= np.float32(1.0e-22)                    # products near FP32's smallest
    b[:, 2900] *= np.float32(1.0e-20)
    c = _gemm(gpu_tensors, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        want = a64 @ b64
        mag = np.abs(a64) @ np.abs(b64)
    big = np.abs(want) > 3.4028235e38
    want[big & np.isfinite(want)] = np.inf * np.sign(want[big & np.isfinite(want)])
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(c), np.isnan(want))
    assert np.array_equal(c[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)].astype(np.float32))
    assert np.all(np.abs(c[finite] - want[finite]) <= 1e-6 * mag[finite] + K * 2.0 ** -149)


def test_replayed(gpu_tensors):
    """Captured and replayed with an infinity in one replay: the next one is as accurate as the first."""
    import ctypes
    T = gpu_tensors
    M = N = 3000
    K = 290
    a, b = inputs.uniform(M * K, 4047).reshape(M, K), inputs.uniform(K * N, 4048).reshape(K, N)
    bad = a.copy()
    bad[10, 10] = np.inf
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)

    def call():
        capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))

    call()  # sizes the scratch
    want = download(T, bc, M * N)
    g = ctypes.c_void_p()
    capi.check(capi.lib.cs_graph_begin_capture(T.stream))
    call()
    capi.check(capi.lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
    for x in (a, bad, a, a):
        capi.check(capi.lib.cs_buffer_write(T.stream, ba.handle, 0, x.ctypes.data_as(ctypes.c_void_p), x.nbytes, 1))
        capi.check(capi.lib.cs_graph_launch(T.stream, g))
        got = download(T, bc, M * N)
        if x is a:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        else:
            assert np.all(np.isinf(got.reshape(M, N)[10])) and np.all(np.isfinite(got.reshape(M, N)[256:]))
    capi.lib.cs_graph_release(g)
    for h in (ba, bb, bc):
        h.release()
