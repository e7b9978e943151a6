"""GEMMs whose K is cut into slices: their edges, values outside the three-part FP32 path, results inside
larger matrices, and a captured stream that has no room for partial results."""
import ctypes

import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs
from test_gemm_gpu import BOUND, VARIANTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", sorted(VARIANTS))
@pytest.mark.parametrize("mnk", [(64, 64, 4096), (17, 401, 2071), (33, 1, 4001), (1, 1, 4096),  # straight from A and B
                                 (600, 500, 4001), (1000, 999, 3001), (370, 1601, 2050)])       # packed
def test_slices(gpu_tensors, variant, mnk):
    T = gpu_tensors
    M, N, K = mnk
    ldc = N + 3
    a, b = inputs.uniform(M * K, 4081).reshape(M, K), inputs.uniform(K * N, 4082).reshape(K, N)
    ba, bb = upload(T, a), upload(T, b)
    for ld in (N, ldc):
        bc = upload(T, np.full(M * ldc + 1, 7.0, np.float32))
        capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr + 4, ld))
        got = download(T, bc, M * ldc + 1)
        c = got[1:1 + M * ld].reshape(M, ld)
        assert got[0] == 7.0 and np.all(c[:, N:] == 7.0) and np.all(got[1 + M * ld:] == 7.0)
        assert fp64.gemm_normalized_error(c[:, :N].copy(), a, b) <= BOUND[variant]
        bc.release()
    for h in (ba, bb):
        h.release()


def test_values_out_of_the_split_range(gpu_tensors):
    """FP32 tiles computed from A and B slice by slice: an infinity in one slice, NaN in another, a row
    of tiny values in all."""
    T = gpu_tensors
    M, N, K = 640, 1300, 3146
    a, b = inputs.uniform(M * K, 4083).reshape(M, K), inputs.uniform(K * N, 4084).reshape(K, N)
    a[5, 3] = np.inf
    a[300, K - 1] = np.nan
    a[500, :] *= np.float32(1.0e-36)
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    c = download(T, bc, M * N).reshape(M, N)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    finite = np.isfinite(want)
    assert np.array_equal(c[~finite], want[~finite].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(c[finite] - want[finite]) <= 1e-6 * mag[finite] + K * 2.0 ** -149)
    for h in (ba, bb, bc):
        h.release()


def test_captured_without_scratch(gpu_tensors):
    """A captured stream that never had scratch: the product runs without partial results."""
    T = gpu_tensors
    M, N, K = 64, 64, 4096
    a, b = inputs.uniform(M * K, 4085).reshape(M, K), inputs.uniform(K * N, 4086).reshape(K, N)
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    s, g = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(capi.lib.cs_stream_create(T.device, ctypes.byref(s)))
    capi.check(capi.lib.cs_stream_synchronize(T.stream))
    capi.check(capi.lib.cs_graph_begin_capture(s))
    capi.check(capi.lib.cs_gemm(s, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    capi.check(capi.lib.cs_graph_end_capture(s, ctypes.byref(g)))
    for _ in range(3):
        capi.check(capi.lib.cs_graph_launch(s, g))
        capi.check(capi.lib.cs_stream_synchronize(s))
        c = download(T, bc, M * N).reshape(M, N)
        assert fp64.gemm_normalized_error(c, a, b) <= BOUND["fp32"]
    capi.check(capi.lib.cs_graph_release(g))
    capi.check(capi.lib.cs_stream_destroy(s))
    for h in (ba, bb, bc):
        h.release()


@pytest.mark.parametrize("variant", sorted(VARIANTS))
def test_captured_after_a_larger_call(gpu_tensors, variant):
    """A stream's first call is large without operand copies; a smaller product is then captured whose plan
    has them, and one whose result lies over an operand."""
    T = gpu_tensors
    s = ctypes.c_void_p()
    capi.check(capi.lib.cs_stream_create(T.device, ctypes.byref(s)))
    big, M, N, K = 1500, 1400, 1300, 60
    a, b = inputs.uniform(M * K, 4087).reshape(M, K), inputs.uniform(K * N, 4088).reshape(K, N)
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, big * big)
    xa = upload(T, np.zeros(big * big, np.float32))
    n = 96
    sq = inputs.uniform(n * n, 4089).reshape(n, n)
    bs = upload(T, sq)
    capi.check(capi.lib.cs_stream_synchronize(T.stream))
    capi.check(capi.lib.cs_gemm(s, VARIANTS[variant], big, 1, big, xa.ptr, big, xa.ptr, 1, bc.ptr, 1))
    capi.check(capi.lib.cs_stream_synchronize(s))
    g = ctypes.c_void_p()
    capi.check(capi.lib.cs_graph_begin_capture(s))
    capi.check(capi.lib.cs_gemm(s, VARIANTS[variant], M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    capi.check(capi.lib.cs_gemm(s, VARIANTS[variant], n, n, n, bs.ptr, n, bb.ptr, n, bs.ptr, n))
    capi.check(capi.lib.cs_graph_end_capture(s, ctypes.byref(g)))
    capi.check(capi.lib.cs_graph_launch(s, g))
    capi.check(capi.lib.cs_stream_synchronize(s))
    c = download(T, bc, M * N).reshape(M, N)
    assert fp64.gemm_normalized_error(c, a, b) <= BOUND[variant]
    right = b.ravel()[:n * n].reshape(n, n).copy()
    assert fp64.gemm_normalized_error(download(T, bs, n * n).reshape(n, n), sq, right) <= BOUND[variant]
    capi.check(capi.lib.cs_graph_release(g))
    capi.check(capi.lib.cs_stream_destroy(s))
    for h in (ba, bb, bc, xa, bs):
        h.release()
