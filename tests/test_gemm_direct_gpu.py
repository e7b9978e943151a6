"""The GEMM without a pre-pass: every launch shape of its plan, remainders in each dimension, leading
dimensions and pointers at any 4-byte boundary, and a C that overlaps an operand."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import fp64, inputs
from test_gemm_gpu import BOUND, VARIANTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", sorted(VARIANTS))
@pytest.mark.parametrize("mnk", [(5000, 9, 20),                       # one wave per tile of 16
                                 (2000, 63, 333), (300, 200, 300),    # 4 and 16 waves per tile of 16
                                 (17, 33, 333), (16, 16, 128),
                                 (600, 511, 20), (601, 512, 133),     # 1 and 4 waves per tile of 32
                                 (512, 512, 260), (511, 509, 130),    # 8 waves per tile of 32
                                 (1025, 1001, 31), (1024, 1023, 97),  # 1 and 4 waves per tile of 64
                                 (1, 1000, 5), (1000, 1, 129), (3, 2, 1)])
def test_direct_shapes(gpu_tensors, variant, mnk):
    T = gpu_tensors
    M, N, K = mnk
    lda, ldb, ldc = K + 3, N + 1, N + 5
    a = inputs.uniform(M * lda, 4021).reshape(M, lda)
    b = inputs.uniform(K * ldb, 4022).reshape(K, ldb)
    ba = upload(T, np.concatenate([[0.0], a.ravel()]))
    bb = upload(T, np.concatenate([[0.0], b.ravel()]))
    bc = upload(T, np.full(M * ldc + 1, 7.0, np.float32))
    capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], M, N, K, ba.ptr + 4, lda, bb.ptr + 4, ldb, bc.ptr + 4, ldc))
    got = download(T, bc, M * ldc + 1)
    c = got[1:].reshape(M, ldc)
    assert got[0] == 7.0 and np.all(c[:, N:] == 7.0)
    assert fp64.gemm_normalized_error(c[:, :N].copy(), a[:, :K].copy(), b[:, :N].copy()) <= BOUND[variant]
    for h in (ba, bb, bc):
        h.release()


@pytest.mark.parametrize("variant", sorted(VARIANTS))
@pytest.mark.parametrize("operand", ["a", "b"])
def test_result_over_an_operand(gpu_tensors, variant, operand):
    """C in the memory of A or of B: the operand is read before it is overwritten."""
    T = gpu_tensors
    n = 96
    a, b = inputs.uniform(n * n, 4031).reshape(n, n), inputs.uniform(n * n, 4032).reshape(n, n)
    ba, bb = upload(T, a), upload(T, b)
    bc = ba if operand == "a" else bb
    capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], n, n, n, ba.ptr, n, bb.ptr, n, bc.ptr, n))
    assert fp64.gemm_normalized_error(download(T, bc, n * n).reshape(n, n), a, b) <= BOUND[variant]
    for h in (ba, bb):
        h.release()


@pytest.mark.parametrize("mnk", [(40, 50, 30), (600, 512, 130)])
def test_direct_special_values(gpu_tensors, mnk):
    """An infinity or NaN reaches its own row or column of C only, as FP32 products give it."""
    T = gpu_tensors
    M, N, K = mnk
    a, b = np.ones((M, K), np.float32), np.ones((K, N), np.float32)
    a[1, K - 1] = np.inf
    a[M - 1, 0] = np.nan
    b[2, N - 1] = -np.inf
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    want = np.full((M, N), K, np.float32)
    want[1, :] = np.inf
    want[:, N - 1] = -np.inf
    want[1, N - 1] = np.nan  # inf - inf
    want[M - 1, :] = np.nan
    assert np.array_equal(download(T, bc, M * N).reshape(M, N), want, equal_nan=True)
    for h in (ba, bb, bc):
        h.release()


@pytest.mark.parametrize("variant", sorted(VARIANTS))
@pytest.mark.parametrize("mnk", [(1500, 1400, 260), (2049, 1031, 300), (640, 4097, 515)])
def test_tiles_of_128(gpu_tensors, variant, mnk):
    """The packed kernels on 128 x 128 tiles: remainders in every dimension."""
    T = gpu_tensors
    M, N, K = mnk
    a, b = inputs.uniform(M * K, 4051).reshape(M, K), inputs.uniform(K * N, 4052).reshape(K, N)
    ba, bb = upload(T, a), upload(T, b)
    bc = upload(T, np.full(M * N + 8, 7.0, np.float32))
    capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    got = download(T, bc, M * N + 8)
    assert np.all(got[M * N:] == 7.0)
    c = got[:M * N].reshape(M, N)
    assert fp64.gemm_normalized_error(c, a, b) <= BOUND[variant]
    for h in (ba, bb, bc):
        h.release()


def test_depth_is_limited_on_every_path(gpu_tensors):
    """A K whose packed rows pass the 32-bit offsets is refused for small products too."""
    T = gpu_tensors
    K = 1 << 21
    a, b, c = alloc(T, K), alloc(T, K), alloc(T, 1)
    with pytest.raises(capi.InvalidValue):
        capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, 1, 1, K, a.ptr, K, b.ptr, 1, c.ptr, 1))
    for h in (a, b, c):
        h.release()


@pytest.mark.parametrize("variant", sorted(set(VARIANTS) - {"fp32"}))
@pytest.mark.parametrize("k", [17, 65, 129, 200, 257, 400, 640])
def test_ring_of_four_stages(gpu_tensors, variant, k):
    """128 x 128 tiles with four stages in LDS: fewer stages than that, exactly as many, more."""
    T = gpu_tensors
    M, N = 1999, 1901
    a, b = inputs.uniform(M * k, 4061).reshape(M, k), inputs.uniform(k * N, 4062).reshape(k, N)
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    for _ in range(2):
        capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], M, N, k, ba.ptr, k, bb.ptr, N, bc.ptr, N))
        c = download(T, bc, M * N).reshape(M, N)
        assert fp64.gemm_normalized_error(c, a, b) <= BOUND[variant]
    for h in (ba, bb, bc):
        h.release()


@pytest.mark.parametrize("variant", sorted(VARIANTS))
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_packed_at_any_4_byte_boundary(gpu_tensors, variant, shift):
    """Packed operands whose rows start off the 16-byte grid, inside larger matrices."""
    T = gpu_tensors
    M, N, K = 1800, 1700, 133
    lda, ldb = K + shift, N + shift
    a = inputs.uniform(M * lda, 4071).reshape(M, lda)
    b = inputs.uniform(K * ldb, 4072).reshape(K, ldb)
    ba = upload(T, np.concatenate([np.full(shift, np.nan), a.ravel()]))
    bb = upload(T, np.concatenate([np.full(shift, np.nan), b.ravel()]))
    bc = alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, VARIANTS[variant], M, N, K, ba.ptr + 4 * shift, lda, bb.ptr + 4 * shift, ldb,
                                bc.ptr, N))
    c = download(T, bc, M * N).reshape(M, N)
    assert fp64.gemm_normalized_error(c, a[:, :K].copy(), b[:, :N].copy()) <= BOUND[variant]
    for h in (ba, bb, bc):
        h.release()
