"""FP32 products on the three-part path where some chunks of 64 K values leave the split's range: those
run on the FP32 matrix cores within the same tile, in any order of chunks, with slices of K and K tails."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu

PATTERNS = {"first": lambda c, n: c == 0, "last": lambda c, n: c == n - 1, "even": lambda c, n: c % 2 == 0,
            "odd": lambda c, n: c % 2 == 1, "all": lambda c, n: True, "one in": lambda c, n: c != n // 2,
            "one out": lambda c, n: c == n // 2}


# 256 x 256 tiles; 128 x 128 tiles; 128 x 128 tiles in slices of K; more than 64 chunks
@pytest.mark.parametrize("mnk", [(4096, 4000, 500), (2048, 2048, 450), (1024, 1024, 4093), (1000, 1100, 8200)])
@pytest.mark.parametrize("pattern", sorted(PATTERNS))
def test_chunks_out_of_range(gpu_tensors, mnk, pattern):
    T = gpu_tensors
    M, N, K = mnk
    a, b = inputs.uniform(M * K, 4061).reshape(M, K), inputs.uniform(K * N, 4062).reshape(K, N)
    chunks = (K + 63) // 64
    tiny = [c for c in range(chunks) if PATTERNS[pattern](c, chunks)]
    rows = [5, M // 2, M - 1]
    a[rows[0]] = 0.0  # these products alone in one row
    for c in tiny:
        k = slice(64 * c, min(64 * c + 64, K))
        a[rows[0], k] = np.float32(1e-37) * inputs.uniform(k.stop - k.start, 4063 + c)
        a[rows[1:], k] *= np.float32(1e-37)
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    c = download(T, bc, M * N).reshape(M, N)
    check = np.unique(rows + list(range(0, M, 61)))
    a64, b64 = a[check].astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(c[check] - a64 @ b64) <= 1e-6 * (np.abs(a64) @ np.abs(b64)) + K * 2.0 ** -149)
    for h in (ba, bb, bc):
        h.release()
