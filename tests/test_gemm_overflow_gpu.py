"""FP32 products on the three-part path whose values come near FP32's largest: what FP32 products and sums
give, not an overflow of the parts, whose leading one may be above the value."""
import numpy as np
import pytest

from compute import _capi as capi
from gpu_util import alloc, download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu

NEAR = np.float32(2.0 ** 64 - 2.0 ** 40)  # its square is FP32's largest but one; its leading part is 2^64


@pytest.mark.parametrize("mnk", [(3000, 3000, 290), (2048, 2048, 300), (1024, 1024, 4096)])
def test_near_the_largest(gpu_tensors, mnk):
    T = gpu_tensors
    M, N, K = mnk
    a, b = inputs.uniform(M * K, 4051).reshape(M, K), inputs.uniform(K * N, 4052).reshape(K, N)
    a[5], a[700], b[:, 7], b[:, 800] = 0.0, 0.0, 0.0, 0.0
    a[5, 3], b[3, 7] = NEAR, NEAR                      # one product
    a[700, [3, 20, K - 1]] = 1.7e38, 1.7e38, 3.0       # a difference of two, and a small term
    b[[3, 20, K - 1], 800] = 2.0, -2.0, 1.0
    ba, bb, bc = upload(T, a), upload(T, b), alloc(T, M * N)
    capi.check(capi.lib.cs_gemm(T.stream, capi.GEMM_FP32, M, N, K, ba.ptr, K, bb.ptr, N, bc.ptr, N))
    c = download(T, bc, M * N).reshape(M, N)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    assert c[5, 7] == np.float32(np.float64(NEAR) ** 2)
    over = np.abs(want) > np.finfo(np.float32).max  # 1.7e38 of row 700 meets NEAR of column 7
    assert np.argwhere(over).tolist() == [[700, 7]] and np.all(c[over] == np.inf)
    assert np.all(np.abs(c[~over] - want[~over]) <= 1e-6 * mag[~over])  # NaN and infinities fail
    for h in (ba, bb, bc):
        h.release()
