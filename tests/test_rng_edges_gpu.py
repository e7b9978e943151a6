"""The random kernels at the ends of their vectors and of their draws' range."""
import numpy as np
import pytest

import oracle
from compute import _capi as capi
from gpu_util import download, upload
from oracle import fp64, inputs

pytestmark = pytest.mark.gpu


def _seed_of(h):
    """The seed whose element 0 hashes to h (the hash is a bijection of 32-bit integers)."""
    m = 0xFFFFFFFF
    v = h ^ (h >> 15) ^ (h >> 30)
    v = v * pow(0x27D4EB2D, -1, 1 << 32) & m
    x = v
    for _ in range(8):
        x = v ^ (x << 4 & m)
    v = x * pow(9, -1, 1 << 32) & m
    v = v ^ (v >> 16)  # undoes (v ^ 61) ^ (v >> 16), but for the constant
    return v ^ 61


def _run(T, f, n, seed, shift):
    guard = 5
    b = upload(T, np.full(shift + n + guard, 7.0, np.float32))
    written = n + (n & 1) if f is capi.lib.cs_random_normal else n
    capi.check(f(T.stream, b.ptr + 4 * shift, n, seed))
    got = download(T, b, shift + n + guard)
    b.release()
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + written:] == 7.0)
    return got[shift:shift + n]


@pytest.mark.parametrize("shift", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1024, 1025, 2050, 5000001])
def test_lengths(gpu_tensors, n, shift):
    T = gpu_tensors
    assert np.array_equal(_run(T, capi.lib.cs_random, n, 99, shift).view(np.uint32), oracle.random(n, 99).view(np.uint32))
    got, want = _run(T, capi.lib.cs_random_normal, n, 99, shift), oracle.random_normal(n, 99)
    finite = np.isfinite(want)
    assert fp64.ulp_distance(got, want)[finite].max() <= 2 or np.abs(got - want)[finite].max() <= 4e-7
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True)


@pytest.mark.parametrize("h", [0, 1, 2, 127, 128, 0x7FFFFFFF, 0x80000000, 0x80000001, 0xFE000000, 0xFEFFFFFF, 0xFF000000,
                               0xFFFFFF00, 0xFFFFFF7F, 0xFFFFFF80, 0xFFFFFFFF])
def test_first_draw(gpu_tensors, h):
    """Draws at the ends of the range and around the logarithm's powers of two: infinite at 0, a zero
    of the right sign where the draw rounds to 1."""
    seed = _seed_of(h)
    assert inputs.wang_hash(np.uint32(seed)) == h
    got, want = _run(gpu_tensors, capi.lib.cs_random_normal, 2, seed, 0), oracle.random_normal(2, seed)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    assert np.array_equal(np.signbit(got), np.signbit(want))
    finite = np.isfinite(want)
    if finite.any():
        assert fp64.ulp_distance(got, want)[finite].max() <= 2
