"""Evaluations that the layer kernels take for their speed: the same bits as the same samples a few at a
time, which the whole-network kernel takes."""
import numpy as np
import pytest

from compute import costmodel
from gpu_util import upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths,n", [([64, 8, 4], 65536), ([32, 16, 1], 70001), ([1000, 1], 30011),
                                      ([512, 8], 65537), ([256, 4, 1], 70001), ([16, 8, 8, 1], 40001),
                                      ([16, 1], 65536), ([200, 8, 1], 65536)])
def test_same_bits_as_few_samples(gpu_tensors, widths, n):
    T, part = gpu_tensors, 777
    net = costmodel.Network(T, widths, seed=4)
    X = np.random.default_rng(n).standard_normal((n, widths[0])).astype(np.float32)
    xb, yb = upload(T, X), T._alloc(n * widths[-1] * 4)
    net.forward_device(xb.ptr, n, yb.ptr)
    y = yb.to_numpy(n * widths[-1]).reshape(n, widths[-1])
    for at in (0, n - part):
        net.forward_device(xb.ptr + 4 * at * widths[0], part, yb.ptr)
        got = yb.to_numpy(part * widths[-1]).reshape(part, widths[-1])
        assert np.array_equal(got.view(np.uint32), y[at:at + part].view(np.uint32))
    for b in (xb, yb):
        b.release()
    net.release()
