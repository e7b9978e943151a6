"""Infinite parameters reach the gradients through the samples there are, not through the zeros that fill
up a workgroup's share of them."""
import numpy as np
import pytest

from compute import costmodel
from gpu_util import upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 9])
def test_infinite_weight_without_effect(gpu_tensors, n):
    """Unit 0 of the first layer is 1 - x, 0 for the samples and 1 for a sample of zeros, so the infinite
    weight behind it meets zeros only: unit 0 of the second layer is relu(NaN) = 0 with it and relu(-1) = 0
    without, and the gradients are the same."""
    T = gpu_tensors
    X, t = np.full((n, 1), 2.0, np.float32), np.arange(n, dtype=np.float32)
    grads = []
    for weight in (0.0, np.inf):
        net = costmodel.Network(T, [1, 2, 2, 1], seed=1)
        net.set_params(np.array([-1.0, 0.5, 1.0, 0.0,                # W1, b1
                                 weight, 0.25, 0.0, 0.5, -1.0, 0.125,  # W2, b2
                                 0.75, -0.5, 0.0625], np.float32))     # W3, b3
        xb, tb = upload(T, X), upload(T, t)
        loss, g = net.gradients_device(xb.ptr, tb.ptr, n)
        grads.append(np.append(g.to_numpy(net.count), loss.to_numpy(1)))
        xb.release()
        tb.release()
        net.release()
    assert np.all(np.isfinite(grads[0])) and np.array_equal(grads[0], grads[1])
