"""The whole-network kernel at the edges of its padding (16), of a wave's units (64) and of its parameter
copy, and evaluation on both sides of the sample count from which a workgroup takes more samples."""
import numpy as np
import pytest

from compute import costmodel
from gpu_util import upload
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths", [[1, 1], [1, 2, 1], [15, 16, 17, 1], [16, 15, 33, 1], [64, 65, 63, 1],
                                    [5, 129, 127, 1], [3, 260, 20, 1]])
@pytest.mark.parametrize("n", [3, 700, 5001])
def test_widths(gpu_tensors, widths, n):
    T = gpu_tensors
    net = costmodel.Network(T, widths, seed=9)
    rng = np.random.default_rng(n)
    X, t = rng.standard_normal((n, widths[0])).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    p = net.get_params()
    xb, tb, yb = upload(T, X), upload(T, t), T._alloc(n * 4)
    net.forward_device(xb.ptr, n, yb.ptr)
    y, y64 = yb.to_numpy(n), mlp_ref.forward(p, widths, X)[-1][:, 0]
    assert np.max(np.abs(y - y64)) <= 1e-5 * max(1.0, np.max(np.abs(y64)))
    net.forward_device(xb.ptr, min(n, 801), yb.ptr)  # fewer samples: the same bits
    assert np.array_equal(yb.to_numpy(min(n, 801)), y[:801])
    for _ in range(2):
        loss_buf, g_buf = net.gradients_device(xb.ptr, tb.ptr, n)
    g, loss = g_buf.to_numpy(net.count), float(loss_buf.to_numpy(1)[0])
    loss64, g64 = mlp_ref.loss_and_grad(p, widths, X, t)
    assert abs(loss - loss64) <= 1e-5 * max(1.0, loss64)
    assert np.max(np.abs(g - g64)) <= 1e-4 * np.max(np.abs(g64))
    for b in (xb, tb, yb):
        b.release()
    net.release()
