"""The cost-model network's kernels at the edges of their plan: whole networks in LDS with all or one
layer's parameters at a time, networks too wide for it, and sample counts around the workgroup's."""
import numpy as np
import pytest

from compute import costmodel
from gpu_util import upload
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths", [[3, 1], [7, 5, 1], [23, 64, 64, 64, 1], [9, 130, 66, 1],
                                    [32, 128, 128, 128, 1],  # one layer's parameters at a time
                                    [200, 300, 1]])          # layer by layer
@pytest.mark.parametrize("n", [1, 8, 13, 2500])
def test_gradients_match_fp64(gpu_tensors, widths, n):
    T = gpu_tensors
    net = costmodel.Network(T, widths, seed=5)
    rng = np.random.default_rng(n)
    X, t = rng.standard_normal((n, widths[0])).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    p = net.get_params()
    xb, tb, yb = upload(T, X), upload(T, t), T._alloc(n * 4)
    net.forward_device(xb.ptr, n, yb.ptr)
    y, y64 = yb.to_numpy(n), mlp_ref.forward(p, widths, X)[-1][:, 0]
    assert np.max(np.abs(y - y64)) <= 1e-5 * max(1.0, np.max(np.abs(y64)))
    for _ in range(2):  # the second call finds the first one's workspace
        loss_buf, g_buf = net.gradients_device(xb.ptr, tb.ptr, n)
    g, loss = g_buf.to_numpy(net.count), float(loss_buf.to_numpy(1)[0])
    loss64, g64 = mlp_ref.loss_and_grad(p, widths, X, t)
    assert abs(loss - loss64) <= 1e-5 * max(1.0, loss64)
    assert np.max(np.abs(g - g64)) <= 1e-4 * np.max(np.abs(g64))
    for b in (xb, tb, yb):
        b.release()
    net.release()


def test_outputs_of_a_wide_last_layer(gpu_tensors):
    """Several outputs per sample, and enough samples of a narrow network for the layer kernels: the
    same bits as the same samples a few at a time."""
    T = gpu_tensors
    net = costmodel.Network(T, [4, 6, 3], seed=2)
    n, part = 70001, 801
    X = np.random.default_rng(3).standard_normal((n, 4)).astype(np.float32)
    xb, yb = upload(T, X), T._alloc(n * 12)
    net.forward_device(xb.ptr, n, yb.ptr)
    y = yb.to_numpy(n * 3)
    net.forward_device(xb.ptr, part, yb.ptr)
    assert np.array_equal(yb.to_numpy(part * 3), y[:part * 3])
    for b in (xb, yb):
        b.release()
    net.release()
