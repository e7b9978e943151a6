"""Evaluations in place under capture: they keep every layer's activations, which the evaluations before
them did not need."""
import ctypes

import numpy as np
import pytest

from compute import _capi as capi
from compute import costmodel
from gpu_util import upload

pytestmark = pytest.mark.gpu
lib = capi.lib


@pytest.mark.parametrize("n", [40, 3000])
def test_in_place_after_an_eager_evaluation(gpu_tensors, n):
    T = gpu_tensors
    net = costmodel.Network(T, [5, 32, 32, 1], seed=3)
    X = np.random.default_rng(n).standard_normal((n, 5)).astype(np.float32)
    xb, yb = upload(T, X), T._alloc(n * 4)
    net.forward_device(xb.ptr, n, yb.ptr)
    want = yb.to_numpy(n)
    graphs = []
    for m in (n // 2, n):  # the workspace grows from one capture to the next
        g = ctypes.c_void_p()
        capi.check(lib.cs_graph_begin_capture(T.stream))
        try:
            net.forward_device(xb.ptr, m, xb.ptr)
        finally:
            capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(g)))
        graphs.append((m, g))
    for m, g in graphs * 3:
        capi.check(lib.cs_buffer_write(T.stream, xb.handle, 0, X.ctypes.data_as(ctypes.c_void_p), X.nbytes, 1))
        capi.check(lib.cs_graph_launch(T.stream, g))
        assert np.max(np.abs(xb.to_numpy(m) - want[:m])) <= 1e-5 * np.max(np.abs(want))
        capi.check(lib.cs_buffer_write(T.stream, xb.handle, 0, X.ctypes.data_as(ctypes.c_void_p), X.nbytes, 1))
        net.forward_device(xb.ptr, n, yb.ptr)  # eager work between the replays
    for _, g in graphs:
        lib.cs_graph_release(g)
    for b in (xb, yb):
        b.release()
    net.release()
