"""A kernel with ragged rows launched into the memory of a leaf runs at another width: that code belongs
to the kernel's handle, not to the device's cache."""
import ctypes

import numpy as np
import pytest

from compute import Tensors
from compute import _capi as capi
from gpu_util import download, upload
from oracle import inputs

pytestmark = pytest.mark.gpu
lib = capi.lib


def test_code_lives_as_long_as_the_handle():
    shape = (33, 61)
    n = shape[0] * shape[1]
    x, y = (inputs.uniform(n, s) for s in (71, 72))
    with Tensors(0) as T:
        a, b = (T.Tensor(v.reshape(shape)).doCache() for v in (x, y))
        e = a * b + a
        f, leaves, _ = T.compile(e.closure, e.shape)
        p = {id(a): upload(T, x), id(b): upload(T, y)}
        ptrs = (ctypes.c_void_p * len(leaves))(*[p[id(leaf.id)].ptr for leaf in leaves])
        out = p[id(a)].ptr
        launch = lambda: capi.check(lib.cs_fused_launch(T.stream, f, ptrs, len(leaves), out))  # noqa: E731
        entries = T.info(capi.INFO_FUSED_CACHE_ENTRIES)
        graph = ctypes.c_void_p()
        capi.check(lib.cs_graph_begin_capture(T.stream))
        launch()
        capi.check(lib.cs_graph_end_capture(T.stream, ctypes.byref(graph)))
        assert T.info(capi.INFO_FUSED_CACHE_ENTRIES) == entries
        capi.check(lib.cs_fused_cache_clear(T.device))
        want = x.copy()
        for k in range(4):  # replays and eager launches in turn
            if k % 2:
                launch()
            else:
                capi.check(lib.cs_graph_launch(T.stream, graph))
            want = want * y + want
            assert np.array_equal(download(T, p[id(a)], n).view(np.uint32), want.view(np.uint32))
        assert T.info(capi.INFO_FUSED_CACHE_ENTRIES) == 0  # not built again
        capi.check(lib.cs_graph_release(graph))
        lib.cs_fused_release(f)
        for t in (a, b) + tuple(p.values()):
            t.release()
