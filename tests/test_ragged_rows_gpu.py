"""Generated kernels whose rows the vector width does not divide: the same bits as one element at a
time, for every way a leaf is read and an output is written."""
import ctypes

import numpy as np
import pytest

from compute import Tensors, _capi as capi
from compute import autotune
from oracle import inputs

pytestmark = pytest.mark.gpu


def _leaf(T, shape, seed):
    return T.Tensor(inputs.normal(int(np.prod(shape)), seed).reshape(shape), padding=0.25)


FORMS = {
    "direct": lambda T, h, w: _leaf(T, (h, w), 1) * _leaf(T, (h, w), 2) + _leaf(T, (h, w), 3),
    "flat": lambda T, h, w: _leaf(T, (h * w,), 1) - _leaf(T, (h * w,), 2),
    "translated": lambda T, h, w: _leaf(T, (h, w), 1).translate([1, 2]) + _leaf(T, (h, w), 2).translate([0, -3]),
    "cut": lambda T, h, w: _leaf(T, (h, w + 3), 1).translate([0, -1], (h, w)) * _leaf(T, (h, 8), 2).translate([0, 1], (h, w)),
    "transposed": lambda T, h, w: _leaf(T, (w, h), 1).transpose() + _leaf(T, (h, w), 2),
    "reversed": lambda T, h, w: _leaf(T, (h, w), 1)._transform((h, w), [1.0, 0.0, 0.0, 0.0, -1.0, w - 1.0]) * _leaf(T, (h, w), 2),
    "scaled": lambda T, h, w: _leaf(T, (h, 2 * w), 1).scale((h, w)) + _leaf(T, (h, max(1, w // 2)), 2).scale((h, w)),
    "broadcast": lambda T, h, w: _leaf(T, (h, w), 1) / _leaf(T, (h,), 2) + _leaf(T, (1, w), 3),
    "rank 3": lambda T, h, w: T.Tensor.tanh(_leaf(T, (3, h, w), 1).permute([1, 0, 2]) + _leaf(T, (h,), 2)),
}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("hw", [(1, 5), (3, 6), (70, 7), (33, 9), (300, 13), (17, 30), (5, 255), (2, 1025), (1500, 4099)])
def test_bits_of_one_element_at_a_time(form, hw):
    with Tensors(0) as T, Tensors(0, vector_width=1, launch_order=capi.ORDER_LINEAR) as one:
        e, f = FORMS[form](T, *hw), FORMS[form](one, *hw)
        assert e.shape[-1] % 4 == 0 or "_v4u" in T.kernel_source(e.closure, e.shape)
        assert "_v1u" in one.kernel_source(f.closure, f.shape)
        got, want = e.flatArray(), f.flatArray()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        exact = want.astype(np.float64).sum()
        if np.isfinite(exact):  # the repeated elements are added once
            assert abs(float(e.sum().flatArray()[0]) - exact) <= 4 * 2.0 ** -23 * np.abs(want).astype(np.float64).sum() + 1e-30


@pytest.mark.parametrize("parts", [2, 3, 4])
@pytest.mark.parametrize("hw", [(3, 5), (40, 11), (9, 130)])
def test_joined_outputs(parts, hw):
    def build(T):
        a, b = _leaf(T, hw, 1), _leaf(T, hw, 2)
        return T.Tensor.join([a * b, a - b, a.translate([0, 1]) + b, T.Tensor.abs(a)][:parts])
    with Tensors(0) as T, Tensors(0, vector_width=1) as one:
        got, want = build(T).flatArray(), build(one).flatArray()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("items,block", [(1, 64), (3, 256), (8, 1024)])
def test_stores_stay_inside(items, block):
    """Non-temporal stores and other launch shapes; what lies around the output stays."""
    h, w, guard = 23, 77, 4
    with Tensors(0) as T:
        a, b = _leaf(T, (h, w), 1).doCache(), _leaf(T, (h, w), 2).doCache()
        e = a + b.translate([0, 1])
        want = e.flatArray()
        cfg = {"vector_width": 0, "items_per_thread": items, "block_size": block, "nontemporal_store": 1}
        f, leaves = autotune.compile_with(T, e.closure, e.shape, cfg)
        out = T.Tensor(np.full(h * w + 2 * guard, 7.0, np.float32)).doCache()
        ptrs = (ctypes.c_void_p * len(leaves))(*[leaf.id.buffer.ptr for leaf in leaves])
        capi.check(capi.lib.cs_fused_launch(T.stream, f, ptrs, len(leaves), out.buffer.ptr + 4 * guard))
        got = out.flatArray()
        assert np.all(got[:guard] == 7.0) and np.all(got[-guard:] == 7.0)
        assert np.array_equal(got[guard:-guard].view(np.uint32), want.view(np.uint32))
        capi.lib.cs_fused_release(f)
        for t in (a, b, out):
            t.release()


@pytest.mark.parametrize("hw", [(3, 5), (257, 7), (64, 1021), (1, 1000003)])
def test_result_over_a_leaf(hw):
    """The output in the memory of a leaf that is read at its own place."""
    with Tensors(0) as T:
        a, b = _leaf(T, hw, 1).doCache(), _leaf(T, hw, 2).doCache()
        e = a * b + a
        want = e.flatArray()
        f, leaves, _ = T.compile(e.closure, e.shape)
        ptrs = (ctypes.c_void_p * len(leaves))(*[leaf.id.buffer.ptr for leaf in leaves])
        capi.check(capi.lib.cs_fused_launch(T.stream, f, ptrs, len(leaves), a.buffer.ptr))
        assert np.array_equal(a.flatArray().view(np.uint32), want.view(np.uint32))
        capi.lib.cs_fused_release(f)
        for t in (a, b):
            t.release()


def test_in_a_batch():
    """The same kernels as members of a persistent batch."""
    with Tensors(0) as T:
        exprs = [FORMS[k](T, 37, 61) for k in ("direct", "translated", "transposed", "rank 3")]
        want = [e.flatArray() for e in exprs]
        handles, args, outs, kept = [], [], [], []
        for e, v in zip(exprs, want):
            f, leaves, _ = T.compile(e.closure, e.shape)
            bufs = [leaf.id.doBuffer() for leaf in leaves]
            out = T._alloc(v.nbytes)
            handles.append(f)
            kept += bufs
            outs.append(out)
            args += [x.ptr for x in bufs] + [out.ptr]
        batch = ctypes.c_void_p()
        capi.check(capi.lib.cs_batch_create(T.device, (ctypes.c_void_p * len(handles))(*handles), len(handles), 256,
                                            ctypes.byref(batch)))
        capi.check(capi.lib.cs_batch_bind(T.stream, batch, (ctypes.c_void_p * len(args))(*args), len(args)))
        capi.check(capi.lib.cs_batch_launch(T.stream, batch))
        for out, v in zip(outs, want):
            assert np.array_equal(out.to_numpy(v.size).view(np.uint32), v.view(np.uint32))
        capi.check(capi.lib.cs_batch_release(batch))
        for f in handles:
            capi.lib.cs_fused_release(f)
        for x in kept + outs:
            x.release()
