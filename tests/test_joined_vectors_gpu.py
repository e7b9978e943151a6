"""Joins of several outputs at their default vector widths: rows that the width divides and rows that it
does not, permuted and translated operands, both sides of every limit on the number of outputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nout,width", [(2, 2), (3, 1), (4, 1), (5, 1), (12, 1), (13, 4)])
@pytest.mark.parametrize("shape", [(3, 8, 64), (5, 7, 33), (2, 9, 6), (1, 1, 5), (300, 3)])
def test_joined(gpu_tensors, nout, width, shape):
    T = gpu_tensors
    rng = np.random.default_rng(17 * nout + len(shape))
    a, b = rng.uniform(-1, 1, shape).astype(np.float32), rng.uniform(-1, 1, shape).astype(np.float32)
    ta, tb = T.Tensor(a), T.Tensor(b)
    parts, want = [], []
    for i in range(nout):
        move = [0] * (len(shape) - 1) + [i % 3 - 1]
        parts.append(ta.translate(move) * T.Tensor.fill(float(i + 1), shape) + tb)
        t = np.zeros_like(a)
        d = move[-1]
        if d == 0:
            t = a
        elif d == 1:
            t[..., 1:] = a[..., :-1]
        else:
            t[..., :-1] = a[..., 1:]
        want.append(t * np.float32(i + 1) + b)
    j = T.Tensor.join(parts)
    last = shape[-1]
    while last % width:
        width //= 2
    (closure,), _ = j.closures()
    assert ("V=%d " % width) in T.kernel_source(closure, shape)
    got = np.asarray(j.flatArray(), np.float32).reshape(shape + (nout,))
    assert np.array_equal(got, np.stack(want, axis=-1))
