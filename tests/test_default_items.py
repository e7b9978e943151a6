"""Vectors per thread of the automatic launch shape, by size, functions and views (CPU: the kernel's text)."""
import re

import pytest

from compute import Tensors

CHAIN = "exp of a view"


def expression(T, kind, shape):
    a, b = (T.Tensor.fill(0.0, shape).nonInline for _ in range(2))
    return {"a*b": lambda: a * b, "exp": lambda: T.Tensor.exp(a) * b, "log": lambda: T.Tensor.log(a),
            CHAIN: lambda: T.Tensor.exp(a + b.translate([0, 1])),
            "transposed": lambda: T.Tensor.tanh(a.transpose())}[kind]()


@pytest.mark.parametrize("kind,rows,items", [
    ("a*b", 4095, 1), ("a*b", 4096, 2), ("exp", 4096, 1), ("exp", 8191, 1), ("exp", 8192, 2), ("log", 4096, 1),
    (CHAIN, 4095, 1), (CHAIN, 4096, 2), ("transposed", 4096, 2)])
def test_items_per_thread(kind, rows, items):
    T = Tensors(offline=True)
    e = expression(T, kind, (rows, 1024))
    assert int(re.search(r"unsigned q\[(\d)\]", T.kernel_source(e.closure, e.shape)).group(1)) == items
