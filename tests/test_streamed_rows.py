"""Vector widths of kernels whose rows four does not divide, by size and views (CPU: the kernel's text)."""
import re

import pytest

from compute import Tensors


def width(T, e, shape):
    return int(re.search(r"v < (\d+); \+\+v", T.kernel_source(e.closure, shape)).group(1))


# rows, columns, leaves, vector width (four: ragged, but for the last)
@pytest.mark.parametrize("rows,cols,leaves,expected", [
    (2048, 2050, 3, 4), (4096, 2050, 3, 2), (8192, 1002, 3, 2), (4096, 2050, 2, 4), (16384, 2050, 2, 2),
    (16384, 2050, 1, 2), (4096, 2049, 3, 4), (8192, 4099, 3, 1), (8192, 4099, 1, 4), (16384, 2052, 3, 4)])
def test_streams_take_a_dividing_width(rows, cols, leaves, expected):
    T = Tensors(offline=True)
    a, b, c = (T.Tensor.fill(0.0, (rows, cols)).nonInline for _ in range(3))
    e = {1: a * a, 2: a * b, 3: a * b + c}[leaves]
    assert width(T, e, (rows, cols)) == expected


def test_views_stay_ragged():
    T = Tensors(offline=True)
    a, b, c = (T.Tensor.fill(0.0, (4096, 2050)).nonInline for _ in range(3))
    assert width(T, a * b + c.translate([0, 1]), (4096, 2050)) == 4
