"""Wide stores written as assembly carry the wait states that keep a later write of their registers from
reaching the data (CPU: the kernel's text)."""
import re

import pytest

from compute import Tensors
from test_codegen import compiles


@pytest.mark.parametrize("width", [256, 257])  # whole and ragged rows
@pytest.mark.parametrize("items", [1, 2])
@pytest.mark.parametrize("nontemporal", [0, 1])
def test_wide_stores_wait(width, items, nontemporal):
    T = Tensors(offline=True, items_per_thread=items)
    T.options.nontemporal_store = nontemporal
    a, b = (T.Tensor.fill(0.0, (64, width)).nonInline for _ in range(2))
    src = T.kernel_source((a * b + a).closure, (64, width))
    stores = re.findall(r'"global_store_dwordx4 ([^"]*)"', src)
    assert stores and all(s.endswith("\\n\\ts_nop 1") for s in stores)
    compiles(src)


@pytest.mark.parametrize("items", [1, 2, 3])
def test_values_come_before_the_stores(items):
    """With several vectors per thread no value is left to be computed behind the first store."""
    T = Tensors(offline=True, items_per_thread=items)
    a, b = (T.Tensor.fill(0.0, (64, 256)).nonInline for _ in range(2))
    src = T.kernel_source((a * b + a).closure, (64, 256))
    first_store = src.index('asm volatile("global_store_dwordx4')
    assert ('asm volatile("" :: "v"(' in src[:first_store]) == (items > 1)
    compiles(src)


@pytest.mark.parametrize("rows,through", [((1 << 22) - 1, False), (1 << 22, True)])
def test_single_floats_write_through_past_the_caches(rows, through):
    T = Tensors(offline=True)
    a = T.Tensor.fill(0.0, (rows, 1)).nonInline
    assert ("global_store_dword %0" in T.kernel_source((a * a).closure, (rows, 1))) == through
