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
