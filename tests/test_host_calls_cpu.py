"""The compiled call layer (csrc/host.cpp) without a GPU: it binds entry points
the library exports, and hands every argument it does not take back to the
Python functions (None), which refuse it with their own errors."""

from __future__ import annotations

import pytest
import torch

from engine import _lib
from engine.quant import int8_matmul


def test_binds_exported_entry_points():
    assert set(_lib.host().names()) <= set(_lib.EXPORTED_SYMBOLS)


@pytest.mark.parametrize("name,n", [("flash", 9), ("paged", 12), ("section", 13), ("append", 12), ("append_seq", 6), ("gather", 4),
                                    ("int8", 4)])
def test_other_arguments_are_handed_back(name, n):
    fn = getattr(_lib.host(), name)
    t = torch.zeros(1, 2, 4, 16, dtype=torch.float16)

    class Sub(torch.Tensor):
        pass

    for x in (None, 3, "q", t, t.as_subclass(Sub), t.to_sparse()):
        assert fn(*([x] * n)) is None
    assert fn() is None and fn(t) is None


def test_refusals_are_unchanged():
    x = torch.zeros(2, 16, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="requires CUDA tensors"):
        int8_matmul(x, torch.zeros(4, 16, dtype=torch.int8), torch.zeros(4))
