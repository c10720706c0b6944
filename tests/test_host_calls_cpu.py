"""The compiled call layer (csrc/host.cpp) without a GPU: it binds entry points
the library exports, and hands every argument it does not take back to the
Python functions (None), which refuse it with their own errors."""

from __future__ import annotations

import struct

import pytest
import torch

from engine import _lib
from engine.quant import int8_matmul


def test_binds_exported_entry_points():
    assert set(_lib.host().names()) <= set(_lib.EXPORTED_SYMBOLS)


def test_extension_has_no_thread_local_storage():
    """A library loaded with thread-local storage that no call touches slows
    every thread-local access of the process (see build_lib.py)."""
    with open(_lib.HOST_PATH, "rb") as f:
        elf = f.read()
    phoff, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, phoff + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS


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
