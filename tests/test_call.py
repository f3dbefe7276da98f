"""hip.call's packed p[] and s[] hold what two padded ctypes arrays would, for every form it takes (no GPU)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from nanocompile_amd import hip


class Array:
    def __init__(self, ptr):
        self.ptr = ptr


@pytest.mark.parametrize("pointers,sizes", [
    ([], []), ([None, 5, Array(1 << 47)], [1, np.int64(2), True, -3]), ((7,), (1.9, np.float32(2.0))),
    (list(range(1, 17)), list(range(16))), (list(range(1, 21)), list(range(-4, 14))), ([0, -8], [2 ** 63, -2 ** 63]),
    ([], [np.array(2.0), np.array(3), np.float64(4.0)])])
def test_arguments(monkeypatch, pointers, sizes):
    seen = []
    # a c_char_p argument is the bytes object itself, not its text up to the first zero
    monkeypatch.setitem(hip._KERNELS, "probe", lambda p, s: seen.append((p, s)) or 0)
    monkeypatch.setattr(hip, "_DEVICE", 0)
    hip.call("probe", pointers, sizes)
    p = (ctypes.c_void_p * max(hip.PAD, len(pointers)))(*[hip._address(x) for x in pointers])
    s = (ctypes.c_int64 * max(hip.PAD, len(sizes)))(*[int(v) for v in sizes])
    assert seen == [(bytes(p), bytes(s))]
