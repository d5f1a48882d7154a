"""Copies between host arrays and the device (csrc/host_pipe.h) over a stand-in
for the runtime: every byte arrives, pageable arrays go through the ring from
4 MiB on, pinned ones straight.  No device is used."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "libpipehost.so")
MIB = 1 << 20


@pytest.fixture(scope="module")
def lib():
    h = ctypes.CDLL(LIB)
    h.pipe_without_pinning.argtypes = [ctypes.c_longlong]
    h.pipe_copies.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_size_t, ctypes.c_void_p]
    return h


def _copies(lib, sizes, pinned, shift=0):
    n, out = np.array(sizes, np.int64), np.zeros(4, np.int64)
    assert lib.pipe_copies(n.ctypes.data, n.size, int(pinned), shift, out.ctypes.data) == 0
    return dict(zip(("copies", "user", "allocs", "bytes"), out.tolist()))


@pytest.mark.parametrize("n", [1, 4 * MIB - 1, 4 * MIB, 4 * MIB + 1, 5 * MIB + 4097, 8 * MIB, 8 * MIB + 1, 31 * MIB + 12345])
def test_pageable_arrays_are_staged(lib, n):
    c = _copies(lib, [n], False)
    if n < 4 * MIB:
        assert c["copies"] == c["user"] == 2 and c["allocs"] == 0
    else:
        assert c["user"] == 0 and c["copies"] >= 8


@pytest.mark.parametrize("shift", [0, 4, 4096])
@pytest.mark.parametrize("n", [1, 4 * MIB - 1, 4 * MIB, 8 * MIB + 1, 31 * MIB + 12345])
def test_pinned_arrays_go_straight(lib, n, shift):
    c = _copies(lib, [n, n], True, shift)
    assert c == {"copies": 4, "user": 4, "allocs": 0, "bytes": 0}


def test_the_ring_is_allocated_once(lib):
    """A longer copy after a first one finds the ring: pinning it again, at its new
    size, costs as much as the first time."""
    c = _copies(lib, [4 * MIB, 5 * MIB, 9 * MIB, 7 * MIB, 64 * MIB], False)
    assert c["allocs"] == 1 and c["bytes"] <= 8 * MIB


@pytest.mark.parametrize("n", [1, 100, 349525, 349526, 1000003])
def test_where_nothing_can_be_pinned(lib, n):
    """The copies are then the runtime's, records are packed in ordinary memory."""
    assert lib.pipe_without_pinning(n) == 0
