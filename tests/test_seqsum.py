"""The parallel form of a sequential FP64 sum (csrc/p2p_seqsum.h), compiled for
the host: whatever the batch size, it must give the plain loop's result bit for
bit, and accept most values in batches where the sum is long.  No device is
used."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "libseqsumhost.so")


@pytest.fixture(scope="module")
def lib():
    h = ctypes.CDLL(LIB)
    h.seqsum_batches.restype = h.seqsum_loop.restype = ctypes.c_double
    h.seqsum_batches.argtypes = [ctypes.c_void_p, ctypes.c_longlong, ctypes.c_longlong, ctypes.POINTER(ctypes.c_longlong)]
    h.seqsum_loop.argtypes = [ctypes.c_void_p, ctypes.c_longlong]
    return h


def _values(kind, n, g):
    grid = g.integers(0, 1 << 30, n).astype(np.float64)
    if kind == "grid":
        return 1.0000000937e-7 * grid
    if kind == "signed":                             # crosses zero often
        return 3.7e-8 * (grid - (1 << 29))
    if kind == "ghosts":                             # mostly positive, some below zero
        return 3.7e-8 * (grid - (1 << 26))
    if kind == "negative":
        return -1.1e-7 * grid
    if kind == "lattice":                            # a grid step of few bits: halfway cases in every long sum
        return grid * (138.671875 / (1 << 30))
    if kind == "halves":                             # 53-bit values, odd last bits
        return np.ldexp(2.0 ** 52 + 2 * g.integers(0, 1 << 20, n) + 1.0, -52)
    if kind == "powers":
        return np.ldexp(1.0, g.integers(-60, 60, n)) * np.where(g.random(n) < 0.3, -1.0, 1.0)
    if kind == "zeros":
        return np.where(g.random(n) < 0.9, 0.0, 1e-3 * grid)
    if kind == "coincident":
        return np.full(n, 1e-7 * 123456789.0)
    v = 1e-7 * grid
    v[n // 2] = np.inf if kind == "inf" else 1e300
    return v


@pytest.mark.parametrize("kind", ["grid", "lattice", "signed", "ghosts", "negative", "halves", "powers", "zeros", "coincident",
                                  "inf", "huge"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 513, 4097, 100003])
def test_equals_the_plain_loop(lib, kind, n):
    v = np.ascontiguousarray(_values(kind, n, np.random.default_rng(n)))
    want = lib.seqsum_loop(v.ctypes.data, n)
    acc = ctypes.c_longlong(0)
    for batch in (1, 64, 512, 4096):
        got = lib.seqsum_batches(v.ctypes.data, n, batch, ctypes.byref(acc))
        assert np.float64(got).tobytes() == np.float64(want).tobytes(), (batch, got, want)
    if kind in ("grid", "lattice", "halves") and n > 100000:
        assert acc.value > 0.9 * n
