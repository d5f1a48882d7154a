"""Values beside a halfway case in the parallel sequential sum (csrc/p2p_seqsum.h,
host build): one unit in the last place above or below half a unit of the sum,
which the rule must not take for halfway, and the halfway values themselves, on
sums of both signs and parities.  No device is used."""
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


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("start", [2.0 ** 52 + 2, 2.0 ** 52 + 3, 2.0 ** 52 + 4095])
@pytest.mark.parametrize("half", [0.5, 1.5, 2.5, -0.5, -1.5, -2.5])
def test_beside_halfway(lib, start, half, sign):
    for v in (np.nextafter(half, -np.inf), half, np.nextafter(half, np.inf)):
        x = sign * np.array([start, v, v, -v, v])
        want = lib.seqsum_loop(x.ctypes.data, x.size)
        acc = ctypes.c_longlong(0)
        for batch in (1, 2, 5):
            got = lib.seqsum_batches(x.ctypes.data, x.size, batch, ctypes.byref(acc))
            assert got == want, (start, v, batch, got, want)
