"""The cut search by groups of 16 lanes, as the device runs it (csrc/p2p_cut.h,
host build): its probes at task indices near 2^30 and up to 2^31 - 1, rows of a few
probes and of a partial last round, and each group's own bits of the wave's vote.
It must give what a sequential scan of the row gives.  No device is used."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "libcuthost.so")
IMAX = 2 ** 31 - 1


@pytest.fixture(scope="module")
def cut():
    lib = ctypes.CDLL(LIB)
    i32, i64, vp = ctypes.c_int, ctypes.c_longlong, ctypes.c_void_p
    lib.cut_var_scan.argtypes = [i32, i32, i64, i64]
    lib.lanes_const.argtypes = [vp, vp, i64, i64, ctypes.c_uint, vp]
    lib.lanes_var.argtypes = [vp, vp, i64, i64, vp]
    return lib


def _rows(beg, lengths):
    b = np.array([min(beg + 7 * k, IMAX - 1) for k in range(4)], np.int32)
    e = np.array([min(int(x) + n, IMAX) for x, n in zip(b, lengths)], np.int32)
    return b, e


@pytest.mark.parametrize("beg", [0, 12345, 2 ** 30 - 7, 2 ** 30 + 98765, 1_650_000_000, 2 ** 31 - 5000, IMAX - 40])
@pytest.mark.parametrize("lengths", [(1, 2, 15, 16), (17, 18, 255, 256), (257, 273, 4000, 4097)])
def test_constant_sizes(cut, beg, lengths):
    b, e = _rows(beg, lengths)
    out = np.zeros(4, np.int32)
    for size, wi, split in [(64, 64, 1 << 22), (37, 192, 1 << 22), (1, 1, 100), (64, 1, 1 << 14), (50, 50, 10 ** 12), (64, 64, 1)]:
        cut.lanes_const(b.ctypes.data, e.ctypes.data, wi, split, size, out.ctypes.data)
        want = [min(int(y), max(int(x) + 1, int(x) + split // (size * wi))) for x, y in zip(b, e)]
        assert out.tolist() == want, (beg, size, wi, split)


@pytest.mark.parametrize("beg", [0, 2 ** 30 - 300, 1_650_000_000, IMAX - 3000])
def test_variable_sizes_equal_the_sequential_scan(cut, beg):
    b, e = _rows(beg, (3, 300, 1500, 2500))
    out = np.zeros(4, np.int32)
    for wi, split in [(64, 1 << 16), (64, 1 << 20), (3, 5000), (192, 1 << 22), (1, 1 << 40)]:
        cut.lanes_var(b.ctypes.data, e.ctypes.data, wi, split, out.ctypes.data)
        assert out.tolist() == [cut.cut_var_scan(int(x), int(y), wi, split) for x, y in zip(b, e)]


def test_a_whole_row_to_the_int_limit(cut):
    """One row of 2^31 - 2 tasks: the probes' spacing and their offsets pass 2^27 and 2^31."""
    b, e = np.full(4, 1, np.int32), np.full(4, IMAX, np.int32)
    out = np.zeros(4, np.int32)
    for split in (1, 10 ** 6, 2 ** 30, 2 ** 31 - 3, 2 ** 31, 2 ** 40):
        cut.lanes_const(b.ctypes.data, e.ctypes.data, 1, split, 1, out.ctypes.data)
        assert out.tolist() == [min(IMAX, max(2, 1 + split))] * 4, split
