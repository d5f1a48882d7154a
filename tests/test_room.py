"""Reservations ahead of need (csrc/p2p_room.h, host build): less is asked for
when memory runs out, down to what is needed, and never after another error.  No
device is used."""
import ctypes
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "libroomhost.so")
OUT_OF_MEMORY, OTHER = 2, 1                  # hipErrorOutOfMemory, hipErrorInvalidValue


@pytest.fixture(scope="module")
def lib():
    h = ctypes.CDLL(LIB)
    i64 = ctypes.c_longlong
    h.room_reserve.argtypes = [i64, i64, i64, ctypes.c_int, ctypes.POINTER(i64), ctypes.POINTER(ctypes.c_int)]
    h.room_modest.argtypes = [i64, i64, i64]
    h.room_modest.restype = i64
    return h


def _ask(lib, want, least, room, error=OUT_OF_MEMORY):
    asked, n = (ctypes.c_longlong * 80)(), ctypes.c_int(0)
    return lib.room_reserve(want, least, room, error, asked, ctypes.byref(n)), list(asked[: n.value])


@pytest.mark.parametrize("want,least,room,asked", [
    (1000, 10, 1000, [1000]), (1000, 10, 999, [1000, 500]), (1000, 10, 130, [1000, 500, 250, 125]),
    (1000, 300, 400, [1000, 500, 300]), (1000, 1000, 1 << 40, [1000]), (5, 1000, 1 << 40, [1000])])
def test_reserves_what_fits(lib, want, least, room, asked):
    assert _ask(lib, want, least, room) == (0, asked)


def test_fails_where_the_least_does_not_fit(lib):
    e, asked = _ask(lib, 1 << 40, 7, 6)
    assert e == OUT_OF_MEMORY and asked[-1] == 7 and len(asked) < 60
    assert _ask(lib, 1000, 7, 500, OTHER) == (OTHER, [1000])


def test_first_reservation_leaves_room(lib):
    assert lib.room_modest(1000, 17, 1 << 30) == 1000
    assert lib.room_modest(1 << 32, 17, 16 << 30) == (4 << 30) // 17
    assert lib.room_modest(1000, 17, 0) == 0
