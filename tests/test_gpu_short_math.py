"""GPU: the walk's short square root and reciprocal are correctly rounded for every
float of [2^-100, 2^126), the range that walk_short and solo_walker use them in
(short_math_check.hip, which __graft_entry__.build() compiles)."""
import ctypes as C
import os

import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libshort_math_check.so")


def test_every_float_of_the_range(shy):
    L = C.CDLL(LIB)
    out = (C.c_ulonglong * 3)()
    print("short arithmetic", flush=True)
    assert L.short_math_check(out) == 0
    assert list(out) == [226 << 23, 0, 0]
