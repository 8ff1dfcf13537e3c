"""The short reciprocals and quotients that the batched traversal uses equal the
correctly rounded division: reciprocals for every float, quotients for corner
significands at the ends of the declared ranges and for random operands."""
import ctypes as C
import os

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def check(what, n=0, seed=0):
    path = os.path.join(ROOT, "tests", "libmath_check.so")
    if not os.path.exists(path):
        from happyray_amd import build
        build.build_checks()
    lib = C.CDLL(path)
    lib.math_check.argtypes = [C.c_int, C.c_ulonglong, C.c_ulonglong, C.POINTER(C.c_ulonglong)]
    out = (C.c_ulonglong * 2)()
    assert lib.math_check(what, n, seed, out) == 0
    assert out[0] == 0, f"{out[0]} mismatches, one at {out[1] >> 32:#010x}, {out[1] & 0xFFFFFFFF:#010x}"


def test_reciprocals_of_every_float():
    check(0)


def test_quotients_of_corner_operands():
    check(1)


@pytest.mark.parametrize("seed", [1, 2])
def test_quotients_of_random_operands(seed):
    check(2, 1 << 31, seed * 0x123456789)
