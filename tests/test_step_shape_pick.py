"""The autotuner keeps the shape it measured fastest (no GPU needed: its choice
is host code of the library)."""
import ctypes as C

import numpy as np
import pytest

from hidem_amd import _abi as A

# us per step of the 8M slab's FP64 form in launch order (3) and in a range per XCD (0)
SLAB = [2440.0, 2700.0, 2450.0, 2423.0, 2710.0, 2460.0, 2800.0]


def pick(us):
    f = A.lib()["_ZN3hdm17pick_step_variantEPKd"]
    f.argtypes, f.restype = [C.POINTER(C.c_double)], C.c_int
    ms = np.asarray(us, dtype=np.float64) * 1e-3
    return f(ms.ctypes.data_as(C.POINTER(C.c_double)))


def test_fastest_by_less_than_a_percent():
    assert pick(SLAB) == 3


@pytest.mark.parametrize("fastest", range(7))
def test_fastest_of_all(fastest):
    us = [100.0 + v for v in range(7)]
    us[fastest] = 99.5
    assert pick(us) == fastest


def test_first_of_equals():
    assert pick([50.0] * 7) == 0
