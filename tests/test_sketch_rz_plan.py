"""Scratch memory of the sketch's R and z: one copy of the sketch, whichever form runs."""
import ctypes

import pytest

from parla_amd import _lib


@pytest.mark.parametrize("n", [64, 257, 1024])
def test_scratch_is_one_copy_of_the_sketch(n):
    lib = _lib.load()

    def query(d):
        b = ctypes.c_int64(0)
        assert lib.pamd_sketch_rz_workspace(d, n, ctypes.byref(b)) == 0
        return b.value

    # d large enough that the products' split over K, and its scratch, no longer grow with d
    d1, d2 = 1 << 20, 1 << 22
    assert query(d2) - query(d1) <= 8 * ((n + 1) * (d2 - d1) + 64)
