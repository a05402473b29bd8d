"""A scattering takes its random words together: the same words in the same
order as one at a time, from every number of words left over and for every
number asked for."""
import ctypes as C
import itertools
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_build", "librng_host.so")
pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="host harness not built")


def compare(calls, packet=5):
    lib = C.CDLL(LIB)
    n = np.asarray(calls, np.int32)
    return lib.rng_take_compare(C.c_uint32(0x12345678), C.c_uint32(0x9ABCDEF0), C.c_uint32(3), C.c_uint64(packet),
                                n.ctypes.data_as(C.POINTER(C.c_int)), len(n))


@pytest.mark.parametrize("left", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4])
def test_every_remainder(left, n):
    # 4 - left single words leave `left` of the first block, then n, then all of 1..4 again
    for tail in itertools.product([1, 2, 3, 4], repeat=3):
        assert compare([left - 4, n, *tail, -2]) == -1, tail


def test_long_mixed_sequences():
    rng = np.random.default_rng(1)
    for k in range(50):
        assert compare(rng.integers(-3, 5, 400), packet=int(rng.integers(0, 1 << 40))) == -1
