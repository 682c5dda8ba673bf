"""Factor initialisation draws (CPU only): long fills run on the generator's
own state and must give rand()'s values, leave the sequence where as many
rand() calls would, and keep working for callers with their own state."""
import ctypes as C

import numpy as np
import pytest

import pysplatt as ps

RAND_MAX = 2147483647


def _fill(n):
    L = ps.lib()
    L.spl_fill_rand.restype = None
    L.spl_fill_rand.argtypes = [C.c_void_p, C.c_uint64]
    out = np.empty(n)
    L.spl_fill_rand(out.ctypes.data, n)
    return out


def _rand_values(libc, n):
    out = np.empty(n)
    for i in range(n):
        a, b = libc.rand(), libc.rand()
        v = 3.0 * (a / RAND_MAX)
        out[i] = -v if b % 2 == 0 else v
    return out


@pytest.mark.parametrize("seed", [1, 4, 20261204])
def test_fill_continues_the_rand_sequence(seed):
    ps.lib()
    libc = C.CDLL(None)
    sizes = [1, 63, 64, 65, 500, 3, 4097]
    libc.srand(C.c_uint(seed))
    want = [_rand_values(libc, n) for n in sizes]
    after = [libc.rand() for _ in range(50)]
    libc.srand(C.c_uint(seed))
    for n, w in zip(sizes, want):
        assert np.array_equal(_fill(n), w)
    assert [libc.rand() for _ in range(50)] == after


@pytest.mark.parametrize("size", [8, 32, 64, 256])
def test_fill_from_a_callers_state(size):
    # a caller's own state of every generator type stays current and advances
    libc = C.CDLL(None)
    libc.initstate.restype = C.c_void_p
    libc.setstate.restype = C.c_void_p
    libc.setstate.argtypes = [C.c_void_p]
    mine = C.create_string_buffer(size)
    before = libc.initstate(C.c_uint(9), mine, C.c_size_t(size))
    try:
        want = _rand_values(libc, 200)
        after = libc.rand()
        libc.srand(C.c_uint(9))
        assert np.array_equal(_fill(200), want)
        assert libc.rand() == after
    finally:
        libc.setstate(before)
