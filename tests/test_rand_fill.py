"""Factor initialisation draws (CPU only): long fills run on the generator's
own state and must give rand()'s values, leave the sequence where as many
rand() calls would, and keep working for callers with their own state."""
import ctypes as C
import threading
import time

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


def _sequence(seed, n):
    """The first n values of the sequence that srand(seed) starts."""
    L = ps.lib()
    L.spd_serve_rand_fill.restype = None
    L.spd_serve_rand_fill.argtypes = [C.c_uint, C.c_void_p, C.c_uint64]
    out = np.empty(n)
    L.spd_serve_rand_fill(seed, out.ctypes.data, n)
    return out


def test_seed_during_a_fill():
    # a seed that another thread sets while a fill runs is the process's
    # seed: what is drawn next is from its sequence
    libc = C.CDLL(None)
    n = 4000000
    seq = _sequence(12345, n + 200)
    _fill(8)
    during = 0
    for attempt in range(20):
        libc.srand(C.c_uint(7))
        t = {}

        def fill():
            t["begin"] = time.perf_counter()
            _fill(n)
            t["end"] = time.perf_counter()
        th = threading.Thread(target=fill)
        th.start()
        time.sleep(0.002)
        t["seed"] = time.perf_counter()
        libc.srand(C.c_uint(12345))
        seeded = time.perf_counter()
        th.join()
        if not t["begin"] + 1e-3 < t["seed"] < seeded < t["end"]:
            continue
        during += 1
        nxt = _fill(20)
        at = np.flatnonzero(seq == nxt[0])
        assert any(np.array_equal(seq[k:k + 20], nxt) for k in at)
        if during == 3:
            break
    assert during


def test_fills_on_two_threads_share_the_sequence():
    # long fills on one thread, short ones on another: every fill is a stretch
    # of the one sequence, none is drawn twice and none is left out
    libc = C.CDLL(None)
    _fill(8)
    libc.srand(C.c_uint(3))
    blocks = []

    def work(sizes):
        for k in sizes:
            blocks.append(_fill(k))
    th = [threading.Thread(target=work, args=([200000] * 12,)),
          threading.Thread(target=work, args=([32, 63, 5, 700] * 300,))]
    for x in th:
        x.start()
    for x in th:
        x.join()
    blocks.append(_fill(10))
    total = sum(len(b) for b in blocks)
    seq = _sequence(3, total)
    at = {}
    for k, v in enumerate(seq):
        at.setdefault(v, []).append(k)
    used = np.zeros(total, dtype=bool)
    for b in blocks:
        k = next(k for k in at.get(b[0], [])
                 if not used[k] and np.array_equal(seq[k:k + len(b)], b))
        assert not used[k:k + len(b)].any()
        used[k:k + len(b)] = True
    assert used.all()


def test_draws_beside_a_fill():
    # a thread that begins to draw while a fill runs gets draws of the
    # sequence, and the sequence goes on after exactly as many
    libc = C.CDLL(None)
    _fill(8)
    n = 1500000
    during = 0
    for attempt in range(20):
        libc.srand(C.c_uint(11))
        t = {}

        def fill():
            t["begin"] = time.perf_counter()
            _fill(n)
            t["end"] = time.perf_counter()
        th = threading.Thread(target=fill)
        th.start()
        time.sleep(0.002)
        t["draw"] = time.perf_counter()
        drawn = [libc.rand() for _ in range(2000)]
        th.join()
        nxt = [libc.rand() for _ in range(8)]
        if not t["begin"] + 1e-3 < t["draw"] < t["end"]:
            continue
        during += 1
        libc.srand(C.c_uint(11))
        seq = [libc.rand() for _ in range(2 * n + len(drawn) + 8)]
        assert set(drawn) <= set(seq)
        assert nxt == seq[-8:]
        if during == 2:
            break
    assert during


def test_fill_of_thousands_from_a_callers_state():
    # long enough to draw from a copy: a caller's own TYPE_3 state stays
    # current, advances, and keeps its place when the caller switches away
    # from it and back
    libc = C.CDLL(None)
    libc.initstate.restype = C.c_void_p
    libc.setstate.restype = C.c_void_p
    libc.setstate.argtypes = [C.c_void_p]
    for size in (32, 128, 256):
        mine = C.create_string_buffer(size)
        before = libc.initstate(C.c_uint(9), mine, C.c_size_t(size))
        try:
            want = _rand_values(libc, 5000)
            after = libc.rand()
            libc.srand(C.c_uint(9))
            assert np.array_equal(_fill(5000), want)
            assert libc.setstate(before) == C.addressof(mine)
            libc.rand()
            libc.setstate(C.addressof(mine))
            assert libc.rand() == after
        finally:
            libc.setstate(before)
