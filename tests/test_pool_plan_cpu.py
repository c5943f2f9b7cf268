"""Sizes of the path pool and the results ring."""
import ctypes as C

import numpy as np
import pytest

from conftest import load_testkernels

RING = 1 << 27


def _sizes(jobs, wanted=0):
    L = load_testkernels()
    n = np.array([j[0] for j in jobs], np.uint32)
    px = np.array([j[1] for j in jobs], np.uint64)
    out = np.zeros(3, np.uint32)
    L.tk_pool_sizes(n.ctypes.data_as(C.c_void_p), px.ctypes.data_as(C.c_void_p), C.c_uint32(len(jobs)),
                    C.c_uint32(wanted), out.ctypes.data_as(C.c_void_p))
    return tuple(int(x) for x in out)


@pytest.mark.parametrize("first", [1, 64, 1000003, RING // 2 + 1, RING + 5])
@pytest.mark.parametrize("other", [1, 999983, RING // 3, RING + 77, 0x7FFFFFFF])
@pytest.mark.parametrize("samples", [1, 3, 200])
def test_ring_holds_a_sample_of_every_job(first, other, samples):
    """A batch that starts with a small film and holds a large one: renderJobs
    refuses a ring smaller than one sample of any job."""
    paths, ring, _ = _sizes([(samples, first), (1, other)])
    assert ring >= max(first, other)
    total = samples * first + other
    assert ring <= max(total, 1) and ring <= max(RING, first, other)
    assert paths == min(1 << 24, max(total, 1 << 16))


def test_pool_wanted_is_an_upper_limit():
    assert _sizes([(1, 100)], wanted=7)[:2] == (7, 100)
    assert _sizes([(64, 1 << 20)], wanted=1 << 10)[0] == 1 << 10


def test_training_records_are_bounded():
    """192 B each: a call trains on 2^20 paths or one sample of the film, and a
    film of 2^30 pixels must not take 200 GB for them."""
    M = 1 << 20
    assert _sizes([(7, 150000)])[2] == 1050000
    assert _sizes([(1, 64 * M)])[2] == 64 * M
    assert _sizes([(1, 1024 * M)])[2] == 64 * M
    assert _sizes([(1, 8 * M)], wanted=M)[2] == 4 * M
    assert _sizes([(1, 8 * M)], wanted=7)[2] == M
    assert _sizes([(1, 5)], wanted=7)[2] == 5


def test_autotuner_tries_the_default_pool():
    """A scene whose pool was set smaller can be tuned back to what an untuned
    scene has."""
    out = np.zeros(8, np.uint32)
    n = load_testkernels().tk_tuned_slots(out.ctypes.data_as(C.c_void_p))
    tried = [int(x) for x in out[:n]]
    assert _sizes([(1, 1 << 30)])[0] in tried and tried == sorted(tried)


def _halving(paths, ring, film, free, error_at=0):
    L = load_testkernels()
    out = np.zeros(3, np.uint32)
    rc = L.tk_alloc_halving(C.c_uint32(paths), C.c_uint32(ring), C.c_uint64(film), C.c_uint64(free),
                            C.c_uint32(error_at), out.ctypes.data_as(C.c_void_p))
    return rc, tuple(int(x) for x in out)


def test_pool_is_halved_until_it_fits():
    M = 1 << 20
    assert _halving(16 * M, 128 * M, 5 * M, 1 << 40) == (0, (16 * M, 128 * M, 1))
    assert _halving(16 * M, 128 * M, 5 * M, 300 * 4 * M + 48 * 32 * M) == (0, (4 * M, 32 * M, 3))
    # not below 2^20 paths and one sample of the largest film
    assert _halving(16 * M, 128 * M, 5 * M, 300 * M + 48 * 5 * M) == (0, (M, 5 * M, 6))
    assert _halving(16 * M, 128 * M, 5 * M, 300 * M + 48 * 5 * M - 1) == (1, (0, 0, 6))
    assert _halving(100, 7, 7, 1000) == (1, (0, 0, 1))


@pytest.mark.parametrize("error_at", [1, 2, 3])
def test_other_errors_are_not_a_shortage(error_at):
    """A lost device or a failed launch is reported, not answered by asking
    for less."""
    M = 1 << 20
    assert _halving(16 * M, 128 * M, M, 300 * M + 48 * M, error_at) == (2, (0, 0, error_at))


def _fit(calls):
    """calls: (paths, ring, film, bytes left to the pool, regrow)."""
    L = load_testkernels()
    cols = [np.array([c[k] for c in calls], t) for k, t in enumerate((np.uint32, np.uint32, np.uint64, np.uint64,
                                                                      np.uint32))]
    out = np.zeros((len(calls), 3), np.uint32)
    L.tk_pool_fit(*(a.ctypes.data_as(C.c_void_p) for a in cols), C.c_uint32(len(calls)),
                  out.ctypes.data_as(C.c_void_p))
    return [tuple(int(x) for x in r) for r in out]


def test_a_passing_shortage_passes():
    M, G = 1 << 20, 1 << 30
    whole = (16 * M, 128 * M, M)
    # short, still short, a little more free, enough again, then kept
    got = _fit([whole + (4 * G, 0), whole + (4 * G, 0), whole + (5 * G, 0), whole + (20 * G, 0), whole + (4 * G, 0)])
    assert got[0] == (4 * M, 32 * M, 3)
    assert got[1] == got[2] == (4 * M, 32 * M, 0)
    assert got[3] == (16 * M, 128 * M, 1)
    assert got[4] == (16 * M, 128 * M, 0)


def test_pool_grows_and_is_kept():
    M, G = 1 << 20, 1 << 30
    got = _fit([(M, M, 100, 100 * G, 0), (M // 2, M, 100, 100 * G, 0), (2 * M, M // 2, 100, 100 * G, 0),
                (M, M, 100, 100 * G, 1)])
    assert got == [(M, M, 1), (M, M, 0), (2 * M, M, 1), (2 * M, M, 1)]


def test_short_pool_still_serves_what_it_must():
    """A larger film than the short ring holds, and buffers of another kind,
    are allocated again whatever is free; a call that cannot be served at all
    leaves no pool behind, and the next one starts afresh."""
    M, G = 1 << 20, 1 << 30
    whole = (16 * M, 128 * M, M)
    got = _fit([whole + (4 * G, 0), (16 * M, 128 * M, 40 * M, 4 * G, 0), whole + (4 * G, 1), whole + (M, 1),
                whole + (20 * G, 0)])
    assert got[0] == (4 * M, 32 * M, 3)
    assert got[1] == (4 * M, 40 * M, 3)
    assert got[2] == (4 * M, 32 * M, 3)
    assert got[3][:2] == (0, 0)
    assert got[4] == (16 * M, 128 * M, 1)
