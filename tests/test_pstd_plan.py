"""Which transform the pseudo-spectral solvers take for an axis of n points
(chosen on the host, no GPU): hand-written over n points, over a padded line,
or hipFFT.

A length without a factor above 13 has radices up to 16.  One round of 512
threads needs every radix to be at least n / 512; a line of at most 28 KiB of
complex values may also take its passes in several rounds, and one of more
than 40 KiB has such radices only if they are the cheapest.  A length with
another factor is padded to at least 2 n - 1 points that one round takes.
"""
from functools import lru_cache

import pytest


def smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


@lru_cache(None)
def factors(n, least, most=16, passes=0):
    """n as 2 to 6 radices from least to 16"""
    if n == 1:
        return passes >= 2
    return passes < 6 and any(n % r == 0 and factors(n // r, least, r, passes + 1)
                              for r in range(min(most, n), least - 1, -1))


@pytest.mark.parametrize("storage,elt", [("f32", 4), ("f64", 8)])
def test_path_of_every_length(storage, elt):
    from seismod_amd.solver import pstd_plan
    for n in range(2, 5000):
        points, rounds = pstd_plan(n, storage)
        if factors(n, max(2, -(-n // 512))):
            assert (points, rounds) == (n, 1) or (2 * n * elt > 40 * 1024 and points == 0), n
        elif factors(n, 2) and 2 * n * elt <= 28 * 1024:
            assert points == n and rounds > 1, n
        elif n <= 2048:
            assert 2 * n - 1 <= points <= 4096 and smooth(points) and rounds == 1, n
        else:
            assert points == 0, n


def test_ordinary_long_axes():
    """Every length without a factor above 13 up to 3402 points in FP32 and
    1694 in FP64 is hand-written, however many threads its passes ask for."""
    from seismod_amd.solver import pstd_plan
    for n in (1617, 1944, 2000, 2187, 2662, 3000, 3003, 3159, 3200, 3402):
        assert pstd_plan(n, "f32")[0] == n
    assert pstd_plan(2000, "f32") == (2000, 1) and pstd_plan(3000, "f32") == (3000, 2)
    for n in (1617, 1694, 1600, 2000, 2376, 2560, 4096):
        assert pstd_plan(n, "f64")[0] == n
    # long lines whose cheapest radices do not fit one round
    for n in (2592, 2916, 3430):
        assert pstd_plan(n, "f64")[0] == 0
    assert pstd_plan(3430, "f32") == (3430, 1) and pstd_plan(4096, "f32") == (4096, 1)
    for storage, most in (("f32", 3402), ("f64", 1694)):
        for n in range(14, most + 1):
            if smooth(n):
                assert pstd_plan(n, storage)[0] == n


def test_refused_arguments():
    from seismod_amd import _lib as L
    import ctypes as C
    p, r = C.c_int(), C.c_int()
    assert L.lib.sm_pstd_plan(0, L.SM_STORE_F32, C.byref(p), C.byref(r)) == L.SM_ERR_ARG
    assert L.lib.sm_pstd_plan(64, L.SM_STORE_BF16, C.byref(p), C.byref(r)) == L.SM_ERR_ARG
    assert L.lib.sm_pstd_plan(64, L.SM_STORE_F32, None, C.byref(r)) == L.SM_ERR_ARG
