"""Spectral derivatives over axis lengths where a transform plan can go wrong:
every radix from 2 to 16 in the first, inner and middle pass, two to four
passes, passes in several rounds, lengths with other factors, odd numbers of
lines (a pair without a partner), row pitches that do and do not allow vector
accesses, grids with one and with two pairs a thread.

A few steps of the SH solver without layers against its numpy oracle; the
spectral derivative spreads the source over every wave number, so the fields
hold each frequency of both axes.  A transform of n points carries a relative
rounding error of a few eps log2(n) (Cooley-Tukey with exact twiddles); eight
derivatives a step in sequence and two transforms each over 3 steps stay
below 100 eps log2(n).
"""
import math

import numpy as np
import pytest
from tolerances import note

from oracle import oracle_sh as S
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

# (nx, nz): two passes at the small end, three and four passes
SIZES = [(4, 6), (9, 4), (10, 15), (21, 22), (26, 35), (48, 39), (49, 64), (99, 60), (121, 96), (117, 130),
         (143, 154), (165, 168), (196, 210), (225, 256), (343, 36), (14, 1001), (1029, 10), (2048, 9), (12, 2197),
         (3003, 8), (6, 4096), (300, 308),
         # FP32 passes in several rounds, the other axis in one, in several, or padded; 2000 points in one
         # round of radices that are not the cheapest
         (1617, 6), (5, 2187), (17, 2662), (3402, 4), (1701, 1617), (2000, 7),
         # other factors: padded lines (2 to 5 points, primes, a prime squared, odd and even)
         (2, 3), (3, 5), (17, 7), (13, 11), (34, 33), (289, 38), (363, 469), (1021, 6), (5, 2039), (204, 418)]


def run(ctx, nx, nz, storage):
    from seismod_amd.solver import ShConfig, ViscoelasticSH
    rng = np.random.default_rng(nx * 10000 + nz)
    h, f0, steps = 10.0, 25.0, 3
    vs = rng.uniform(1200, 2500, (nx, nz))
    rho = rng.uniform(1800, 2600, (nx, nz))
    gamma, Q, f = rng.uniform(0, 0.3, (nx, nz)), rng.uniform(15, 80, (nx, nz)), rng.uniform(10, 40, (nx, nz))
    mu = vs * vs * rho * 1e-9
    dt = 0.15 * h / 2500.0
    types = np.array([S.SYZ, S.SXY], np.intc)
    idx = np.array([(nx // 2) * nz + nz // 2, (nx // 3) * nz + nz // 3], np.uintp)
    L, fct = O.source_functions([1.0, 0.7], [f0, f0], 0.5 * dt)
    s = ViscoelasticSH(ctx, ShConfig(nx=nx, nz=nz, np=0, dx=h, dz=h, dt=dt, f0=f0, abs=False, storage=storage),
                       mu, rho, gamma, Q, f)
    s.set_sources(types, idx, L, fct)
    s.run(steps)
    got = np.stack([s.field(k) for k in ("txy", "tyz", "vy")])
    s.close()
    off = np.concatenate([[0], np.cumsum(L)]).astype(np.int64)
    src = [(int(t), int(i), fct[off[k]:off[k + 1]]) for k, (t, i) in enumerate(zip(types, idx))]
    cfg = dict(nx=nx, nz=nz, np=0, dx=h, dz=h, dt=dt, alpha_max=math.pi * f0, iwipe=0)
    _, W = S.sh_run(cfg, mu, rho, gamma, Q, f, src, idx[:1], np.array([S.VY]), steps)
    return got, W[:3]


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_derivatives_of_every_length(ctx, size, storage):
    from seismod_amd.solver import pstd_plan
    # no length here goes through hipFFT, but for the longest in FP64
    assert all(pstd_plan(n, storage)[0] or (storage == "f64" and n > 2048) for n in size)
    got, want = run(ctx, *size, storage)
    eps = 2.0 ** -52 if storage == "f64" else 2.0 ** -23
    tol = 100 * eps * math.log2(max(size))
    for k in range(3):
        # a grid of two rows has no interior node: v_y stays 0
        e = float(np.linalg.norm(got[k] - want[k]) / (np.linalg.norm(want[k]) or 1.0))
        note("pstd_lengths", size=f"{size[0]}x{size[1]}", storage=storage, field=k, error=e, tol=tol)
        assert e < tol and (np.abs(want[k]).max() > 0 or min(size) < 3), (k, e, tol)
