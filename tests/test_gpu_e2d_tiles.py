"""Several FP32 2D steps per launch (halos recomputed in registers) against
the same steps run one launch each: the expressions are the same, so the
results are compared bit for bit.  A run of one step always takes the
one-step kernel (its forms and launch shapes: test_gpu_e2d_fused.py).

Grids around the tile's edges (owned rows and columns depend on the number of
steps of a launch), layers thinner and thicker than a wave's rows, step
counts that leave a short last launch, several sources in one wave and on
one cell, more receivers than a wave lists and several at one cell, receivers
set in the middle of a run, and batches wide enough for the largest tiles.
"""
import numpy as np
import pytest

import decks
from test_gpu_e2d_fused import deck, make, outputs

pytestmark = pytest.mark.gpu


def by_steps(s, n):
    for _ in range(n):
        s.run(1)


def same(a, b):
    (ta, fa), (tb, fb) = outputs(a), outputs(b)
    assert np.abs(fa).max() > 0
    assert np.array_equal(ta, tb) and np.array_equal(fa, fb)


SIZES = [dict(nx=2, nz=2, npml=1), dict(nx=7, nz=3, npml=2), dict(nx=30, nz=62, npml=1), dict(nx=61, nz=44, npml=3),
         dict(nx=200, nz=111, npml=20), dict(nx=111, nz=300, npml=30), dict(nx=333, nz=401, npml=10)]


@pytest.mark.parametrize("steps", [2, 3, 47])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s['nx']}x{s['nz']}_np{s['npml']}")
def test_tiles_equal_single_steps(ctx, size, steps):
    d = deck(seed=sum(size.values()) + steps, nsteps=40 + steps, src_type=[decks.BULK, decks.SX, decks.SXZ][steps % 3],
             **size)
    a, b = make(ctx, d), make(ctx, d)
    a.run(40), a.run(steps)
    by_steps(b, 40 + steps)
    same(a, b)
    a.close(), b.close()


def test_many_sources_and_receivers(ctx):
    d = deck(nx=70, nz=150, npml=6, seed=3, nsteps=33)
    nz = 150
    d["src_idx"] = np.array([20 * nz + 40, 20 * nz + 40, 21 * nz + 44, 22 * nz + 100, 69 * nz + 149], np.uintp)
    d["src_type"] = np.array([decks.BULK, decks.SX, decks.SXZ, decks.SZ, decks.BULK], np.intc)
    d["A"], d["f"] = [1.0, 0.5, -0.7, 0.3, 0.9], [25.0, 30.0, 20.0, 35.0, 15.0]
    # all five components at every cell of three rows, then a sparse grid twice
    full = np.array([i * nz + j for i in (30, 31, 33) for j in range(nz) for _ in range(5)])
    grid = np.array([i * nz + j for i in range(0, 70, 9) for j in range(0, nz, 13)] * 2)
    d["rec_idx"] = np.concatenate([full, grid]).astype(np.uintp)
    comps = np.array([0, 2, 5, 6, 7])
    d["rec_comp"] = np.concatenate([np.tile(comps, 3 * nz), comps[np.arange(grid.size) % 5]]).astype(np.intc)
    a, b = make(ctx, d), make(ctx, d)
    a.run(20), a.run(13)
    by_steps(b, 33)
    same(a, b)
    a.close(), b.close()


def test_receivers_set_during_a_run(ctx):
    d = deck(nx=50, nz=60, npml=5, seed=9, nsteps=60)
    a, b = make(ctx, d), make(ctx, d)
    a.run(21)
    by_steps(b, 21)
    for s in (a, b):
        s.set_receivers(d["rec_idx"], d["rec_comp"], 17)   # records steps 21..37 only
    a.run(30)
    by_steps(b, 30)
    ta, tb = a.traces(0, 17), b.traces(0, 17)
    assert np.abs(ta).max() > 0 and np.array_equal(ta, tb)
    a.close(), b.close()


def test_wide_batch_equals_single_steps(ctx):
    from seismod_amd.solver import E2dBatch
    ds = [deck(nx=400 + 37 * k, nz=620 - 41 * k, npml=20, seed=50 + k, nsteps=19 + 5 * k) for k in range(6)]
    a, b = [make(ctx, d) for d in ds], [make(ctx, d) for d in ds]
    batch = E2dBatch(ctx)
    batch.run(a, [d["nsteps"] for d in ds])
    batch.close()
    for x, y, d in zip(a, b, ds):
        by_steps(y, d["nsteps"])
        same(x, y)
        x.close(), y.close()
