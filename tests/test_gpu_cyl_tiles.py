"""e_cyl_iso: receivers recorded by the tiles that own them, and the torsional
fields of mode 0, which are advanced only once a source has excited them."""
import numpy as np
import pytest

from test_gpu_cyl import FR, FT, FZ, TRR, TRT, TRZ, TTT, TTZ, TZZ, VR, VT, VZ, deck

pytestmark = pytest.mark.gpu

FIELDS = {"vr": VR, "vt": VT, "vz": VZ, "trr": TRR, "ttt": TTT, "tzz": TZZ, "trz": TRZ, "trt": TRT, "ttz": TTZ}


def solver(ctx, d, storage):
    from seismod_amd.solver import CylConfig, Cylindrical
    c = d["cfg"]
    s = Cylindrical(ctx, CylConfig(nx=c["nx"], nz=c["nz"], np=c["np"], dr=c["dx"], dz=c["dz"], dt=c["dt"], f0=d["f0"],
                                   mode=c["n"], alpha_max=d["alpha_max"], storage=storage), d["vp"], d["vs"], d["rho"])
    s.set_sources(d["types"], d["idx"], d["L"], d["fct"])
    s.set_receivers(d["ridx"], d["rcomp"], d["nsteps"])
    return s


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("n", [0, 1])
def test_receivers_at_every_cell(ctx, n, storage):
    """More receivers than threads in a tile, tiles cut by the grid's edges,
    every field: the last recorded row is the fields themselves."""
    d = deck(nx=37, nz=101, np_=7, n=n, seed=21, src=((FR, 6, 40), (FT, 9, 50)), nsteps=40)
    names = list(FIELDS)
    cells = d["vp"].size
    d["ridx"] = np.concatenate([np.arange(cells), np.arange(cells - 1, -1, -3)]).astype(np.uintp)
    comp = [FIELDS[k] for k in names]
    d["rcomp"] = np.array(comp, np.intc)[(np.arange(d["ridx"].size) * 7 + 3) % len(comp)]
    s = solver(ctx, d, storage)
    s.run(d["nsteps"])
    last = s.traces(d["nsteps"] - 1, 1)[0]
    for k in names:
        where = d["rcomp"] == FIELDS[k]
        want = s.field(k).reshape(-1)[d["ridx"][where].astype(np.int64)]
        assert np.abs(want).max() > 0 and np.array_equal(last[where], want), k
    s.close()


def test_torsional_fields_survive_their_source(ctx):
    """Mode 0: the torsional fields are advanced once a source has excited
    them, also after that source is gone, until the next reset."""
    d = deck(nx=30, nz=60, np_=6, n=0, seed=22, src=((FZ, 5, 30), (FT, 7, 25)), nsteps=80)
    L = np.array(d["L"])
    cut = d["fct"].copy()
    off = int(L[0])
    cut[off + 20:off + int(L[1])] = 0.0            # FT ends after 20 steps
    a = solver(ctx, dict(d, fct=cut), "f64")
    a.run(80)
    b = solver(ctx, d, "f64")
    b.run(20)
    b.set_sources(d["types"][:1], d["idx"][:1], L[:1], d["fct"][:off])
    b.run(60)
    for k in FIELDS:
        fa, fb = a.field(k), b.field(k)
        assert np.abs(fa).max() > 0 and np.array_equal(fa, fb), k
    b.reset()
    b.run(40)
    assert not b.field("vt").any() and b.field("vz").any()
    a.close(), b.close()
