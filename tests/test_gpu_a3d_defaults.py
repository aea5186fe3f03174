"""GPU tests of the 3D solver's choices at creation: the row pitch (padded to
cache lines or to 8 cells) and the kernel variant (one cell a lane, or tiles
where the wavefields leave the last-level cache).  Either choice only moves
data and work around, so traces and fields are bit-identical to the other.
And of reading slices and fields between runs."""
import numpy as np
import pytest

import decks
from test_gpu_variants import run

pytestmark = pytest.mark.gpu


# z cells with layers; storage; does a row end at a cache line (at most 1/7
# more cells in 16 bits, 1/16 in FP32) or at a multiple of 8 cells
PITCH = [(55, "bf16", False), (56, "bf16", True), (57, "f16", True), (58, "bf16", True),
         (150, "f32", False), (152, "f32", True), (177, "f32", False), (180, "f32", False), (181, "f32", True),
         (64, "f32", True)]


@pytest.mark.parametrize("nz2,storage,lines", PITCH)
def test_pitch_equals_forced_lines(ctx, nz2, storage, lines):
    from seismod_amd.solver import A3dConfig
    np_ = 2 + nz2 % 2
    d = decks.a3d_deck(nx=7, ny=9, nz=nz2 - 2 * np_, np_=np_, seed=nz2, nsteps=50)
    c = d["cfg"]
    need = [A3dConfig(nx=c["nx"], ny=c["ny"], nz=c["nz"], np=np_, dx=c["dx"], dy=c["dy"], dz=c["dz"],
                      dt=c["dt"], f0=c["f0"], storage=storage, sround=s, pad64=p).bytes_needed()
            for s, p in ((False, False), (False, True), (storage != "f32", False))]
    # bytes of a cell of pitch: two halves of four fields, three sets of x and y layer arrays, two of material
    nx2, ny2, e = c["nx"] + 2 * np_, c["ny"] + 2 * np_, 4 if storage == "f32" else 2
    cell = e * (8 * nx2 * ny2 + 3 * 2 * np_ * (nx2 + ny2)) + 4 * 2 * nx2 * ny2
    up = lambda q: -(-nz2 // q) * q
    pitch = [up(64) - (need[1] - n) / cell for n in need]
    line = 32 if storage == "f32" else 64
    assert pitch[0] == (up(line) if lines else up(8))
    # the rounding bits hash the index: with them the limit of 16 bits stays 1/10
    assert pitch[2] == (pitch[0] if storage == "f32" else up(8) if 10 * (up(64) - nz2) > nz2 else up(64))
    a = run(ctx, d, storage, "tile")
    b = run(ctx, d, storage, "cell", pad64=True)
    assert np.abs(a[0]).max() > 0
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


# below and above the line between the variants, few and many items a slot
@pytest.mark.parametrize("shape,storage,variant", [
    ((20, 9, 6, 3), "f32", "cell"), ((40, 150, 60, 4), "f32", "cell"),
    ((178, 170, 176, 4), "f32", "tile"), ((20, 9, 6, 3), "bf16", "tilesplit"),
    ((60, 150, 61, 4), "f16", "tilesplit")])
def test_default_variant_equals_cell(ctx, shape, storage, variant):
    from seismod_amd.solver import A3dConfig, Acoustic3D, source_functions
    nx, ny, nz, np_ = shape
    d = decks.a3d_deck(nx=nx, ny=ny, nz=nz, np_=np_, seed=5, nsteps=24)
    c = d["cfg"]
    got = []
    for v in (None, "cell"):
        s = Acoustic3D(ctx, A3dConfig(nx=nx, ny=ny, nz=nz, np=np_, dx=c["dx"], dy=c["dy"], dz=c["dz"],
                                      dt=c["dt"], f0=c["f0"], vmax=c["vmax"], storage=storage),
                       d["vp"], d["rho"])
        if v is None:
            assert s.variant() == variant
        else:
            s.set_variant(v)
            s.set_launch(4, 1)
        L, fct = source_functions(d["A"], d["f"], c["dt"])
        s.set_sources(d["src_idx"], L, fct)
        s.run(24)
        got.append([s.field(k) for k in (8, 0, 1, 2)])
        s.close()
    assert np.abs(got[0][0]).max() > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)


# padded and whole rows, every element size, with and without a second half
@pytest.mark.parametrize("nx,ny,nz,np_,storage", [
    (9, 7, 13, 3, "f32"), (9, 7, 58, 3, "f32"), (9, 7, 13, 3, "bf16"), (3, 6, 61, 0, "f16"),
    (3, 3, 9, 0, "f32"), (40, 33, 51, 2, "bf16"), (9, 7, 13, 3, "f64")])
def test_slices_between_runs(ctx, nx, ny, nz, np_, storage):
    """Slices and fields taken between runs agree with each other and leave
    the run as it is without them."""
    from seismod_amd.solver import A3dConfig, Acoustic3D, source_functions
    d = decks.a3d_deck(nx=nx, ny=ny, nz=nz, np_=np_, seed=3, nsteps=30)
    c = d["cfg"]
    got = []
    for look in (False, True):
        s = Acoustic3D(ctx, A3dConfig(nx=nx, ny=ny, nz=nz, np=np_, dx=c["dx"], dy=c["dy"], dz=c["dz"],
                                      dt=c["dt"], f0=c["f0"], vmax=c["vmax"], storage=storage),
                       d["vp"], d["rho"])
        L, fct = source_functions(d["A"], d["f"], c["dt"])
        s.set_sources(d["src_idx"], L, fct)
        s.set_receivers(d["rec_idx"], d["rec_comp"], 30)
        for n in (1, 12, 2, 15):
            if look:
                for comp in (8, 1):
                    f = s.field(comp)
                    for iy in (0, f.shape[1] - 1):
                        assert np.array_equal(s.slice_xz(comp, iy), f[:, iy, :])
                    assert np.array_equal(s.field(comp), f)
            s.run(n)
        got.append([s.traces(0, 30)] + [s.field(k) for k in (8, 0, 1, 2)])
        s.close()
    assert np.abs(got[0][1]).max() > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
