"""GPU tests of the 3D solver's choices at creation: the row pitch, padded to
cache lines or to 8 cells.  The choice only moves data around, so traces and
fields are bit-identical to the other."""
import numpy as np
import pytest

import decks
from test_gpu_variants import run

pytestmark = pytest.mark.gpu


# z cells with layers; storage; does a row end at the next cache line
PITCH = [(55, "bf16", False), (56, "bf16", True), (57, "f16", True), (58, "bf16", True),
         (150, "f32", False), (152, "f32", True), (177, "f32", True), (64, "f32", True)]


@pytest.mark.parametrize("nz2,storage,lines", PITCH)
def test_pitch_equals_forced_lines(ctx, nz2, storage, lines):
    from seismod_amd.solver import A3dConfig
    np_ = 2 + nz2 % 2
    d = decks.a3d_deck(nx=7, ny=9, nz=nz2 - 2 * np_, np_=np_, seed=nz2, nsteps=50)
    c = d["cfg"]
    need = [A3dConfig(nx=c["nx"], ny=c["ny"], nz=c["nz"], np=np_, dx=c["dx"], dy=c["dy"], dz=c["dz"],
                      dt=c["dt"], f0=c["f0"], storage=storage, sround=s, pad64=p).bytes_needed()
            for s, p in ((False, False), (False, True), (True, False))]
    wide = nz2 if nz2 % 64 == 0 else (nz2 // 64 + 1) * 64
    if wide - nz2 >= 8 and storage != "f32":
        assert (need[0] == need[1]) == lines
        assert need[2] < need[1]       # the rounding bits hash the index: their pitch stays
    a = run(ctx, d, storage, "tile")
    b = run(ctx, d, storage, "cell", pad64=True)
    assert np.abs(a[0]).max() > 0
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
