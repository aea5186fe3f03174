"""The workgroups of the spectral transforms stay within the LDS the runtime
grants (65536 bytes where it refuses more) and within 512 threads, over grids
of every kind of axis length.  Host code only, compiled here."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
LIBDIR = ROOT / "seismod_amd" / "lib"

SOURCE = r"""
#include "pstd.hpp"
using namespace sm::pstd;
int main()
{
    const int len[] = {8, 100, 256, 363, 640, 1000, 1040, 1039, 1617, 2000, 2048, 2187, 3000, 3402, 4096};
    int made = 0;
    for (size_t lds : {(size_t)65536, FFT_LDS})
        for (size_t elt : {4, 8})
            for (int nx : len)
                for (int nz : len) {
                    Grid g;
                    g.nx2 = nx; g.nz2 = nz; g.N = (size_t)nx * nz; g.elt = elt; g.lds = lds;
                    int count[2];
                    for (int ax = 0; ax < 2; ++ax)
                        count[ax] = fft_plan(ax ? nz : nx, elt, g.fft[ax]) && fft_lds(g.fft[ax], 1, 1, elt) <= lds ? 2 : 0;
                    if (count[0] && count[1] && g.fft[0].loop != g.fft[1].loop) count[1] = 0;
                    if (!count[0] && !count[1]) continue;
                    const FftShape s = fft_shape(g, elt, count[0], count[1]);
                    for (int ax = 0; ax < 2; ++ax)
                        if (count[ax] && (fft_lds(g.fft[ax], s.V, s.P, elt) > lds || fft_threads(g.fft[ax], s.P) > 512)) {
                            printf("%d x %d, %zu bytes a value, limit %zu: V %d P %d take %zu\n", nx, nz, elt, lds, s.V,
                                   s.P, fft_lds(g.fft[ax], s.V, s.P, elt));
                            return 1;
                        }
                    ++made;
                }
    printf("%d grids\n", made);
    return made > 500 ? 0 : 2;
}
"""


def test_workgroups_fit_the_granted_lds(tmp_path):
    from seismod_amd.build import CSRC, HIPCC, INCLUDE
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "shape.hip", tmp_path / "shape"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--cuda-host-only", "-O1", "-std=c++17", f"-I{CSRC}", f"-I{INCLUDE}", str(src), "-o", str(exe),
                    f"-L{LIBDIR}", "-lseismod_hip", f"-Wl,-rpath,{LIBDIR}"], check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
