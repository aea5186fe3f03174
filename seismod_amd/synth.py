"""Seeded synthetic models and shot geometries for the benchmark workloads.

There is no field data in this project; every workload is generated here
from a seed so runs are reproducible:
  - a_iso_3d 256^3 (and 512^3): layered Vp with sorted random interface
    depths, plus a Gaussian-smoothed random perturbation, Gardner density
    rho = 310 Vp^0.25, padded into the CPML by edge replication exactly as
    read_model_a does (io_utils.c:1089-1143);
  - e_iso 400x400 two-layer model with a surface receiver line;
  - batches of e_iso shots of random size, layering, frequency and length;
  - an e_cyl_iso borehole: fluid column around the axis inside a bedded
    formation, Kurkjian monopole source on the axis, receiver array in the
    fluid.
"""
from __future__ import annotations

from dataclasses import dataclass, field

import numpy as np

VX, VY, VZ, P = 0, 1, 2, 8
BULK = 6


def smoothed_noise(shape, sigma: float, rng: np.random.Generator) -> np.ndarray:
    """N(0,1) field smoothed by a Gaussian of `sigma` cells, peak |.| = 1."""
    from scipy.ndimage import gaussian_filter
    noise = rng.standard_normal(shape, dtype=np.float32)
    noise = gaussian_filter(noise, sigma=sigma, mode="reflect", truncate=3.0)
    noise /= max(float(np.abs(noise).max()), 1e-30)
    return noise


def layered_vp(nz: int, rng: np.random.Generator, vmin: float, vmax: float,
               nlayers: tuple[int, int] = (4, 8)) -> np.ndarray:
    """Vp(z) with a random number of layers, increasing with depth."""
    nl = int(rng.integers(nlayers[0], nlayers[1] + 1))
    tops = np.sort(rng.choice(np.arange(1, nz), size=nl - 1, replace=False))
    vals = np.sort(rng.uniform(vmin, vmax, size=nl))
    return vals[np.searchsorted(tops, np.arange(nz), side="right")]


@dataclass
class A3dShot:
    nx: int
    ny: int
    nz: int
    np: int
    dx: float
    dt: float
    f0: float
    nsteps: int
    vp: np.ndarray          # padded (nx2, ny2, nz2), FP64
    rho: np.ndarray
    src_idx: np.ndarray
    rec_idx: np.ndarray
    rec_comp: np.ndarray
    meta: dict = field(default_factory=dict)

    @property
    def shape(self):
        return self.vp.shape

    @property
    def cells(self) -> int:
        return int(np.prod(self.vp.shape))


def a3d_layered_shot(n: int = 256, np_: int = 20, dx: float = 10.0, seed: int = 2,
                     vmin: float = 1500.0, vmax: float = 4500.0, perturb: float = 0.05,
                     sigma: float = 8.0, dt: float = 6.0e-4, f0: float = 15.0,
                     nsteps: int = 1500, nrec_side: int = 32) -> A3dShot:
    """3D acoustic CPML shot: centre-top Bulk source, Vz receiver plane.

    256^3 defaults: source at (1280, 1280, 100) m, receivers at z = 50 m on
    x, y = 40 + 80 r m (r < 32), dt = 0.6 ms, 1500 steps.
    """
    rng = np.random.default_rng(seed)
    vz = layered_vp(n, rng, vmin, vmax)
    vp = np.empty((n, n, n), dtype=np.float64)
    vp[:] = vz[None, None, :]
    if perturb:
        vp *= 1.0 + perturb * smoothed_noise((n, n, n), sigma, rng).astype(np.float64)
    rho = 310.0 * vp ** 0.25
    vp = np.pad(vp, np_, mode="edge")
    rho = np.pad(rho, np_, mode="edge")
    nx2 = ny2 = nz2 = n + 2 * np_
    sx = sy = n // 2
    sz = max(1, int(round(100.0 / dx)))
    src = np.array([((sx + np_) * ny2 + sy + np_) * nz2 + sz + np_], dtype=np.uintp)
    step = max(1, n // nrec_side)
    off = step // 2
    rz = int(round(50.0 / dx))
    rec = [((off + step * a + np_) * ny2 + off + step * b + np_) * nz2 + rz + np_
           for a in range(nrec_side) for b in range(nrec_side)]
    return A3dShot(nx=n, ny=n, nz=n, np=np_, dx=dx, dt=dt, f0=f0, nsteps=nsteps, vp=vp,
                   rho=rho, src_idx=src, rec_idx=np.array(rec, dtype=np.uintp),
                   rec_comp=np.full(len(rec), VZ, dtype=np.intc),
                   meta=dict(seed=seed, vmin=vmin, vmax=vmax, perturb=perturb, sigma=sigma))


def algorithmic_bytes_a3d(nx2: int, ny2: int, nz2: int, np_: int, state_bytes: int = 4,
                          mat_bytes: int = 4) -> float:
    """Minimal HBM bytes per padded cell per step of the 3D CPML update.

    P, vx, vy, vz read and written once, rho and K*dt read once, and the two
    memory variables of each axis read and written only in that axis's
    absorbing slabs (fraction 2np/n2 of the cells).
    """
    frac = sum(2.0 * np_ / n for n in (nx2, ny2, nz2))
    return state_bytes * 8 + mat_bytes * 2 + state_bytes * 4 * frac


def algorithmic_bytes_e2d(nx: int, nz: int, npml: int, state_bytes: int = 4) -> float:
    """Minimal HBM bytes per padded cell per step of the 2D split-PML update.

    Interior cell: vx, vz, txx, tzz, txz read and written once and three
    material values (rho, lambda, mu) read once: 13 words.  PML cell: the ten
    split fields read and written: 20 words.
    """
    NX, NZ = nx + 2 * npml, nz + 2 * npml
    interior = nx * nz
    pml = NX * NZ - interior
    return state_bytes * (13.0 * interior + 20.0 * pml) / (NX * NZ)


@dataclass
class E2dShot:
    nx: int
    nz: int
    npml: int
    h: float
    dt: float
    f0: float
    nsteps: int
    vp: np.ndarray          # interior (nx, nz), FP64
    vs: np.ndarray
    rho: np.ndarray
    src_type: np.ndarray
    src_idx: np.ndarray
    rec_idx: np.ndarray
    rec_comp: np.ndarray
    meta: dict = field(default_factory=dict)

    @property
    def cells(self) -> int:
        return (self.nx + 2 * self.npml) * (self.nz + 2 * self.npml)


def e2d_two_layer_shot(n: int = 400, npml: int = 20, h: float = 5.0, dt: float = 5.0e-4,
                       nsteps: int = 2000, f0: float = 25.0) -> E2dShot:
    """e_iso two-layer shot: (Vp, Vs, rho) = (2500, 1400, 2000) above node
    z = n/2 and (3500, 2000, 2400) below, Bulk source at node (n/2, n/8),
    Vz receivers on the surface row every 4 nodes (100 at n = 400)."""
    vp = np.empty((n, n)); vs = np.empty((n, n)); rho = np.empty((n, n))
    zc = n // 2
    vp[:, :zc], vs[:, :zc], rho[:, :zc] = 2500.0, 1400.0, 2000.0
    vp[:, zc:], vs[:, zc:], rho[:, zc:] = 3500.0, 2000.0, 2400.0
    src = np.array([(n // 2) * n + n // 8], dtype=np.uintp)
    rec = np.array([4 * r * n for r in range(n // 4)], dtype=np.uintp)
    return E2dShot(nx=n, nz=n, npml=npml, h=h, dt=dt, f0=f0, nsteps=nsteps, vp=vp, vs=vs,
                   rho=rho, src_type=np.array([BULK], dtype=np.intc), src_idx=src,
                   rec_idx=rec, rec_comp=np.full(len(rec), VZ, dtype=np.intc))


def e2d_batch_shots(count: int = 64, seed: int = 4, npml: int = 20, h: float = 5.0,
                    nx_range=(300, 1200), nz_range=(300, 800), steps_range=(1000, 3000),
                    f_range=(10.0, 40.0)) -> list[E2dShot]:
    """Independent e_iso shots: grid nx ~ U{300..1200} by nz ~ U{300..800},
    3-6 layers with Vp ~ U[2000, 5000] (sorted with depth), Vs = Vp/U[1.7, 1.9],
    rho ~ U[1800, 2700], Ricker f ~ U[10, 40] Hz, steps ~ U{1000..3000},
    dt at half the CFL limit, Bulk source at the top centre, Vz receivers
    every 4 nodes on row 0."""
    rng = np.random.default_rng(seed)
    shots = []
    for _ in range(count):
        nx = int(rng.integers(nx_range[0], nx_range[1] + 1))
        nz = int(rng.integers(nz_range[0], nz_range[1] + 1))
        nl = int(rng.integers(3, 7))
        tops = np.sort(rng.choice(np.arange(1, nz), size=nl - 1, replace=False))
        vpl = np.sort(rng.uniform(2000.0, 5000.0, size=nl))
        ratio = rng.uniform(1.7, 1.9, size=nl)
        rhol = rng.uniform(1800.0, 2700.0, size=nl)
        layer = np.searchsorted(tops, np.arange(nz), side="right")
        vp = np.broadcast_to(vpl[layer], (nx, nz)).copy()
        vs = np.broadcast_to((vpl / ratio)[layer], (nx, nz)).copy()
        rho = np.broadcast_to(rhol[layer], (nx, nz)).copy()
        f0 = float(rng.uniform(*f_range))
        nsteps = int(rng.integers(steps_range[0], steps_range[1] + 1))
        dt = 0.5 * h / (np.sqrt(2.0) * vp.max())
        src = np.array([(nx // 2) * nz + 1], dtype=np.uintp)
        rec = np.array([4 * r * nz for r in range((nx + 3) // 4)], dtype=np.uintp)
        shots.append(E2dShot(nx=nx, nz=nz, npml=npml, h=h, dt=dt, f0=f0, nsteps=nsteps,
                             vp=vp, vs=vs, rho=rho, src_type=np.array([BULK], dtype=np.intc),
                             src_idx=src, rec_idx=rec,
                             rec_comp=np.full(len(rec), VZ, dtype=np.intc),
                             meta=dict(seed=seed)))
    return shots


# ---------------------------------------------------------------------------
# Model files: the seeded models above written in the text format the
# drop-in programs (and the reference) read, by the parallel writer of the
# host I/O library (values with 17 significant digits read back bit for bit).

def _hostio():
    import ctypes as C
    from pathlib import Path
    lib = C.CDLL(str(Path(__file__).resolve().parent / "lib" / "libsm_hostio.so"))
    dbl = C.POINTER(C.c_double)
    lib.sm_write_model_a.argtypes = [C.c_char_p, C.c_size_t, C.c_size_t, C.c_size_t] + \
        [C.c_double] * 6 + [dbl, dbl, C.c_int]
    lib.sm_write_model_e.argtypes = [C.c_char_p, C.c_size_t, C.c_size_t] + [C.c_double] * 4 + \
        [dbl, dbl, dbl, C.c_int]
    return lib, dbl


def write_model_a(path, shot: A3dShot, digits: int = 17) -> None:
    """The interior of a 3D shot's model as an isotropic_acoustic_3d file
    (io_utils.c:1029-1072 format), origin 0."""
    lib, dbl = _hostio()
    p = shot.np
    vp = np.ascontiguousarray(shot.vp[p:-p, p:-p, p:-p] if p else shot.vp)
    rho = np.ascontiguousarray(shot.rho[p:-p, p:-p, p:-p] if p else shot.rho)
    if lib.sm_write_model_a(str(path).encode(), shot.nx, shot.ny, shot.nz, shot.dx, shot.dx, shot.dx,
                            0.0, 0.0, 0.0, vp.ctypes.data_as(dbl), rho.ctypes.data_as(dbl),
                            digits) != 0:
        raise OSError(f"cannot write {path}")


def write_model_e(path, shot: E2dShot, digits: int = 17) -> None:
    """A 2D shot's model as an isotropic_elastic file (io_utils.c:892-947
    format), origin 0."""
    lib, dbl = _hostio()
    a = [np.ascontiguousarray(x, dtype=np.float64) for x in (shot.vp, shot.vs, shot.rho)]
    if lib.sm_write_model_e(str(path).encode(), shot.nx, shot.nz, shot.h, shot.h, 0.0, 0.0,
                            *(x.ctypes.data_as(dbl) for x in a), digits) != 0:
        raise OSError(f"cannot write {path}")


def main(argv=None) -> None:
    """python -m seismod_amd.synth a3d --n 512 --seed 3 --out model.dat
       python -m seismod_amd.synth e2d --n 400 --out model2d.dat"""
    import argparse
    ap = argparse.ArgumentParser(description="write a seeded model file")
    ap.add_argument("kind", choices=["a3d", "e2d"])
    ap.add_argument("--n", type=int, default=256)
    ap.add_argument("--seed", type=int, default=2)
    ap.add_argument("--vmax", type=float, default=4500.0)
    ap.add_argument("--digits", type=int, default=17)
    ap.add_argument("--out", required=True)
    args = ap.parse_args(argv)
    if args.kind == "a3d":
        write_model_a(args.out, a3d_layered_shot(n=args.n, seed=args.seed, vmax=args.vmax),
                      args.digits)
    else:
        write_model_e(args.out, e2d_two_layer_shot(n=args.n), args.digits)


if __name__ == "__main__":
    main()


@dataclass
class CylShot:
    nx: int
    nz: int
    np: int
    dr: float
    dt: float
    f0: float
    mode: int
    nsteps: int
    vp: np.ndarray          # padded (nx + np, nz + 2 np), row i at r = i dr, FP64
    vs: np.ndarray
    rho: np.ndarray
    src_idx: np.ndarray     # one Kurkjian source on the axis
    src_r: float
    rec_idx: np.ndarray
    rec_comp: np.ndarray

    @property
    def cells(self) -> int:
        return int(self.vp.size)


def cyl_borehole_shot(nx: int = 1000, nz: int = 4000, np_: int = 20, dr: float = 0.01,
                      seed: int = 5, mode: int = 0, f0: float = 8000.0, nsteps: int = 2000,
                      borehole_cells: int = 10, rec_every: int = 20) -> CylShot:
    """e_cyl_iso borehole model: water (1500 m/s, 1000 kg/m^3) for r below
    `borehole_cells` cells, a formation of 6-12 beds along z with Vp ~
    U[2500, 4500], Vs = Vp / U[1.7, 1.9], rho ~ U[2100, 2600]; a Kurkjian
    source on the axis at mid-depth, trr receivers in the fluid (row 1)
    every `rec_every` cells and a few Vr / Vz receivers in the formation.
    Padded like read_model_e_cyl: np extra rows at large r, np rows at each
    z end, copied from the edge."""
    rng = np.random.default_rng(seed)
    nbeds = int(rng.integers(6, 13))
    tops = np.sort(rng.choice(np.arange(1, nz), size=nbeds - 1, replace=False))
    bed = np.searchsorted(tops, np.arange(nz), side="right")
    vpb = rng.uniform(2500.0, 4500.0, size=nbeds)
    vsb = vpb / rng.uniform(1.7, 1.9, size=nbeds)
    rhob = rng.uniform(2100.0, 2600.0, size=nbeds)
    vp = np.repeat(vpb[bed][None, :], nx, axis=0)
    vs = np.repeat(vsb[bed][None, :], nx, axis=0)
    rho = np.repeat(rhob[bed][None, :], nx, axis=0)
    vp[:borehole_cells] = 1500.0
    vs[:borehole_cells] = 0.0
    rho[:borehole_cells] = 1000.0
    nx2, nz2 = nx + np_, nz + 2 * np_

    def pad(a):
        out = np.empty((nx2, nz2))
        out[:nx, np_:np_ + nz] = a
        out[:nx, :np_] = a[:, :1]
        out[:nx, np_ + nz:] = a[:, -1:]
        out[nx:, :] = out[nx - 1:nx, :]
        return out

    vp, vs, rho = pad(vp), pad(vs), pad(rho)
    dt = 0.6 * 0.5 * (dr + dr) / (np.sqrt(2.0) * vp.max())
    zc = np_ + nz // 2
    src_idx = np.array([0 * nz2 + zc], dtype=np.uintp)
    TRR, VR, VZ_ = 15, 13, 2
    rec = [(1 * nz2 + j, TRR) for j in range(np_, np_ + nz, rec_every)]
    for i in (borehole_cells + 5, nx // 4, nx // 2):
        rec += [(i * nz2 + zc + 200, VR), (i * nz2 + zc - 200, VZ_)]
    return CylShot(nx=nx, nz=nz, np=np_, dr=dr, dt=float(dt), f0=f0, mode=mode, nsteps=nsteps,
                   vp=vp, vs=vs, rho=rho, src_idx=src_idx, src_r=0.0,
                   rec_idx=np.array([r[0] for r in rec], dtype=np.uintp),
                   rec_comp=np.array([r[1] for r in rec], dtype=np.intc))


def algorithmic_bytes_cyl(nx2: int, nz2: int, np_: int, elt: int = 4, torsional: bool = True) -> float:
    """Minimal HBM bytes per padded cell per step of the e_cyl_iso update.

    The nine fields (v_r, v_theta, v_z and six stresses) read and written
    once and the eight material arrays (lambda, lambda+2mu, three mu and
    three buoyancy averages) read once: 26 values; plus the CPML memory
    variables, read and written once where they exist (18 arrays over the
    np+1 outer rows, 6 over the 2np+1 slots of every row).  Without the
    torsional fields (mode 0, no Ft source): six fields, five material
    arrays, 8 and 4 memory variables."""
    cells = nx2 * nz2
    values, r, z = (26.0, 18, 6) if torsional else (17.0, 8, 4)
    mem = (r * (np_ + 1) * nz2 + z * nx2 * (2 * np_ + 1)) if np_ else 0
    return elt * (values + 2.0 * mem / cells)


@dataclass
class ShShot:
    nx: int
    nz: int
    np: int
    h: float
    dt: float
    f0: float
    nsteps: int
    mu: np.ndarray          # padded (nx + 2np, nz + 2np), GPa, as read_model_ve_sh leaves it
    rho: np.ndarray
    gamma: np.ndarray
    Q: np.ndarray
    f: np.ndarray
    src_idx: np.ndarray     # one Syz source
    rec_idx: np.ndarray
    rec_comp: np.ndarray

    @property
    def cells(self) -> int:
        return int(self.mu.size)


def sh_layered_shot(n: int = 1000, np_: int = 20, h: float = 5.0, seed: int = 7, f0: float = 25.0,
                    nsteps: int = 1000, nrec: int = 200) -> ShShot:
    """ve_vti_sh_pml workload: n x n nodes of h metres plus np CPML layers,
    5-10 horizontal layers with Vs0 ~ U[800, 2500] m/s, rho ~ U[1800, 2600],
    gamma ~ U[0, 0.25], Q ~ U[20, 100], relaxation frequency f0; a Syz source
    at (n/2, 20) nodes and a line of nrec Vy receivers at depth 10 nodes.
    dt at 40% of the RK4 pseudo-spectral stability limit."""
    rng = np.random.default_rng(seed)
    nl = int(rng.integers(5, 11))
    tops = np.sort(rng.choice(np.arange(1, n), size=nl - 1, replace=False))
    lay = np.searchsorted(tops, np.arange(n), side="right")
    vs = np.sort(rng.uniform(800.0, 2500.0, nl))[lay] * np.ones((n, 1))
    rho = rng.uniform(1800.0, 2600.0, nl)[lay] * np.ones((n, 1))
    gamma = rng.uniform(0.0, 0.25, nl)[lay] * np.ones((n, 1))
    Q = rng.uniform(20.0, 100.0, nl)[lay] * np.ones((n, 1))
    pad = lambda a: np.pad(a, np_, mode="edge")
    mu = pad(vs * vs * rho * 1e-9)
    vmax = float((vs * np.sqrt(1 + 2 * gamma)).max())
    dt = 0.4 * 2.0 * h / (np.pi * vmax * np.sqrt(2.0))
    nz2 = n + 2 * np_
    src = np.array([(n // 2 + np_) * nz2 + 20 + np_], dtype=np.uintp)
    xs = np.linspace(np_, n + np_ - 1, nrec).astype(int)
    rec = np.array([x * nz2 + 10 + np_ for x in xs], dtype=np.uintp)
    return ShShot(nx=n, nz=n, np=np_, h=h, dt=float(dt), f0=f0, nsteps=nsteps, mu=mu, rho=pad(rho),
                  gamma=pad(gamma), Q=pad(Q), f=np.full(mu.shape, f0), src_idx=src, rec_idx=rec,
                  rec_comp=np.full(nrec, 1, dtype=np.intc))


def algorithmic_bytes_sh(elt: int = 8) -> float:
    """HBM bytes per padded cell per step of the ve_vti_sh_pml update, as the
    streaming minimum of its structure when every FFT derivative is one pass
    (read the field, write the derivative) and the rest of a Runge-Kutta
    stage is one pointwise pass: 4 stages x 4 derivatives x 2 values (32),
    and per stage the layer corrections, right-hand sides and update reading
    the 4 derivatives, 9 material arrays, the 5 step-start values, the 5
    accumulated values (stages 2-4) and the stage input's 2 relaxation
    variables (stages 2-4), writing 5 accumulated values and 5 next-stage
    inputs (stages 1-3): 28 + 35 + 35 + 30 = 128.  160 values per step."""
    return elt * 160.0


@dataclass
class VeShot:
    nx: int
    nz: int
    np: int
    h: float
    dt: float
    f0: float
    nsteps: int
    L: int
    model: tuple            # read_model_ve's padded arrays: K, mu, rho, eps, delta, Q1, f1, Q2, f2
    src_idx: np.ndarray     # one Bulk source
    rec_idx: np.ndarray
    rec_comp: np.ndarray

    @property
    def cells(self) -> int:
        return int(self.model[0].size)


def ve_layered_shot(n: int = 1000, np_: int = 20, h: float = 5.0, seed: int = 11, f0: float = 25.0,
                    nsteps: int = 1000, nrec: int = 200, L: int = 2) -> VeShot:
    """ve_vti_pml workload: n x n nodes of h metres plus np CPML layers,
    5-10 horizontal layers with Vp0 ~ U[1800, 4000] m/s (sorted with depth),
    Vp0/Vs0 ~ U[1.7, 2.2], rho ~ U[1800, 2600], epsilon ~ U[0, 0.25],
    delta ~ U[-0.05, 0.15], L quasi-dilatational mechanisms with Q ~
    U[20, 100] and relaxation frequencies spread over [5, 60] Hz, shear
    Q ~ U[20, 100] at f0; a Bulk source at (n/2, 20) nodes and a line of
    nrec Vz receivers at depth 10 nodes.  dt at 40% of the RK4
    pseudo-spectral stability limit."""
    rng = np.random.default_rng(seed)
    nl = int(rng.integers(5, 11))
    tops = np.sort(rng.choice(np.arange(1, n), size=nl - 1, replace=False))
    lay = np.searchsorted(tops, np.arange(n), side="right")
    one = np.ones((n, 1))
    vp = np.sort(rng.uniform(1800.0, 4000.0, nl))[lay] * one
    vs = vp / rng.uniform(1.7, 2.2, nl)[lay]
    rho = rng.uniform(1800.0, 2600.0, nl)[lay] * one
    eps = rng.uniform(0.0, 0.25, nl)[lay] * one
    dlt = rng.uniform(-0.05, 0.15, nl)[lay] * one
    Q1 = [rng.uniform(20.0, 100.0, nl)[lay] * one for _ in range(L)]
    f1 = [np.full((n, n), 5.0 + 55.0 * (m + 0.5) / L) for m in range(L)]
    Q2 = rng.uniform(20.0, 100.0, nl)[lay] * one
    pad = lambda a: np.pad(a, np_, mode="edge")
    mu_pa = vs * vs * rho
    model = (pad(1e-9 * (vp * vp * rho - 4. / 3. * mu_pa)), pad(mu_pa * 1e-9), pad(rho), pad(eps), pad(dlt),
             np.stack([pad(q) for q in Q1]), np.stack([pad(q) for q in f1]), pad(Q2), pad(np.full((n, n), f0)))
    vmax = float((vp * np.sqrt(1 + 2 * eps)).max())
    dt = 0.4 * 2.0 * h / (np.pi * vmax * np.sqrt(2.0))
    nz2 = n + 2 * np_
    src = np.array([(n // 2 + np_) * nz2 + 20 + np_], dtype=np.uintp)
    xs = np.linspace(np_, n + np_ - 1, nrec).astype(int)
    rec = np.array([x * nz2 + 10 + np_ for x in xs], dtype=np.uintp)
    return VeShot(nx=n, nz=n, np=np_, h=h, dt=float(dt), f0=f0, nsteps=nsteps, L=L, model=model, src_idx=src,
                  rec_idx=rec, rec_comp=np.full(nrec, 2, dtype=np.intc))


def algorithmic_bytes_ve(L: int = 2, elt: int = 8) -> float:
    """HBM bytes per padded cell per step of the ve_vti_pml update, counted as
    for algorithmic_bytes_sh: 4 stages x 8 derivatives x 2 values (64), and
    the fused pointwise pass per stage reading the 8 derivatives, 12 + 2L
    material arrays, the 7 + L step-start values, the 7 + L accumulated
    values (stages 2-4) and the stage input's L + 2 relaxation variables
    (stages 2-4), writing 7 + L accumulated values and 7 + L next-stage
    inputs (stages 1-3): 184 + 25 L.  248 + 25 L values per step."""
    return elt * (248.0 + 25.0 * L)


@dataclass
class PveShot:
    nx: int
    nz: int
    np: int
    h: float
    dt: float
    f0: float
    nsteps: int
    model: tuple            # read_model's padded arrays: K_m, K_s, K_f, phi, mu, rho_s, rho_f, T, eta, kappa, Q, fq
    src_idx: np.ndarray     # one Bulk source
    rec_idx: np.ndarray
    rec_comp: np.ndarray

    @property
    def cells(self) -> int:
        return int(self.model[0].size)


def biot_fast_velocity(K_m, K_s, K_f, phi, mu, rho_s, rho_f, T) -> np.ndarray:
    """Fast P velocity (m/s) of the unrelaxed, inviscid Biot medium: the
    square root of the larger eigenvalue of R^-1 C, C the undrained stiffness
    [[K_m + 4/3 mu + alpha^2 M, alpha M], [alpha M, M]] and R the density
    matrix [[rho, rho_f], [rho_f, T rho_f / phi]] (moduli in GPa, densities
    in kg/m^3; elementwise)."""
    Km, Ks, Kf, G = (np.asarray(a, np.float64) * 1e9 for a in (K_m, K_s, K_f, mu))
    phi, rs, rf, T = (np.asarray(a, np.float64) for a in (phi, rho_s, rho_f, T))
    alpha = 1 - Km / Ks
    M = 1. / ((alpha - phi) / Ks + phi / Kf)
    c11, c12, c22 = Km + 4. / 3. * G + alpha * alpha * M, alpha * M, M
    r11, r12, r22 = (1 - phi) * rs + phi * rf, rf, T * rf / phi
    # eigenvalues of R^-1 C from det(C - lambda R) = 0
    a = r11 * r22 - r12 * r12
    b = -(c11 * r22 + c22 * r11 - 2 * c12 * r12)
    c = c11 * c22 - c12 * c12
    return np.sqrt((-b + np.sqrt(b * b - 4 * a * c)) / (2 * a))


def pve_layered_shot(n: int = 1000, np_: int = 20, h: float = 5.0, seed: int = 13, f0: float = 25.0,
                     nsteps: int = 1000, nrec: int = 200) -> PveShot:
    """pve_iso_pml workload: n x n nodes of h metres plus np CPML layers,
    5-10 horizontal layers of water-saturated sandstone: K_s ~ U[33, 39] GPa,
    K_m ~ U[4, 16] GPa (stiffer with depth), K_f = 2.25 GPa, phi ~
    U[0.1, 0.32], mu ~ U[3, 12] GPa, rho_s ~ U[2600, 2700], rho_f = 1000
    kg/m^3, T ~ U[1.5, 3], eta = 1 cP, kappa ~ U[50, 2000] mD, Q ~ U[20,
    100] at f0; a Bulk source at (n/2, 20) nodes and a line of nrec Vz
    receivers at depth 10 nodes.  dt at 40% of the RK4 pseudo-spectral
    stability limit of the fast P wave."""
    rng = np.random.default_rng(seed)
    nl = int(rng.integers(5, 11))
    tops = np.sort(rng.choice(np.arange(1, n), size=nl - 1, replace=False))
    lay = np.searchsorted(tops, np.arange(n), side="right")
    one = np.ones((n, 1))
    layer = lambda lo, hi, sort=False: (np.sort(rng.uniform(lo, hi, nl)) if sort else
                                        rng.uniform(lo, hi, nl))[lay] * one
    K_s = layer(33.0, 39.0)
    K_m = layer(4.0, 16.0, sort=True)
    K_f = np.full((n, n), 2.25)
    phi = layer(0.1, 0.32)
    mu = layer(3.0, 12.0, sort=True)
    rho_s = layer(2600.0, 2700.0)
    rho_f = np.full((n, n), 1000.0)
    T = layer(1.5, 3.0)
    eta = np.full((n, n), 1.0)
    kappa = layer(50.0, 2000.0)
    Q = layer(20.0, 100.0)
    fq = np.full((n, n), f0)
    vals = (K_m, K_s, K_f, phi, mu, rho_s, rho_f, T, eta, kappa, Q, fq)
    vmax = float(biot_fast_velocity(*vals[:8]).max())
    dt = 0.4 * 2.0 * h / (np.pi * vmax * np.sqrt(2.0))
    pad = lambda a: np.pad(a, np_, mode="edge")
    nz2 = n + 2 * np_
    src = np.array([(n // 2 + np_) * nz2 + 20 + np_], dtype=np.uintp)
    xs = np.linspace(np_, n + np_ - 1, nrec).astype(int)
    rec = np.array([x * nz2 + 10 + np_ for x in xs], dtype=np.uintp)
    return PveShot(nx=n, nz=n, np=np_, h=h, dt=float(dt), f0=f0, nsteps=nsteps, model=tuple(pad(a) for a in vals),
                   src_idx=src, rec_idx=rec, rec_comp=np.full(nrec, 2, dtype=np.intc))


def algorithmic_bytes_pve(elt: int = 8) -> float:
    """HBM bytes per padded cell per step of the pve_iso_pml update, counted as
    for algorithmic_bytes_sh: 4 stages x 12 derivatives x 2 values (96); the
    analytic step reading v, q and their 4 coefficients and writing v and q
    (12); the fused pointwise pass per stage reading the 12 derivatives, 13
    material arrays and the 9 step-start values, writing 9 accumulated
    values, with 9 accumulated values read in stages 2-4, 9 next-stage
    inputs written in stages 1-3 and the stage input's relaxation variable
    read in stages 2-4 (the step-start values in stage 1): 52 + 62 + 62 + 53
    = 229.  337 values per step."""
    return elt * 337.0


def pve_vti_layered_shot(n: int = 1000, np_: int = 20, h: float = 5.0, seed: int = 17, f0: float = 25.0,
                         nsteps: int = 1000, nrec: int = 200) -> PveShot:
    """pve_vti_pml workload: the layered porous rock of pve_layered_shot
    made VTI: per layer Thomsen epsilon ~ U[0, 0.25] and delta ~
    U[-0.05, 0.15] of the frame, tortuosity along z T3 = T1 U[1, 1.6] and
    permeability along z kappa3 = kappa1 U[0.1, 1]; model arrays in
    sm_pve_create_vti's order (K_m K_s K_f phi mu rho_s rho_f T1 T3 eta
    kappa1 kappa3 Q fq epsilon delta).  dt at 40% of the RK4 pseudo-spectral
    stability limit of the fastest (horizontal) qP wave."""
    base = pve_layered_shot(n=n, np_=np_, h=h, seed=seed, f0=f0, nsteps=nsteps, nrec=nrec)
    rng = np.random.default_rng(seed + 1000)
    K_m, K_s, K_f, phi, mu, rho_s, rho_f, T, eta, kappa, Q, fq = base.model
    nz2 = base.model[0].shape[1]
    # layers of the interior model, extended into the layers like the others
    tops_src = base.model[0][n // 2 + np_]          # the K_m column identifies the layers
    _, lay = np.unique(tops_src, return_inverse=True)
    nl = int(lay.max()) + 1
    per = lambda lo, hi: rng.uniform(lo, hi, nl)[lay][None, :] * np.ones((base.model[0].shape[0], 1))
    eps, dl = per(0.0, 0.25), per(-0.05, 0.15)
    T3, kappa3 = T * per(1.0, 1.6), kappa * per(0.1, 1.0)
    model = (K_m, K_s, K_f, phi, mu, rho_s, rho_f, T, T3, eta, kappa, kappa3, Q, fq, eps, dl)
    vmax = float((biot_fast_velocity(K_m, K_s, K_f, phi, mu, rho_s, rho_f, T) * np.sqrt(1 + 2 * eps)).max())
    dt = 0.4 * 2.0 * h / (np.pi * vmax * np.sqrt(2.0))
    return PveShot(nx=n, nz=n, np=np_, h=h, dt=float(dt), f0=f0, nsteps=nsteps, model=model, src_idx=base.src_idx,
                   rec_idx=base.rec_idx, rec_comp=base.rec_comp)


def algorithmic_bytes_pve_vti(elt: int = 8) -> float:
    """As algorithmic_bytes_pve with the two further material arrays (c33,
    alpha3) read in each of the 4 stages: 345 values per step."""
    return elt * 345.0
