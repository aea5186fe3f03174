"""Measured workloads of the wave-propagation solvers.

One pass of a case is one shot (or one batch of shots) as a program of this
framework runs it: zero the wavefields, advance every time step, copy the
recorded traces (and for some cases a snapshot) back.  The model, geometry,
wavelet and tuned launch are in place before.  `exact` runs the same shot in
plain torch FP64, written from the schemes' equations.

Every solver runs FP32 and FP64 (its program selects either); the 3D solver
also stores its state in 16 bits.  Axis lengths, layer widths and step counts
come from the configurations, tests and benchmarks of this repository.
"""
from __future__ import annotations

import math

import numpy as np
import torch

SX, SZ, SXZ, SYZ, BULK, FZ, KURKJIAN = 0, 2, 4, 5, 6, 11, 12
VX, VY, VZ, QX, QZ, TXX, TZZ, TXZ, P, TXY, TYZ = 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10
VR, VT, TRR, TRT, TRZ, TTT, TTZ = 13, 14, 15, 16, 17, 18, 19


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # 3D acoustic: the headline shot (256^3 nodes, 20 layers), the launch
        # tuned once as the benchmark and a long survey do
        dict(name="a3d_f32_256", solver="a3d", nx=256, ny=256, nz=256, np=20, steps=120, storage="f32",
             mat16=False, tune=True),
        # a large grid with 16-bit state and material, the fast form of the
        # throughput configuration
        dict(name="a3d_bf16_360", solver="a3d", nx=360, ny=360, nz=300, np=20, steps=50, storage="bf16",
             mat16=True, tune=True),
        # an odd, flat grid as a drop-in program runs it: no tuning
        dict(name="a3d_f32_ragged", solver="a3d", nx=141, ny=203, nz=75, np=10, steps=200, storage="f32",
             mat16=False, tune=False),
        # 2D elastic: a small interactive shot, bound by latency
        dict(name="e2d_f32_small", solver="e2d", nx=150, nz=111, np=20, steps=250, storage="f32", shots=1),
        # the two-layer 400 x 400 configuration
        dict(name="e2d_f32_400", solver="e2d", nx=400, nz=400, np=20, steps=1000, storage="f32", shots=1),
        # a survey: independent shots of 300-1200 x 300-800 nodes and their
        # own step counts, advanced together and tuned as a batch
        dict(name="e2d_f32_batch", solver="e2d", nx=1200, nz=800, np=20, steps=300, storage="f32", shots=24),
        # cylindrical elastic: the borehole workload
        dict(name="cyl_f32_borehole", solver="cyl", nx=1000, nz=4000, np=20, steps=200, storage="f32", mode=0),
        # the program's default precision, azimuthal mode 1, odd sizes
        dict(name="cyl_f64_mode1", solver="cyl", nx=333, nz=1201, np=15, steps=250, storage="f64", mode=1,
             snapshot=True),
        # pseudo-spectral, SH waves: the 1000 x 1000 shot
        dict(name="sh_f32_1000", solver="sh", nx=1000, nz=1000, np=20, steps=150, storage="f32", L=1, snapshot=True),
        # P-SV waves at the program's default precision; axis lengths as a
        # model happens to have them (469 = 7*67 and 363 = 3*11*11 with layers)
        dict(name="ve_f64_ragged", solver="ve", nx=437, nz=331, np=16, steps=150, storage="f64", L=2, snapshot=True),
        # porous media: the 1000 x 1000 shot, and a VTI shot in FP64
        dict(name="pve_f32_1000", solver="pve", nx=1000, nz=1000, np=20, steps=100, storage="f32", L=1),
        dict(name="pve_vti_f64", solver="pve_vti", nx=600, nz=440, np=20, steps=100, storage="f64", L=1,
             snapshot=True),
    ]


MOST_BYTES = 1.0e11      # about the work of the largest listed case


def draw(rng):
    """One more case of the same solvers, sizes and options."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["a3d", "a3d", "e2d", "e2d", "cyl", "sh", "ve", "pve", "pve_vti"])
    if kind == "a3d":
        storage = rng.choice(["f32", "f32", "f32", "bf16", "f16", "f64"])
        c = dict(solver=kind, nx=size(40, 320), ny=size(40, 320), nz=size(40, 320), np=rng.choice([8, 10, 16, 20]),
                 steps=size(40, 200), storage=storage,
                 mat16=storage in ("bf16", "f16") and rng.random() < 0.5, tune=rng.random() < 0.3)
    elif kind == "e2d":
        c = dict(solver=kind, nx=size(60, 1200), nz=size(60, 800), np=rng.choice([10, 20, 30]), steps=size(60, 600),
                 storage="f32", shots=rng.choice([1, 1, rng.randint(2, 24)]))
        if c["shots"] == 1 and rng.random() < 0.25:
            c["storage"] = "f64"
    elif kind == "cyl":
        c = dict(solver=kind, nx=size(100, 1000), nz=size(200, 4000), np=rng.choice([10, 15, 20]),
                 steps=size(50, 250), storage=rng.choice(["f32", "f64"]), mode=rng.choice([0, 0, 1, 2]))
    else:
        c = dict(solver=kind, nx=size(100, 1000), nz=size(100, 1000), np=rng.choice([10, 16, 20]),
                 steps=size(30, 120), storage=rng.choice(["f32", "f64"]), L=rng.choice([1, 2]) if kind == "ve" else 1)
    if kind not in ("a3d", "e2d"):
        c["snapshot"] = rng.random() < 0.5
    w = work(c)["bytes"]
    if w > MOST_BYTES:
        c["steps"] = max(10, int(c["steps"] * MOST_BYTES / w))
    return c


def work(case):
    """Streaming minimum of the time steps: the state read and written and
    the material read once per update of the scheme (per step for leapfrog,
    per stage for the four Runge-Kutta stages of the spectral solvers)."""
    e = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}[case["storage"]]
    s, n = case["solver"], case["np"]
    if s == "a3d":
        d = [case[k] + 2 * n for k in ("nx", "ny", "nz")]
        me = 2 if case["mat16"] else 8 if e == 8 else 4
        per = 8 * e + 2 * me + 4 * e * sum(2.0 * n / x for x in d)
        cells, flops = float(np.prod(d)), 30.0
    elif s == "e2d":
        total = pml = 0.0
        for nx, nz, steps in _e2d_shots(case):
            t = (nx + 2 * n) * (nz + 2 * n)
            total += t * steps
            pml += (t - nx * nz) * steps
        return {"bytes": e * (13.0 * (total - pml) + 20.0 * pml), "flops": 40.0 * total}
    elif s == "cyl":
        nx2, nz2 = case["nx"] + n, case["nz"] + 2 * n
        cells = float(nx2 * nz2)
        per = e * (26.0 + 2.0 * (18 * (n + 1) * nz2 + 6 * nx2 * (2 * n + 1)) / cells)
        flops = 90.0
    else:
        nx2, nz2 = case["nx"] + 2 * n, case["nz"] + 2 * n
        cells = float(nx2 * nz2)
        state, mat, deriv = {"sh": (5, 9, 4), "ve": (7 + case["L"], 12 + 2 * case["L"], 8), "pve": (9, 13, 12),
                             "pve_vti": (9, 15, 12)}[s]
        per = 4 * e * (2.0 * state + mat)
        flops = 4 * (deriv * 5.0 * math.log2(nx2 * nz2) / 2 + 6.0 * state)
    return {"bytes": per * cells * case["steps"], "flops": flops * cells * case["steps"]}


def tolerance(case):
    """About four times the distance from `exact` over the listed cases: up
    to 2.5e-6 in FP32 and 1e-14 in FP64 (transforms
    over arbitrary lengths differ by more: the tests see 2e-14); the 16-bit
    state rounds every step, and an equally good rounding is as far off."""
    return {"rel": {"f64": 1e-13, "f32": 1e-5, "f16": 1e-2, "bf16": 3e-2}[case["storage"]]}


# ---------------------------------------------------------------------------
# models and geometry, from the seed alone
# ---------------------------------------------------------------------------
def _layers(rng, nz, count, *ranges):
    """Depth profiles of `count` layers, one per (lo, hi, sorted) range."""
    tops = np.sort(rng.choice(np.arange(1, nz), size=count - 1, replace=False))
    lay = np.searchsorted(tops, np.arange(nz), side="right")
    out = []
    for lo, hi, ordered in ranges:
        v = rng.uniform(lo, hi, count)
        out.append((np.sort(v) if ordered else v)[lay])
    return out


def _ripple(rng, n, modes=3):
    """A smooth unit-size profile along an axis of n nodes."""
    x = np.arange(n) / n
    return sum(np.cos(2 * np.pi * (k + 1) * x + rng.uniform(0, 2 * np.pi)) for k in range(modes)) / modes


def _ricker(f0, dt):
    """Ricker wavelet of peak 1 delayed by 1 / f0."""
    n = math.ceil(2.0 / (f0 * dt))
    t = np.arange(n) * dt - 1.0 / f0
    k = (math.pi * f0 * t) ** 2
    w = 2.0 * (math.pi * f0) ** 2 * (1.0 - 2.0 * k) * np.exp(-k)
    return w / np.abs(w).max()


def _lattice(rng, dims, count):
    """Flat indices of about `count` nodes spread over the whole grid."""
    per = max(2, int(round(count ** (1.0 / len(dims)))))
    axes = [np.unique(np.linspace(0, n - 1, min(per, n)).astype(np.int64)) for n in dims]
    return np.ravel_multi_index(np.meshgrid(*axes, indexing="ij"), dims).reshape(-1).astype(np.uintp)


def _a3d_shot(case, seed):
    rng = np.random.default_rng([seed, 1])
    n, dims = case["np"], (case["nx"], case["ny"], case["nz"])
    h, f0 = 10.0, 15.0
    (vz,) = _layers(rng, dims[2], 6, (1500.0, 4500.0, True))
    rip = [1.0 + 0.02 * _ripple(rng, d) for d in dims]
    vp = (rip[0][:, None, None] * rip[1][None, :, None]) * (vz * rip[2])[None, None, :]
    vp = np.pad(vp, n, mode="edge")
    rho = 310.0 * np.sqrt(np.sqrt(vp))
    dims2 = vp.shape
    dt = 0.49 * h / (math.sqrt(3.0) * vp.max())
    src = np.ravel_multi_index([[n + dims[0] // 2], [n + dims[1] // 2], [n + min(8, dims[2] - 1)]], dims2)
    side = 24
    rx = n + np.linspace(0, dims[0] - 1, side).astype(np.int64)
    ry = n + np.linspace(0, dims[1] - 1, side).astype(np.int64)
    surf = np.ravel_multi_index(np.meshgrid(rx, ry, [n + min(5, dims[2] - 1)], indexing="ij"), dims2).reshape(-1)
    near = np.clip(src[0] + np.arange(-6, 7)[:, None] * np.array([1, dims2[2], dims2[1] * dims2[2]])[None, :], 0,
                   np.prod(dims2) - 1).reshape(-1)
    lat = _lattice(rng, dims2, 512)
    rec = np.concatenate([surf, near, lat]).astype(np.uintp)
    comp = np.concatenate([np.full(surf.size, VZ), np.arange(near.size + lat.size) % 4 * 1]).astype(np.intc)
    comp[surf.size:] = np.array([P, VX, VY, VZ], np.intc)[comp[surf.size:]]
    return dict(vp=vp, rho=rho, h=h, f0=f0, dt=dt, src=src.astype(np.uintp), wav=_ricker(f0, dt), rec=rec, comp=comp)


def _e2d_shots(case):
    """Sizes and step counts of a case's shots (the same for every seed)."""
    if case["shots"] == 1:
        return [(case["nx"], case["nz"], case["steps"])]
    rng = np.random.default_rng([case["nx"], case["nz"], case["shots"]])
    return [(int(rng.integers(max(60, case["nx"] // 4), case["nx"] + 1)),
             int(rng.integers(max(60, case["nz"] * 3 // 8), case["nz"] + 1)),
             int(rng.integers(max(1, case["steps"] // 3), case["steps"] + 1))) for _ in range(case["shots"])]


def _e2d_shot(case, seed, k):
    rng = np.random.default_rng([seed, 2, k])
    nx, nz, steps = _e2d_shots(case)[k]
    h, f0 = 5.0, float(rng.uniform(15.0, 40.0))
    vp, ratio, rho = _layers(rng, nz, int(rng.integers(2, 7)), (2000.0, 5000.0, True), (1.7, 1.9, False),
                             (1800.0, 2700.0, False))
    lift = (1.0 + 0.01 * _ripple(rng, nx))[:, None]
    vp2, vs2 = lift * vp, lift * (vp / ratio)
    rho2 = np.broadcast_to(rho, (nx, nz)).copy()
    dt = 0.5 * h / (math.sqrt(2.0) * vp2.max())
    surf = np.arange(0, nx, 4) * nz
    lat = _lattice(rng, (nx, nz), 200)
    comp = np.concatenate([np.full(surf.size, VZ), np.array([VX, VZ, TXX, TZZ, TXZ])[np.arange(lat.size) % 5]])
    return dict(nx=nx, nz=nz, steps=steps, vp=vp2, vs=vs2, rho=rho2, h=h, f0=f0, dt=dt, type=BULK,
                src=np.array([(nx // 2) * nz + min(6, nz - 1)], np.uintp), wav=_ricker(f0, dt),
                rec=np.concatenate([surf, lat]).astype(np.uintp), comp=comp.astype(np.intc))


def _cyl_shot(case, seed):
    rng = np.random.default_rng([seed, 3])
    nx, nz, n = case["nx"], case["nz"], case["np"]
    dr, f0, hole = 0.01, 8000.0, 10
    vp, ratio, rho = _layers(rng, nz, 9, (2500.0, 4500.0, False), (1.7, 1.9, False), (2100.0, 2600.0, False))
    model = []
    for formation, fluid in ((vp, 1500.0), (vp / ratio, 0.0), (rho, 1000.0)):
        a = np.repeat(formation[None, :], nx, axis=0)
        a[:hole] = fluid
        model.append(np.pad(a, ((0, n), (n, n)), mode="edge"))
    nx2, nz2 = nx + n, nz + 2 * n
    dt = 0.6 * dr / (math.sqrt(2.0) * vp.max())
    zc = n + nz // 2
    lam = float(model[2][0, zc] * model[0][0, zc] ** 2)
    kind, src, wav = KURKJIAN, zc, 1e-6 * lam / math.pi / (dr * dr * dr) * _ricker(f0, dt)
    if case["mode"]:              # a force off the axis: the monopole wavelet vanishes there for n > 0
        kind, src, wav = FZ, 12 * nz2 + zc, _ricker(f0, dt)
    line = nz2 + np.arange(n, n + nz, 20)
    near = (np.arange(2, 40)[:, None] * nz2 + zc + np.array([-15, 15])[None, :]).reshape(-1)
    lat = _lattice(rng, (nx2, nz2), 300)
    comps = np.array([VR, VT, VZ, TRR, TTT, TZZ, TRZ, TRT, TTZ])
    comp = np.concatenate([np.full(line.size, TRR), comps[np.arange(near.size + lat.size) % 9]])
    return dict(model=model, dr=dr, f0=f0, dt=dt, type=kind, src=np.array([src], np.uintp), wav=wav,
                rec=np.concatenate([line, near, lat]).astype(np.uintp), comp=comp.astype(np.intc))


def _pstd_shot(case, seed):
    rng = np.random.default_rng([seed, 4])
    s, nx, nz, n = case["solver"], case["nx"], case["nz"], case["np"]
    h, f0 = 5.0, 25.0
    lift = 1.0 + 0.01 * _ripple(rng, nx)[:, None]
    grid = lambda a: np.pad(np.broadcast_to(a, (nx, nz)), n, mode="edge")
    count = int(rng.integers(5, 11))
    if s == "sh":
        vs, rho, gamma, Q = _layers(rng, nz, count, (800.0, 2500.0, True), (1800.0, 2600.0, False),
                                    (0.0, 0.25, False), (20.0, 100.0, False))
        vs = vs * lift
        model = [vs * vs * rho * 1e-9, rho, gamma, Q, f0]
        vmax, kind, comps = (vs * np.sqrt(1 + 2 * gamma)).max(), SYZ, [VY, TXY, TYZ]
    elif s == "ve":
        vp, ratio, rho, eps, dl, Q2, *Q1 = _layers(
            rng, nz, count, (1800.0, 4000.0, True), (1.7, 2.2, False), (1800.0, 2600.0, False), (0.0, 0.25, False),
            (-0.05, 0.15, False), (20.0, 100.0, False), *[(20.0, 100.0, False)] * case["L"])
        vp = vp * lift
        mu = (vp / ratio) ** 2 * rho
        f1 = [5.0 + 55.0 * (m + 0.5) / case["L"] for m in range(case["L"])]
        model = [1e-9 * (vp * vp * rho - 4.0 / 3.0 * mu), mu * 1e-9, rho, eps, dl, Q1, f1, Q2, f0]
        vmax, kind, comps = (vp * np.sqrt(1 + 2 * eps)).max(), BULK, [VX, VZ, TXX, TZZ, TXZ]
    else:
        Ks, Km, phi, mu, rs, T, kap, Q, eps, dl, t3, k3 = _layers(
            rng, nz, count, (33.0, 39.0, False), (4.0, 16.0, True), (0.1, 0.32, False), (3.0, 12.0, True),
            (2600.0, 2700.0, False), (1.5, 3.0, False), (50.0, 2000.0, False), (20.0, 100.0, False),
            (0.0, 0.25, False), (-0.05, 0.15, False), (1.0, 1.6, False), (0.1, 1.0, False))
        mu = mu * lift
        alpha = 1 - Km / Ks
        M = 1.0 / ((alpha - phi) / Ks + phi / 2.25)
        rho = (1 - phi) * rs + phi * 1000.0
        # above the fast wave for any coupling of solid and fluid
        vmax = 1.05 * np.sqrt(1e9 * (Km + 4.0 / 3.0 * mu + alpha * alpha * M) / (rho - 1000.0 * phi / T)).max()
        kind, comps = BULK, [VX, VZ, QX, QZ, TXX, TZZ, TXZ, P]
        if s == "pve":
            model = [Km, Ks, 2.25, phi, mu, rs, 1000.0, T, 1.0, kap, Q, f0]
        else:
            vmax = vmax * math.sqrt(1 + 2 * eps.max())
            model = [Km, Ks, 2.25, phi, mu, rs, 1000.0, T, T * t3, 1.0, kap, kap * k3, Q, f0, eps, dl]
    model = [np.stack([grid(b) for b in a]) if isinstance(a, list) else grid(a) for a in model]
    dt = 0.4 * 2.0 * h / (math.pi * float(vmax) * math.sqrt(2.0))
    dims2 = (nx + 2 * n, nz + 2 * n)
    src = (nx // 2 + n) * dims2[1] + n + 6
    line = np.linspace(n, nx + n - 1, 200).astype(np.int64) * dims2[1] + n + 10
    near = (src + np.arange(-10, 11)[:, None] * np.array([1, dims2[1], dims2[1] + 1])[None, :]).reshape(-1)
    lat = _lattice(rng, dims2, 300)
    comp = np.concatenate([np.full(line.size, VY if s == "sh" else VZ),
                           np.array(comps)[np.arange(near.size + lat.size) % len(comps)]])
    return dict(model=model, h=h, f0=f0, dt=dt, type=kind, src=np.array([src], np.uintp),
                wav=_ricker(f0, 0.5 * dt) / (h * h), rec=np.concatenate([line, near, lat]).astype(np.uintp),
                comp=comp.astype(np.intc))


# ---------------------------------------------------------------------------
# the framework's side
# ---------------------------------------------------------------------------
_CTX = None


def _context():
    """One context for the process, as a program has."""
    global _CTX
    if _CTX is None:
        from seismod_amd.solver import Context
        _CTX = Context(0)
    return _CTX


def prepare(case, seed):
    from seismod_amd import autotune, solver as S
    ctx, s = _context(), case["solver"]
    if s == "a3d":
        d = _a3d_shot(case, seed)
        sim = S.Acoustic3D(ctx, S.A3dConfig(
            nx=case["nx"], ny=case["ny"], nz=case["nz"], np=case["np"], dx=d["h"], dy=d["h"], dz=d["h"], dt=d["dt"],
            f0=d["f0"], storage=case["storage"], mat16=case["mat16"]), d["vp"], d["rho"])
        sim.set_sources(d["src"], [d["wav"].size], d["wav"])
        if case["tune"] and case["storage"] != "f64":
            autotune.tune_a3d(sim, ctx)
    elif s == "e2d":
        sims, steps = [], []
        for k in range(case["shots"]):
            d = _e2d_shot(case, seed, k)
            sim = S.Elastic2D(ctx, S.E2dConfig(nx=d["nx"], nz=d["nz"], npml=case["np"], h=d["h"], dt=d["dt"],
                                               storage=case["storage"]), d["vp"], d["vs"], d["rho"])
            sim.set_sources([d["type"]], d["src"], [d["wav"].size], d["wav"])
            sim.set_receivers(d["rec"], d["comp"], d["steps"])
            sims.append(sim)
            steps.append(d["steps"])
        if case["shots"] > 1:
            batch = S.E2dBatch(ctx)
            batch.set_variant(autotune.tune_e2d_batch(sims, ctx)[1])
            autotune.tune_e2d_groups(batch, sims)
            return dict(batch=batch, sims=sims, steps=steps)
        return dict(sim=sim, steps=steps[0], snapshot=VZ)
    elif s == "cyl":
        d = _cyl_shot(case, seed)
        sim = S.Cylindrical(ctx, S.CylConfig(nx=case["nx"], nz=case["nz"], np=case["np"], dr=d["dr"], dz=d["dr"],
                                             dt=d["dt"], f0=d["f0"], mode=case["mode"], storage=case["storage"]),
                            *d["model"])
        sim.set_sources([d["type"]], d["src"], [d["wav"].size], d["wav"])
    else:
        d = _pstd_shot(case, seed)
        make, config = {"sh": (S.ViscoelasticSH, S.ShConfig), "ve": (S.ViscoelasticPSV, S.VeConfig),
                        "pve": (S.Poroviscoelastic, S.PveConfig),
                        "pve_vti": (S.PoroviscoelasticVTI, S.PveConfig)}[s]
        more = {"L": case["L"]} if s == "ve" else {}
        sim = make(ctx, config(nx=case["nx"], nz=case["nz"], np=case["np"], dx=d["h"], dz=d["h"], dt=d["dt"],
                               f0=d["f0"], storage=case["storage"], **more), *d["model"])
        sim.set_sources([d["type"]], d["src"], [d["wav"].size], d["wav"])
    sim.set_receivers(d["rec"], d["comp"], case["steps"])
    return dict(sim=sim, steps=case["steps"], slice=(P, case["ny"] // 2 + case["np"]) if s == "a3d" else None,
                snapshot=("vy" if s == "sh" else "vz") if case.get("snapshot") else None)


def run(state):
    if "batch" in state:
        for sim in state["sims"]:
            sim.reset()
        state["batch"].run(state["sims"], state["steps"])
        return [sim.traces(0, n) for sim, n in zip(state["sims"], state["steps"])]
    sim = state["sim"]
    sim.reset()
    sim.run(state["steps"])
    out = {"traces": sim.traces(0, state["steps"])}
    if state.get("slice"):
        out["snapshot"] = sim.slice_xz(*state["slice"])
    elif state.get("snapshot") is not None:
        out["snapshot"] = sim.field(state["snapshot"])
    return out


# ---------------------------------------------------------------------------
# the same shots in plain torch, FP64
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=_dev())


class _Recorder:
    """Values of field comp[r] at flat index rec[r] after every step."""

    def __init__(self, d, steps, fields):
        self.out = torch.zeros((steps, d["rec"].size), dtype=torch.float64, device=_dev())
        self.groups = []
        for c in np.unique(d["comp"]):
            where = np.nonzero(d["comp"] == c)[0]
            self.groups.append((fields[int(c)], torch.as_tensor(where, device=_dev()),
                                torch.as_tensor(d["rec"][where].astype(np.int64), device=_dev())))

    def __call__(self, it, W):
        for key, where, idx in self.groups:
            self.out[it, where] = W[key].reshape(-1)[idx]


def exact(case, seed):
    s = case["solver"]
    if s == "a3d":
        return _exact_a3d(case, _a3d_shot(case, seed))
    if s == "e2d":
        if case["shots"] > 1:
            return [_exact_e2d(case, _e2d_shot(case, seed, k))["traces"] for k in range(case["shots"])]
        return _exact_e2d(case, _e2d_shot(case, seed, 0))
    if s == "cyl":
        return _exact_cyl(case, _cyl_shot(case, seed))
    return _exact_pstd(case, _pstd_shot(case, seed))


def _exact_a3d(case, d):
    """Pressure-velocity leapfrog; convolutional PML of profile (x/L)^2,
    reflection 1e-5 at 5000 m/s, alpha falling from pi f0 at the interior."""
    n, h, dt = case["np"], d["h"], d["dt"]
    vp, rho = _t(d["vp"]), _t(d["rho"])
    dims = vp.shape

    def table(ax, half):
        pos = np.arange(dims[ax]) + (0.5 if half else 0.0)
        x = np.maximum(np.maximum(n - pos, pos - (dims[ax] - 1 - n)), 0.0) / n
        dd, al = -3.0 * 5000.0 * math.log(1e-5) / (2.0 * n * h) * x ** 2, math.pi * d["f0"] * (1.0 - x)
        b = np.where(x > 0, np.exp(-(dd + al) * dt), 1.0)
        a = np.where(x > 0, dd * (b - 1.0) / np.where(x > 0, dd + al, 1.0), 0.0)
        shape = [1, 1, 1]
        shape[ax] = -1
        return _t(a).reshape(shape), _t(b).reshape(shape)

    K = rho * vp * vp * dt
    Pf = torch.zeros_like(vp)
    v, mv, mp, tab, irho = [], [], [], [], []
    for ax in range(3):
        m = dims[ax]
        lo, hi = rho.narrow(ax, 0, m - 1), rho.narrow(ax, 1, m - 1)
        irho.append(2.0 * dt / (lo + hi))
        v.append(torch.zeros_like(vp))
        mv.append(torch.zeros_like(lo))
        mp.append(torch.zeros_like(vp))
        ah, bh = table(ax, True)
        tab.append((ah.narrow(ax, 0, m - 1), bh.narrow(ax, 0, m - 1)) + table(ax, False))
    del vp, rho
    inner = tuple(slice(1, None) for _ in range(3))
    W = {P: Pf, VX: v[0], VY: v[1], VZ: v[2]}
    rec = _Recorder(d, case["steps"], {k: k for k in W})
    si = int(d["src"][0])
    for it in range(case["steps"]):
        for ax in range(3):
            m = dims[ax]
            dp = (Pf.narrow(ax, 1, m - 1) - Pf.narrow(ax, 0, m - 1)) / h
            mv[ax].mul_(tab[ax][1]).addcmul_(tab[ax][0].expand_as(dp), dp)
            v[ax].narrow(ax, 0, m - 1).sub_(irho[ax] * dp.add_(mv[ax]))
        div = None
        for ax in range(3):
            m = dims[ax]
            prev = [slice(1, None)] * 3
            prev[ax] = slice(0, m - 1)
            dv = (v[ax][inner] - v[ax][tuple(prev)]) / h
            a, b = tab[ax][2], tab[ax][3]
            a, b = a.narrow(ax, 1, m - 1), b.narrow(ax, 1, m - 1)
            q = mp[ax][inner]
            q.mul_(b).addcmul_(a.expand_as(dv), dv)
            dv.add_(q)
            div = dv if div is None else div.add_(dv)
        Pf[inner].sub_(K[inner] * div)
        if it < d["wav"].size:
            Pf.reshape(-1)[si] += dt * d["wav"][it] * 1e6
        rec(it, W)
    return {"traces": rec.out, "snapshot": Pf[:, case["ny"] // 2 + n, :].contiguous()}


def _exact_e2d(case, d):
    """Velocity-stress leapfrog on the padded grid with split fields in the
    layers, damping d0 (distance / width)^2 at each staggered position."""
    nx, nz, n, h, dt = d["nx"], d["nz"], case["np"], d["h"], d["dt"]
    NX, NZ = nx + 2 * n, nz + 2 * n
    vp, vs, rho = d["vp"], d["vs"], d["rho"]
    mu0, lam0, b0 = rho * vs * vs, rho * (vp * vp - 2.0 * vs * vs), 1.0 / rho
    l2m0 = lam0 + 2.0 * mu0
    la, l2m, mu, bm = lam0.copy(), l2m0.copy(), mu0.copy(), b0.copy()
    mu[:, :-1] = 0.5 * (mu0[:, :-1] + mu0[:, 1:])
    la[:-1] = 0.5 * (lam0[:-1] + lam0[1:])
    l2m[:-1] = 0.5 * (l2m0[:-1] + l2m0[1:])
    bm[:-1, :-1] = 0.25 * (b0[:-1, :-1] + b0[1:, :-1] + b0[:-1, 1:] + b0[1:, 1:])
    bm[:-1, -1] = 0.5 * (b0[:-1, -1] + b0[1:, -1])
    bm[-1, :-1] = 0.5 * (b0[-1, :-1] + b0[-1, 1:])
    at = np.ix_(np.clip(np.arange(NX) - n, 0, nx - 1), np.clip(np.arange(NZ) - n, 0, nz - 1))
    B, BM, LA, L2M, MU = (a[at] for a in (b0, bm, la, l2m, mu))
    if nx <= nz:          # the scheme's lower-right corner takes the material of cell nx*nx - 1
        q = divmod(nx * nx - 1, nz)
        LA[n + nx:, n + nz:], L2M[n + nx:, n + nz:] = la[q], l2m[q]
    B, BM, LA, L2M, MU = (_t(a) * (dt / h) for a in (B, BM, LA, L2M, MU))
    d0 = math.log(1e3) * 1.5 * vp.mean() / (n * h)

    def damp(m, count, half):
        """Factors of the old value and of the increment."""
        pos = np.arange(count) - n + (0.5 if half else 0.0)
        r = dt * d0 * (np.maximum(np.maximum(-pos, pos - (m - 1)), 0.0) / n) ** 2
        r[n:n + m] = 0.0
        return _t((2.0 - r) / (2.0 + r)), _t(2.0 / (2.0 + r))

    xi, xh = ([a[:, None] for a in damp(nx, NX, f)] for f in (False, True))
    zi, zh = ([a[None, :] for a in damp(nz, NZ, f)] for f in (False, True))

    def down(a, ax):      # value of the next node, 0 past the end
        o = torch.zeros_like(a)
        o.narrow(ax, 0, a.shape[ax] - 1).copy_(a.narrow(ax, 1, a.shape[ax] - 1))
        return o

    def up(a, ax):
        o = torch.zeros_like(a)
        o.narrow(ax, 1, a.shape[ax] - 1).copy_(a.narrow(ax, 0, a.shape[ax] - 1))
        return o

    # halves split by the direction of the derivative (their sum is the field)
    names = (VX, VZ, TXX, TZZ, TXZ)
    X = {k: torch.zeros((NX, NZ), dtype=torch.float64, device=_dev()) for k in names}
    Z = {k: torch.zeros_like(X[k]) for k in names}
    F = {k: torch.zeros_like(X[k]) for k in names}

    def step(k, dxv, cx, kx, dzv, cz, kz):
        X[k] = kx[0] * X[k] + kx[1] * (cx * dxv)
        Z[k] = kz[0] * Z[k] + kz[1] * (cz * dzv)
        F[k] = X[k] + Z[k]

    inside = {k: k for k in names}
    rec = _Recorder(d, d["steps"], inside)
    si, sj = divmod(int(d["src"][0]), nz)
    for it in range(d["steps"]):
        txx, tzz, txz = F[TXX], F[TZZ], F[TXZ]
        step(VX, txx - up(txx, 0), B, xi, txz - up(txz, 1), B, zi)
        step(VZ, down(txz, 0) - txz, BM, xh, down(tzz, 1) - tzz, BM, zh)
        vx, vz = F[VX], F[VZ]
        exx, ezz = down(vx, 0) - vx, vz - up(vz, 1)
        step(TXX, exx, L2M, xh, ezz, LA, zi)
        step(TZZ, exx, LA, xh, ezz, L2M, zi)
        step(TXZ, vz - up(vz, 0), MU, xi, down(vx, 1) - vx, MU, zh)
        if it < d["wav"].size:
            for k in (TXX, TZZ):
                X[k][si + n, sj + n] += dt * d["wav"][it]
                F[k][si + n, sj + n] += dt * d["wav"][it]
        rec(it, {k: F[k][n:n + nx, n:n + nz] for k in names})
    return {"traces": rec.out, "snapshot": F[VZ][n:n + nx, n:n + nz].contiguous()}


def _exact_cyl(case, d):
    """Velocity-stress leapfrog in (r, z) for azimuthal mode m, staggered
    (trz at nodes; vz, ttz half a cell along r; vr, trt along z; vt and the
    normal stresses along both), convolutional PML on the outer r side and
    both z ends."""
    nx, nz, n, h, dt, mode = case["nx"], case["nz"], case["np"], d["dr"], d["dt"], case["mode"]
    vp, vs, rho = (_t(a) for a in d["model"])
    nx2, nz2 = vp.shape
    m = rho * vs * vs
    lam = rho * (vp * vp - 2.0 * vs * vs)
    l2m, bij = lam + 2.0 * m, 1.0 / rho

    def harm(*q):
        """Harmonic mean, 0 where two or more of four (any of two) vanish."""
        if len(q) == 2:
            den, num = q[0] + q[1], 2.0 * q[0] * q[1]
        else:
            p, a, b, c = q
            den, num = a * b * c + p * b * c + p * a * c + p * a * b, 4.0 * p * a * b * c
        return torch.where(den == 0.0, torch.zeros_like(den), num / torch.where(den == 0.0, torch.ones_like(den), den))

    muj, mui, mu = m.clone(), m.clone(), m.clone()
    bj, bi = bij.clone(), bij.clone()
    muj[:, 1:] = harm(m[:, 1:], m[:, :-1])
    bj[:, 1:] = 2.0 / (rho[:, 1:] + rho[:, :-1])
    mui[1:] = harm(m[1:], m[:-1])
    bi[1:] = 2.0 / (rho[1:] + rho[:-1])
    mu[0, 1:], mu[1:, 0] = harm(m[0, 1:], m[0, :-1]), harm(m[1:, 0], m[:-1, 0])
    mu[1:, 1:] = harm(m[1:, 1:], m[1:, :-1], m[:-1, 1:], m[:-1, :-1])

    d0 = -3.0 * 5000.0 * math.log(1e-5) / (2.0 * n * h)

    def bc(x, alpha):
        dd = d0 * x ** 2
        b = np.exp(-(dd + alpha) * dt)
        return b, dd * (b - 1.0) / (dd + alpha)

    k, amax = np.arange(n), math.pi * d["f0"]
    kk = np.arange(n + 1)
    node = bc((n - k) / n, k * amax / n)                                   # whole nodes, outermost first
    near = bc((n - k - 0.5) / n, (k + 0.5) * amax / n)                     # half nodes of the low side
    far = bc((kk + 0.5) / n, (n - kk - 0.5) * amax / (n + 1))              # half nodes of the high side, inner first

    def zcoef(half, bottom):
        """Rows b and c along z: layers at the top and from `bottom` on."""
        b, c = np.ones(nz2), np.zeros(nz2)
        if half:
            b[:n], c[:n] = near
            w = nz2 - bottom
            b[bottom:], c[bottom:] = far[0][:w], far[1][:w]
        else:
            b[:n], c[:n] = node
            b[nz + n:], c[nz + n:] = node[0][::-1], node[1][::-1]
        on = c != 0.0
        return _t(b)[None, :], _t(c)[None, :], torch.as_tensor(on, device=_dev())[None, :]

    def rcoef(half, start):
        b, c = np.ones(nx2), np.zeros(nx2)
        w = nx2 - start
        if half:
            b[start:], c[start:] = far[0][:w], far[1][:w]
        else:
            b[start:], c[start:] = node[0][::-1], node[1][::-1]
        on = c != 0.0
        return _t(b)[:, None], _t(c)[:, None], torch.as_tensor(on, device=_dev())[:, None]

    zh, zt, zn = zcoef(True, nz + n - 1), zcoef(True, nz + n), zcoef(False, 0)
    rn, rh, rt = rcoef(False, nx), rcoef(True, nx - 1), rcoef(True, nx)
    mem = {}

    def pml(name, coef, x, rows, cols):
        """x of cells [rows) x [cols) corrected by its memory variable."""
        b, c, on = coef
        b, c, on = ((q[rows] if q.shape[0] > 1 else q[:, cols]) for q in (b, c, on))
        q = mem.get(name)
        q = c * x if q is None else b * q + c * x
        mem[name] = q = torch.where(on, q, torch.zeros_like(q))
        return x + q

    F = {f: torch.zeros((nx2, nz2), dtype=torch.float64, device=_dev())
         for f in (VR, VT, VZ, TRR, TTT, TZZ, TRZ, TRT, TTZ)}
    r_ = (torch.arange(nx2, dtype=torch.float64, device=_dev()) * h)[:, None]
    rhalf = r_ + 0.5 * h
    a1, a0, up1, lo = slice(1, None), slice(0, None), slice(1, None), slice(0, -1)
    rec = _Recorder(d, case["steps"], {f: f for f in F})
    si = int(d["src"][0])
    for it in range(case["steps"]):
        # v_r, rows 1.. (row 0 in odd modes), columns ..-1
        ddz = pml("vr_z", zh, (F[TRZ][:, 1:] - F[TRZ][:, :-1]) / h, a0, lo)
        s = (up1, lo)
        t, u = F[TRR][:, :-1], F[TTT][:, :-1]
        acc = pml("vr_r", rn, (t[1:] - t[:-1]) / h, a1, lo) + pml("vr_t", rn, (t[1:] + t[:-1]) / (2 * r_[1:]), a1, lo)
        acc = acc - pml("vr_u", rn, (u[1:] + u[:-1]) / (2 * r_[1:]), a1, lo) + ddz[1:]
        if mode:
            acc = acc + mode * pml("vr_m", rn, F[TRT][s] / r_[1:], a1, lo)
        if mode % 2:
            F[VR][0, :-1] += dt * bj[0, :-1] * (2.0 * t[0] / h + ddz[0])
        F[VR][s] += dt * bj[s] * acc
        # v_theta, rows ..-1, columns ..-1
        s = (lo, lo)
        t = F[TRT][:, :-1]
        acc = pml("vt_t", rh, (t[1:] + t[:-1]) / rhalf[:-1], lo, lo) + pml("vt_r", rh, (t[1:] - t[:-1]) / h, lo, lo)
        acc = acc + pml("vt_z", zh, (F[TTZ][:-1, 1:] - F[TTZ][:-1, :-1]) / h, lo, lo)
        if mode:
            acc = acc - mode * pml("vt_m", rh, F[TTT][s] / rhalf[:-1], lo, lo)
        F[VT][s] += dt * bij[s] * acc
        # v_z, rows ..-1, columns 1..
        s = (lo, up1)
        t = F[TRZ][:, 1:]
        acc = pml("vz_z", zn, (F[TZZ][:-1, 1:] - F[TZZ][:-1, :-1]) / h, lo, up1)
        acc = acc + pml("vz_r", rh, (t[1:] - t[:-1]) / h, lo, up1)
        acc = acc + pml("vz_t", rh, (t[1:] + t[:-1]) / (2 * rhalf[:-1]), lo, up1)
        if mode:
            acc = acc + mode * pml("vz_m", rh, F[TTZ][s] / rhalf[:-1], lo, up1)
        F[VZ][s] += dt * bi[s] * acc
        if d["type"] == FZ and it < d["wav"].size:
            F[VZ].reshape(-1)[si] += dt * bi.reshape(-1)[si] * d["wav"][it]
        # normal stresses, rows ..-1, columns ..-1
        s = (lo, lo)
        t = F[VR][:, :-1]
        err = pml("n_r", rh, (t[1:] - t[:-1]) / h, lo, lo)
        ett = pml("n_t", rh, (t[1:] + t[:-1]) / (2 * rhalf[:-1]), lo, lo)
        ezz = pml("n_z", zh, (F[VZ][:-1, 1:] - F[VZ][:-1, :-1]) / h, lo, lo)
        if mode:
            ett = ett + mode * pml("n_m", rh, F[VT][s] / rhalf[:-1], lo, lo)
        F[TRR][s] += dt * (l2m[s] * err + lam[s] * (ett + ezz))
        F[TTT][s] += dt * (l2m[s] * ett + lam[s] * (err + ezz))
        F[TZZ][s] += dt * (l2m[s] * ezz + lam[s] * (err + ett))
        # tau_rz, rows 1.., columns 1..
        s = (up1, up1)
        F[TRZ][s] += dt * mu[s] * (pml("rz_z", zt, (F[VR][1:, 1:] - F[VR][1:, :-1]) / h, a1, up1) +
                                   pml("rz_r", rt, (F[VZ][1:, 1:] - F[VZ][:-1, 1:]) / h, a1, up1))
        # tau_rtheta, rows 1.. (row 0 in odd modes)
        t = F[VT]
        if mode % 2:
            F[TRT][0] += dt * muj[0] * (2.0 * t[0] / h)
        acc = pml("rt_r", rn, (t[1:] - t[:-1]) / h, a1, a0) - pml("rt_t", rn, (t[1:] + t[:-1]) / (2 * r_[1:]), a1, a0)
        if mode:
            acc = acc - mode * pml("rt_m", rn, F[VR][1:] / r_[1:], a1, a0)
        F[TRT][1:] += dt * muj[1:] * acc
        # tau_thetaz, rows ..-1, columns 1..
        s = (lo, up1)
        acc = pml("tz_z", zn, (F[VT][:-1, 1:] - F[VT][:-1, :-1]) / h, lo, up1)
        if mode:
            acc = acc - mode * pml("tz_m", rh, F[VZ][s] / rhalf[:-1], lo, up1)
        F[TTZ][s] += dt * mui[s] * acc
        if d["type"] == KURKJIAN and it < d["wav"].size:
            F[TRR].reshape(-1)[si] += dt * d["wav"][it]
            F[TZZ].reshape(-1)[si] += dt * d["wav"][it]
        rec(it, F)
    return {"traces": rec.out, "snapshot": F[VZ]} if case.get("snapshot") else {"traces": rec.out}


def _exact_pstd(case, d):
    """Runge-Kutta 4 with spectral derivatives at half-cell shifts; the layers
    correct each derivative by memory variables stepped semi-implicitly."""
    s, n, h, dt, L = case["solver"], case["np"], d["h"], d["dt"], case["L"]
    model = [_t(a) for a in d["model"]]
    nx2, nz2 = model[0].shape
    N = nx2 * nz2
    half = {}                                       # i k e^{+-i k h / 2} per axis and direction
    for ax, m in ((0, nx2), (1, nz2)):
        k = 2.0 * math.pi * torch.arange(m // 2 + 1, dtype=torch.float64, device=_dev()) / (h * m)
        for sgn in (1, -1):
            q = 1j * k * torch.exp(0.5j * sgn * k * h)
            half[ax, sgn] = q[:, None] if ax == 0 else q[None, :]

    def deriv(f, ax, sgn):
        return torch.fft.irfft(torch.fft.rfft(f, dim=ax) * half[ax, sgn], n=f.shape[ax], dim=ax)

    d0, amax = -3.0 * 5000.0 * math.log(1e-5) / (2.0 * n * h), math.pi * d["f0"]
    m_ = np.arange(n + 1)

    def rows(shift, step):
        """b and c of the layer rows, outermost first; step 0: none."""
        x = np.where(n - m_ + shift > 0, (n - m_ + shift) / n, 0.0)
        dd, al = d0 * x ** 2, (m_ - shift) * amax / n
        if step == 0.0:
            return torch.ones(n + 1, 1, dtype=torch.float64, device=_dev()), _t(np.zeros(n + 1))[:, None]
        q = 1.0 + 0.5 * step * (dd + al)
        return _t((1.0 - 0.5 * step * (dd + al)) / q)[:, None], _t(-dd * step / q)[:, None]

    tabs = [{k: rows(sh, st) for k, sh in (("n", 0.0), ("i", -0.5), ("o", 0.5))} for st in (0.0, 0.5 * dt, dt)]
    slots = (2 * n + 1) * max(nx2, nz2)
    mem = {}

    def layer(name, t, ax, tab, sgn, limit):
        """t with its layers corrected; ax: direction of the layers.  sgn -1
        takes node rows on both sides, +1 inner half nodes on the low side and
        outer half nodes on the far side, one row more."""
        if name not in mem:
            mem[name] = [torch.zeros(slots, dtype=torch.float64, device=_dev()) for _ in range(3)] + [limit]
        m0, m1, m2, _ = mem[name]
        far = n + 1 if sgn > 0 or name == "dx_txy" else n
        u = t if ax == 0 else t.T
        cols, last = u.shape[1], u.shape[0]
        for q0, w, view, (b, c) in ((0, n, slice(0, n), tab["i" if sgn > 0 else "n"]),
                                    (n * cols, far, slice(last - far, last), tab["o" if sgn > 0 else "n"])):
            q = slice(q0, q0 + w * cols)
            x = u[view] if q0 == 0 else u[view].flip(0)
            m1[q] = (b[:w] * m0[q].view(w, cols) + c[:w] * x).reshape(-1)
            y = x + m2[q].view(w, cols)
            u[view] = y if q0 == 0 else y.flip(0)
        return t

    def avg(a, ax):
        """Mean with the next node; the last row or column as the one before."""
        o = torch.empty_like(a)
        m = a.shape[ax]
        o.narrow(ax, 0, m - 1).copy_(0.5 * (a.narrow(ax, 0, m - 1) + a.narrow(ax, 1, m - 1)))
        o.narrow(ax, m - 1, 1).copy_(o.narrow(ax, m - 2, 1))
        return o

    def corner(a, harmonic=False):
        r = 1.0 / a if harmonic else a
        o = torch.empty_like(a)
        c = 0.25 * (r[:-1, :-1] + r[1:, :-1] + r[:-1, 1:] + r[1:, 1:])
        o[:-1, :-1] = 1.0 / c if harmonic else c
        o[-1, :-1] = o[-2, :-1]
        o[:, -1] = o[:, -2]
        return o

    def relax(Q, f):
        """tau_s and tau_s / tau_e of a standard linear solid."""
        r = torch.sqrt(Q * Q + 1.0)
        return (r - 1.0) / (2.0 * math.pi * f * Q), (r - 1.0) / (r + 1.0)

    X1, Z1 = (2 * n + 1) * nz2, (2 * n + 1) * nx2
    D = lambda W, q, name, ax, sgn, tab, lay=None: layer(
        name, deriv(W[q], ax, sgn), ax if lay is None else lay, tab, sgn, (X1, Z1)[ax])
    inner = (slice(1, -1), slice(1, -1))

    if s == "sh":
        fields, nstate, inject = {TXY: 0, TYZ: 1, VY: 2}, 5, (1,)
        mu, rho, gamma, Q, f = model
        mu, irho = mu * 1e3, 1e6 / rho
        ts2, eta2 = relax(avg(Q, 0), avg(f, 0))
        ts1, eta1 = relax(avg(Q, 1), avg(f, 1))
        cx = avg(mu, 0) * (1.0 + 2.0 * avg(gamma, 0))
        cz = avg(mu, 1)
        cz0 = cz * eta2
        cz0[:, -1] = cz0[:, -2]

        def rhs(W, o, tab):
            t = D(W, 0, "dx_txy", 0, -1, tab) + D(W, 1, "dz_tyz", 1, -1, tab)
            o[2][inner] = (irho * t)[inner]
            t = D(W, 2, "dz_vy", 1, 1, tab)
            o[3] = ((1.0 - 1.0 / eta1) * t - W[3]) / ts1
            o[1] = cz * t + cz0 * W[3]
            # the scheme corrects D_x v_y in the z layers, inner rows by the x tables
            t = D(W, 2, "dx_vy", 0, 1, tab, lay=1)
            o[4] = ((1.0 - 1.0 / eta2) * t - W[4]) / ts2
            o[0] = cx * t + cx * eta2 * W[4]
    elif s == "ve":
        fields, nstate, inject = {TXX: 0, TZZ: 1, TXZ: 2, VX: 3, VZ: 4}, 7 + L, (0, 1)
        K, mu, rho, eps, dl, Q1, f1, Q2, f2 = model
        K, mu, rho = K * 1e3, mu * 1e3, rho * 1e-6
        c33 = K + 4.0 / 3.0 * mu
        c11 = (1.0 + 2.0 * eps) * c33
        c13 = torch.sqrt(2.0 * dl * c33 * (c33 - mu) + (c33 - mu) ** 2) - mu
        ts1, eta1 = relax(Q1, f1)
        ts2, eta2 = relax(Q2, f2)
        K0 = (0.5 * (c11 + c33) - mu) * eta1.sum(0)
        ci, ts_ij, eta_ij = corner(mu, True), corner(ts2), corner(eta2)
        irx, irz = 1.0 / avg(rho, 0), 1.0 / avg(rho, 1)

        def rhs(W, o, tab):
            o[3][inner] = (irx * (D(W, 0, "dx_txx", 0, 1, tab) + D(W, 2, "dz_txz", 1, -1, tab)))[inner]
            o[4][inner] = (irz * (D(W, 2, "dx_txz", 0, -1, tab) + D(W, 1, "dz_tzz", 1, 1, tab)))[inner]
            t1, t2 = D(W, 3, "dx_vx", 0, -1, tab), D(W, 4, "dz_vz", 1, -1, tab)
            e2 = W[5 + L]
            for m in range(L):
                o[5 + m] = ((1.0 - 1.0 / eta1[m]) / L * (t1 + t2) - W[5 + m]) / ts1[m]
            o[5 + L] = 0.5 / ts2 * ((1.0 - 1.0 / eta2) * (t1 + t2) - 2.0 * e2)
            # the scheme's relaxation sum reads the state at offset 6 N + m
            q = sum(W.reshape(-1)[6 * N + m:7 * N + m] for m in range(L)).view(nx2, nz2)
            o[0] = c11 * t1 + c13 * t2 + K0 * q + 2.0 * mu * eta2 * e2
            o[1] = c13 * t1 + c33 * t2 + K0 * q - 2.0 * mu * eta2 * e2
            t = D(W, 3, "dz_vx", 1, 1, tab) + D(W, 4, "dx_vz", 0, 1, tab)
            o[6 + L] = ((1.0 - 1.0 / eta_ij) * t - W[6 + L]) / ts_ij
            o[2] = ci * t
    else:
        fields, nstate, inject = {TXX: 0, TZZ: 1, TXZ: 2, P: 3, VX: 4, VZ: 5, QX: 6, QZ: 7}, 9, (3, 0, 1)
        if s == "pve":
            Km, Ks, Kf, phi, mu, rs, rf, Tx, eta, kx, Q, f = model
            Tz, kz, eps, dl = Tx, kx, torch.zeros_like(Km), torch.zeros_like(Km)
        else:
            Km, Ks, Kf, phi, mu, rs, rf, Tx, Tz, eta, kx, kz, Q, f, eps, dl = model
        Km, Ks, Kf, mu, rs, rf = Km * 1e3, Ks * 1e3, Kf * 1e3, mu * 1e3, rs * 1e-6, rf * 1e-6
        eta = eta * 1.013249965828145e6
        c33 = Km + 4.0 / 3.0 * mu
        c11 = (1.0 + 2.0 * eps) * c33
        c13 = torch.sqrt(2.0 * dl * c33 * (c33 - mu) + (c33 - mu) ** 2) - mu
        c12 = c11 - 2.0 * mu
        M = Ks * Ks / (Ks * (1.0 + phi * (Ks / Kf - 1.0)) - (2.0 * c11 + c33 + 2.0 * c12 + 4.0 * c13) / 9.0)
        al1, al3 = 1.0 - (c11 + c12 + c13) / (3.0 * Ks), 1.0 - (2.0 * c13 + c33) / (3.0 * Ks)
        ts, ratio = relax(Q, f)
        vphi = M * (1.0 - ratio)                    # M varphi / (1 + varphi), varphi = tau_e / tau_s - 1
        rho = (1.0 - phi) * rs + phi * rf
        side = []
        for ax, T, kap in ((0, Tx, kx), (1, Tz, kz)):
            r, q, mm, nk = avg(rho, ax), avg(rf, ax), avg(T * rf / phi, ax), avg(eta / kap, ax)
            cq = torch.exp(nk * r / (q * q - r * mm) * dt)
            side.append((q / r, q * q / r - mm, 1.0 / r, cq, -(q / r) * (cq - 1.0)))
        cm = corner(mu, True)

        def rhs(W, o, tab):
            for v, ax, shear, normal in ((4, 0, ("dz_txz", 2, 1, -1), ("dx_txx", 0, 0, 1)),
                                         (5, 1, ("dx_txz", 2, 0, -1), ("dz_tzz", 1, 1, 1))):
                t = D(W, normal[1], normal[0], normal[2], normal[3], tab)
                t = t + D(W, shear[1], shear[0], shear[2], shear[3], tab)
                rr, mm, ir, _, _ = side[ax]
                q = (D(W, 3, ("dx_p", "dz_p")[ax], ax, 1, tab) + rr * t) / mm
                o[v + 2][inner] = q[inner]
                o[v][inner] = (ir * t - rr * q)[inner]
            t1, t2 = D(W, 4, "dx_vx", 0, -1, tab), D(W, 5, "dz_vz", 1, -1, tab)
            e = al1 * t1 + al3 * t2 + D(W, 6, "dx_qx", 0, -1, tab) + D(W, 7, "dz_qz", 1, -1, tab)
            o[8] = -(vphi * e + W[8]) / ts
            e = M * e + W[8]
            o[3] = -e
            o[0] = c11 * t1 + c13 * t2 + al1 * e
            o[1] = c13 * t1 + c33 * t2 + al3 * e
            o[2] = cm * (D(W, 4, "dz_vx", 1, 1, tab) + D(W, 5, "dx_vz", 0, 1, tab))

    W = torch.zeros((nstate, nx2, nz2), dtype=torch.float64, device=_dev())
    out = torch.zeros_like(W)
    rec = _Recorder(d, case["steps"], fields)
    si = int(d["src"][0])
    kept = 2 * n + 1 if s == "pve" else 2 * n       # rows of the memory variables carried into a step
    for it in range(case["steps"]):
        Ws = W.clone()
        if s.startswith("pve"):
            for v, q, ax in ((4, 6, 0), (5, 7, 1)):
                Ws[v] = W[v] + side[ax][4] * W[q]
                Ws[q] = side[ax][3] * W[q]
        for m0, m1, m2, limit in mem.values():
            lim = limit // (2 * n + 1) * kept
            m0[:lim] = m1[:lim]
        W, Wt = Ws.clone(), Ws
        for a, b, tab in ((0.5, 1 / 6, 0), (0.5, 1 / 3, 1), (1.0, 1 / 3, 1), (0.0, 1 / 6, 2)):
            rhs(Wt, out, tabs[tab])
            for m0, m1, m2, limit in mem.values():
                m2[:limit] = m1[:limit]
            W = W + b * dt * out
            Wt = Ws + a * dt * out
            if 2 * it + 1 < d["wav"].size:
                for q in inject:
                    W[q].reshape(-1)[si] += b * dt * d["wav"][2 * it + 1]
                    Wt[q].reshape(-1)[si] += a * dt * d["wav"][2 * it + 1]
        rec(it, W)
    if case.get("snapshot"):
        return {"traces": rec.out, "snapshot": W[fields[VY if s == "sh" else VZ]]}
    return {"traces": rec.out}
