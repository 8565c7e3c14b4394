"""The performance cases of the time-stepping path.

Each case is work that a program using this framework has it do over and over:
time steps of the solver (one grid, 16-bit storage, curvilinear topography,
discontinuous mesh with plasticity), the same steps through the C launchers as
a pmcl3d-style host program calls them, a misfit gradient, and the
Lagrange-interpolated receivers and sources of an input-file run.

Kinds of case and their parameters:
  solver    awp_amd.solver.Solver / Solver16: n x, y, z, steps per pass,
            storage "fp32" | "bf16" | "fp16", texture "arrays" (the default
            of Solver) | "auto", q (anelastic) and topo (curvilinear grid 0)
  launch    the C ABI of libawp_hip.so, caller-owned arrays: one step
  dm        two grids with plasticity (nz: fine levels, nzc: coarse levels;
            x, y: coarse cells, three times as many on the fine grid)
  adjoint   AdjointProblem.forward + backward over `steps` steps
  points    Lagrange receivers (3 components) and sources (6 components)

Media are layered (vs 1500 -> 4500 m/s) with a smooth 5 % perturbation and
Qs = 50 vs[km/s], the workloads' own; wavefields are smooth random fields of
ground-motion size, so every cell carries data, as in the middle of a run.
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.nn.functional as F

from awp_amd import _lib
from awp_amd.configs import PointSources, Receivers, ricker
from awp_amd.dm import checkmesh
from awp_amd.grid import ALIGN, NGSL, Dims
from awp_amd.media import Medium, cerjan, q_model

VEL = ("u1", "v1", "w1")
STRESS = ("xx", "yy", "zz", "xy", "xz", "yz")
MEM = ("r1", "r2", "r3", "r4", "r5", "r6")
WAVE = VEL + STRESS + MEM
DEV = "cuda"


def listed():
    return [
        # the elastic half-space example: the smallest grid anyone steps, ten
        # steps a pass; launches and host time count
        dict(name="halfspace-64", kind="solver", x=64, y=64, z=64, steps=10, storage="fp32",
             texture="arrays", q=False, topo=False),
        # an odd-sized anelastic grid through the solver's defaults
        dict(name="anelastic-ragged", kind="solver", x=243, y=187, z=101, steps=2,
             storage="fp32", texture="arrays", q=True, topo=False),
        # an ordinary anelastic run, texture table where the medium allows it
        dict(name="anelastic-256", kind="solver", x=256, y=256, z=128, steps=2, storage="fp32",
             texture="auto", q=True, topo=False),
        # a host program that keeps the per-cell texture arrays (dstrqc_H)
        dict(name="launch-arrays", kind="launch", x=320, y=320, z=192, storage="fp32",
             texture="arrays"),
        # the headline grid: the largest call
        dict(name="launch-512", kind="launch", x=512, y=512, z=256, storage="fp32",
             texture="rule"),
        # 16-bit storage at production size
        dict(name="launch-bf16", kind="launch", x=384, y=384, z=256, storage="bf16",
             texture="rule"),
        # binary16 storage with its scale check every eight steps
        dict(name="fp16-check", kind="solver", x=150, y=130, z=90, steps=8, storage="fp16",
             texture="arrays", q=True, topo=False),
        # curvilinear topography at an ordinary size
        dict(name="topography", kind="solver", x=256, y=256, z=192, steps=1, storage="fp32",
             texture="auto", q=True, topo=True),
        # a small curvilinear grid of odd sizes, per-cell texture arrays
        dict(name="topography-ragged", kind="solver", x=131, y=97, z=85, steps=2,
             storage="fp32", texture="arrays", q=True, topo=True),
        # discontinuous mesh + plasticity
        dict(name="dm-plastic", kind="dm", x=96, y=96, z=48, zc=64, steps=1),
        # gradient of a receiver misfit: forward, recompute and adjoint steps
        dict(name="adjoint", kind="adjoint", x=96, y=96, z=64, steps=24, every=8),
        # input-file receivers and sources of one step
        dict(name="points", kind="points", x=192, y=192, z=96, nrec=12000, nsrc=3000),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(("solver", "solver", "solver", "launch", "launch", "dm", "adjoint",
                       "points"))
    if kind == "launch":
        while True:
            x, y, z = _log(rng, 64, 512), _log(rng, 64, 512), _log(rng, 48, 320)
            if x * y * z <= 4.0e7:
                break
        return dict(kind=kind, x=x, y=y, z=z, storage=rng.choice(("fp32", "fp32", "bf16", "fp16")),
                    texture=rng.choice(("arrays", "rule")))
    if kind == "solver":
        topo = rng.random() < 0.4
        while True:
            x, y, z = _log(rng, 48, 300), _log(rng, 48, 300), _log(rng, 48, 200)
            if x * y * z <= 8.0e6:
                break
        storage = rng.choice(("fp32", "fp32", "bf16", "fp16"))
        return dict(kind=kind, x=x, y=y, z=z, steps=8 if storage == "fp16" else rng.choice((1, 2, 4)),
                    storage=storage, texture=rng.choice(("arrays", "auto")), q=rng.random() < 0.8,
                    topo=topo)
    if kind == "dm":
        return dict(kind=kind, x=_log(rng, 48, 100), y=_log(rng, 48, 100), z=_log(rng, 24, 72),
                    zc=_log(rng, 40, 90), steps=rng.choice((1, 2)))
    if kind == "adjoint":
        return dict(kind=kind, x=_log(rng, 56, 110), y=_log(rng, 56, 110), z=_log(rng, 48, 80),
                    steps=rng.choice((12, 16, 20, 24)), every=rng.choice((4, 6, 8)))
    return dict(kind=kind, x=_log(rng, 64, 256), y=_log(rng, 64, 256), z=_log(rng, 48, 128),
                nrec=_log(rng, 200, 20000), nsrc=_log(rng, 50, 4000))


# --------------------------------------------------------------------------
# Inputs

def _gen(seed, k=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 16 + k)
    return g


def _smooth(gen, n, cells):
    """A smooth random field of unit standard deviation, features of about
    `cells` cells."""
    low = [max(3, math.ceil(a / cells) + 1) for a in n]
    a = torch.randn((1, 1, *low), generator=gen, device=DEV)
    a = F.interpolate(a, size=tuple(n), mode="trilinear", align_corners=True)[0, 0]
    return a / a.std()


def _medium(d, DH, DT, seed, q=True, ND=20, lowest=True, z0=0.0, zmax=None):
    """Padded binary32 medium arrays on the device (k = nzt+31 the surface)."""
    nx, ny, nz = d.nxt, d.nyt, d.nzt
    zmax = zmax or nz * DH
    depth = z0 + (nz - 1 - torch.arange(nz, device=DEV) + 0.5) * DH
    layer = torch.clamp((depth / zmax * 6).floor(), max=5.0)
    vs = (1500.0 + 3000.0 * layer / 5.0)[None, None, :] * (1.0 + 0.05 * _smooth(_gen(seed, 1), (nx, ny, nz), 8).clamp(-3, 3))
    vp = 1.73 * vs
    rho = 310.0 * vp ** 0.25
    I, J, K = d.interior()

    def pad(v, shell):
        out = torch.zeros(d.shape, device=DEV)
        if shell:  # one ghost cell all round
            w = F.pad(v[None, None], (1, 1, 1, 1, 1, 1), mode="replicate")[0, 0]
            out[I.start - 1:I.stop + 1, J.start - 1:J.stop + 1, K.start - 1:K.stop + 1] = w
        else:      # the level above the surface only
            out[I, J, K] = v
            out[I, J, K.stop] = v[:, :, -1]
        return out

    m = dict(d1=pad(rho, True), mu=pad(1.0 / (rho * vs * vs), True),
             lam=pad(1.0 / (rho * (vp * vp - 2.0 * vs * vs)), True))
    qm = q_model(0.0, 0.005, 2.5)
    Qs = 0.05 * vs
    m["qs"] = pad(1.0 / Qs / qm.facex if q else torch.zeros_like(vs), False)
    m["qp"] = pad(0.5 / Qs / qm.facex if q else torch.zeros_like(vs), False)
    del vp, rho, vs, Qs
    # relaxation texture: the parity rule and its three per-mechanism values
    ni = torch.arange(nx, device=DEV)[:, None, None]
    col = ni * ny + torch.arange(ny, device=DEV)[None, :, None]
    nk = torch.arange(nz, device=DEV)[None, None, :]
    ww = (1 + 4 * ((ni + 1) & 1) + 2 * ((col + 1) & 1) + ((nz + col * nz + nk) & 1)).to(torch.int32)
    tau2 = np.exp(-DT / qm.tau)
    tab = np.stack([0.5 * (1.0 - tau2), tau2, 8.0 * qm.weights]).reshape(3, 8).astype(np.float32)
    m["ww"] = torch.zeros(d.shape, dtype=torch.int32, device=DEV)
    m["ww"][I, J, K] = ww
    for name, t in zip(("vx1", "vx2", "wwo"), tab):
        m[name] = torch.zeros(d.shape, device=DEV)
        m[name][I, J, K] = torch.from_numpy(t).to(DEV)[(ww - 1).long()]
    del ww
    xl = 1.0 / m["lam"][I, J, d.ktop].double()
    m["lam_mu"] = torch.zeros(d.shape[:2], device=DEV)
    m["lam_mu"][I, J] = (xl / (2.0 / m["mu"][I, J, d.ktop].double() + xl)).float()
    dx, dy, dz = cerjan(d, ND=min(ND, nx // 3, ny // 3, nz // 2), islowest=lowest)
    for name, v in (("dcrjx", dx), ("dcrjy", dy), ("dcrjz", dz), ("coeff", qm.coeff)):
        m[name] = torch.from_numpy(np.ascontiguousarray(v, dtype=np.float32)).to(DEV)
    return m, qm, tab


def _host_medium(d, DH, DT, m, qm):
    h = {k: v.cpu().numpy() for k, v in m.items()}
    return Medium(dims=d, DH=DH, DT=DT, qmodel=qm, **h)


AMP = dict(v=0.01, s=1.0e5, r=1.0e3)


def _wave(d, seed, scale=1.0):
    """The wavefield and memory variables in the middle of a run."""
    I, J, K = d.interior()
    g = _gen(seed, 2)
    out = {}
    for n in WAVE:
        a = AMP["v" if n in VEL else "s" if n in STRESS else "r"] * scale
        out[n] = torch.zeros(d.shape, device=DEV)
        out[n][I, J, K] = a * _smooth(g, (d.nxt, d.nyt, d.nzt), 5)
    return out


NT = 1000  # samples of a source and recording slots of a run


def _sources(d, seed, n, M0, DT, zlo=None, zhi=None):
    rng = np.random.default_rng(seed + 77)
    cells = set()
    while len(cells) < n:
        cells.add((int(rng.integers(d.nxt // 4, 3 * d.nxt // 4)),
                   int(rng.integers(d.nyt // 4, 3 * d.nyt // 4)),
                   int(rng.integers(zlo or d.nzt // 3, zhi or 2 * d.nzt // 3))))
    rates = M0 * rng.uniform(0.5, 1.5, (n, 1, 6)) * ricker(np.arange(NT) * DT, 1.0)[None, :, None]
    return PointSources(np.array(sorted(cells)), np.float32(rates).astype(np.float64))


def _receivers(d, seed, n=8):
    rng = np.random.default_rng(seed + 78)
    return Receivers(np.stack([rng.integers(1, d.nxt + 1, n), rng.integers(1, d.nyt + 1, n)], 1))


def _topography(d, DH, seed):
    rng = np.random.default_rng(seed + 79)
    e = np.zeros((d.nxt + 2 * NGSL, d.nyt + 2 * NGSL))
    X, Y = np.meshgrid(*[np.arange(a) for a in e.shape], indexing="ij")
    for _ in range(6):
        cx, cy = rng.uniform(0, e.shape[0]), rng.uniform(0, e.shape[1])
        w = rng.uniform(20, 80)
        e += rng.uniform(0.3, 1.0) * np.exp(-((X - cx) ** 2 + (Y - cy) ** 2) / w ** 2)
    return (e / e.max() * min(1500.0, 0.1 * d.nzt * DH)).astype(np.float32).astype(np.float64)


def _spacing(case):
    return (100.0, 0.005) if case["kind"] in ("adjoint",) or case.get("topo") else (50.0, 0.0025)


def _f32(x):
    return float(np.float32(x))


FMT = {"bf16": 1, "fp16": 2}
KIND16 = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _unit_scales(d, m, storage, sources, DH, DT):
    """The scales a 16-bit run starts with: 1 for bfloat16; for binary16 the
    power of two that puts the sources' bound at 2^12."""
    if storage == "bf16":
        return {n: 1.0 for n in WAVE}
    I, J, K = d.interior()
    sig = float(np.abs(sources.rates).sum(axis=1).max()) * DT / DH ** 3
    imp = float((m["d1"][I, J, K] / m["mu"][I, J, K]).sqrt().min())
    p2 = lambda b: 2.0 ** (math.floor(math.log2(b)) - 12)  # noqa: E731
    return {n: p2(sig / imp) if n in VEL else p2(sig) for n in WAVE}


def _wave16(d, seed, storage, scales):
    """Stored values: bfloat16 of the field, or binary16 of magnitude 2^9
    (largest), where the drift check wants them."""
    w = _wave(d, seed)
    out = {}
    for n, a in w.items():
        if storage == "fp16":
            a = a / a.abs().max() * 700.0
        out[n] = (a / (1.0 if storage == "fp16" else scales[n])).to(KIND16[storage])
    return out


def _lib_constants(lib, ds, DHs, DT):
    G = len(ds)
    lib.SetDeviceConstValue((C.c_float * G)(*DHs), C.c_float(DT), (C.c_int * G)(*[d.nxt for d in ds]),
                            (C.c_int * G)(*[d.nyt for d in ds]), (C.c_int * G)(*[d.nzt for d in ds]),
                            G, 0.0, 0.0, (C.c_float * 9)(), (C.c_float * 9)())
    _lib.check()


def _fill(level, wave):
    for n, t in wave.items():
        f = level.f[n]
        f.copy_(t if t.dtype == f.dtype else t.view(f.dtype))


def _plastic(d, m, DH, seed, z0):
    """sigma2 (lithostatic), cohesion 5 MPa with a smooth variation, friction
    angle 36.87 degrees, on the device."""
    ov = m["d1"].flip(2).double().cumsum(2).flip(2)
    s2 = -(ov * DH - 0.5 * DH * m["d1"]) * 9.81 - 9.81 * 2200.0 * z0
    out = torch.zeros(d.shape, device=DEV)
    I, J, K = d.interior()
    box = (slice(I.start - 1, I.stop + 1), slice(J.start - 1, J.stop + 1), slice(K.start - 1, K.stop + 1))
    out[box] = s2[box].float()
    coh = torch.full(d.shape, 5.0e6, device=DEV)
    coh[I, J, K] *= 1.0 + 0.1 * _smooth(_gen(seed, 5), (d.nxt, d.nyt, d.nzt), 12).clamp(-3, 3)
    return dict(sigma2=out, cohes=coh,
                phi=torch.full(d.shape, float(np.degrees(np.arctan(0.75))), device=DEV))


def _dm_inputs(case, seed):
    DT, DHs = 0.0025, (25.0, 75.0)
    ds = [Dims(3 * case["x"], 3 * case["y"], case["z"]), Dims(case["x"], case["y"], case["zc"])]
    z0 = (0.0, (ds[0].nzt - 9) * DHs[0])
    zmax = z0[1] + ds[1].nzt * DHs[1]
    meds, pls = [], []
    for p, d in enumerate(ds):
        m, qm, _ = _medium(d, DHs[p], DT, seed + p, ND=(24, 8)[p], lowest=p == 1, z0=z0[p], zmax=zmax)
        pls.append(_plastic(d, m, DHs[p], seed + p, z0[p]))
        meds.append(_host_medium(d, DHs[p], DT, m, qm))
    checkmesh(meds[0], meds[1])  # the coarse grid's top levels carry the fine medium
    waves = [_wave(d, seed + p, 40.0) for p, d in enumerate(ds)]  # strong motion: cells yield
    return DT, DHs, ds, meds, pls, waves, _sources(ds[1], seed, 20, 1.0e15, DT)


def _point_inputs(case, seed):
    d = Dims(case["x"], case["y"], case["z"])
    h = 50.0
    rng = np.random.default_rng(seed + 80)
    # one grid of each direction: index 0 is field index 2 (32 in z)
    ax = [np.float32(h) * np.arange(n, dtype=np.float32)
          for n in (d.nxt + 2 * NGSL, d.nyt + 2 * NGSL, d.nzt)]
    q = lambda n, box: [np.float32(rng.uniform(lo * a[-1], hi * a[-1], n))  # noqa: E731
                        for a, (lo, hi) in zip(ax, box)]
    rec = q(case["nrec"], ((0.1, 0.9), (0.1, 0.9), (0.2, 0.9)))
    # a fault plane: overlapping stencils
    src = q(case["nsrc"], ((0.3, 0.7), (0.49, 0.51), (0.3, 0.8)))
    return d, h, 0.0025, ax, rec, src


def prepare(case, seed):
    kind = case["kind"]
    if kind == "points":
        from awp_amd.interpolation import Interpolation, metric_grid
        d, h, DT, ax, rec, src = _point_inputs(case, seed)
        g = metric_grid(d)
        wave = _wave(d, seed)
        val = torch.randn((6, case["nsrc"]), generator=_gen(seed, 3), device=DEV) * 1.0e12
        return dict(case=case, f=wave, val=val, h=h, DT=DT, ip_rec=Interpolation(*ax, g, *rec),
                    ip_src=Interpolation(*ax, g, *src),
                    out=torch.zeros((3, case["nrec"]), device=DEV))
    if kind == "dm":
        from awp_amd.plasticity import PlasticMedium, PlasticParams
        from awp_amd.solver import Solver
        DT, DHs, ds, meds, pls, waves, src = _dm_inputs(case, seed)
        par = PlasticParams(fmajor=1.0, fminor=1.0, Tv=0.01)
        pl = [PlasticMedium(params=par, **{k: v.cpu().numpy() for k, v in p.items()}) for p in pls]
        s = Solver(meds, [None, src], _receivers(ds[0], seed), nt_record=NT, plastic=pl,
                   texture="auto")
        for L, w in zip(s.levels, waves):
            _fill(L, w)
        s.cur_step = 1
        return dict(case=case, s=s)
    d = Dims(case["x"], case["y"], case["z"])
    DH, DT = _spacing(case)
    if kind == "adjoint":
        from awp_amd.adjoint import AdjointProblem
        m, qm, _ = _medium(d, DH, DT, seed)
        src, rec = _adjoint_points(d, DT, seed)
        p = AdjointProblem(_host_medium(d, DH, DT, m, qm), src, rec, case["steps"],
                           np.zeros((case["steps"], len(rec.xy), 3), np.float32),
                           checkpoint_every=case["every"], resident_steps=case["every"])
        return dict(case=case, p=p)
    storage = case["storage"]
    src = _sources(d, seed, 4, 1.0e13, DT)
    m, qm, tab = _medium(d, DH, DT, seed, q=case.get("q", True))
    scales = _unit_scales(d, m, storage, src, DH, DT) if storage != "fp32" else None
    if kind == "launch":
        lib = _lib.load()
        _lib_constants(lib, [d], [DH], DT)
        f = _wave(d, seed) if storage == "fp32" else _wave16(d, seed, storage, scales)
        return dict(case=case, lib=lib, d=d, m=m, f=f, tex=(C.c_float * 24)(*tab.reshape(-1).tolist()),
                    psrc=torch.from_numpy(src.psrc(d).reshape(-1)).to(DEV), nsrc=src.npsrc,
                    cols=[torch.from_numpy(c.astype(np.float32)).to(DEV) for c in src.columns()],
                    sc=(C.c_float * 15)(*[scales[n] for n in WAVE]) if scales else None)
    from awp_amd.solver import Solver, Solver16
    med = _host_medium(d, DH, DT, m, qm)
    del m
    topo = None
    if case["topo"]:
        from awp_amd.topography import Topography
        topo = Topography(_topography(d, DH, seed))
    rec = _receivers(d, seed)
    if storage == "fp32":
        s = Solver(med, src, rec, nt_record=NT, topography=topo, texture=case["texture"])
        wave = _wave(d, seed)
    else:
        s = Solver16(med, src, rec, nt_record=NT, storage=storage, topography=topo,
                     texture=case["texture"])
        wave = _wave16(d, seed, storage, scales)
    if not case["q"]:
        for n in MEM:
            wave[n].zero_()
    _fill(s.levels[0], wave)
    s.cur_step = 1 if storage != "fp16" else 0
    return dict(case=case, s=s)


def _adjoint_points(d, DT, seed):
    """Explosive-plus-shear shallow sources under a grid of surface receivers."""
    src = _sources(d, seed, 12, 1.0e20, DT, 4, 8)
    gx = np.linspace(d.nxt // 4, 3 * d.nxt // 4, 8).round().astype(int)
    gy = np.linspace(d.nyt // 4, 3 * d.nyt // 4, 8).round().astype(int)
    return src, Receivers(np.array([[a, b] for a in gx for b in gy]))


# --------------------------------------------------------------------------
# One pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "points":
        ir, isrc = state["ip_rec"], state["ip_src"]
        f = state["f"]
        for c, n in enumerate(VEL):
            ir.interp(state["out"][c], f[n])
        for c, n in enumerate(STRESS):
            isrc.add_cartesian(f[n], state["val"][c], state["h"], state["DT"])
        return [state["out"]] + [f[n] for n in STRESS]
    if kind == "adjoint":
        p = state["p"]
        J = p.forward()
        return [J, *p.backward()]
    if kind == "launch":
        return _launch_step(state)
    s = state["s"]
    if s.cur_step + case["steps"] >= NT:  # the next shot
        s.cur_step = 1
    s.run(case["steps"])
    if kind == "dm":
        return [L.f[n] for L in s.levels for n in WAVE + ("yldfac", "neta")] + [s.rec["out"]]
    f = s.levels[0].f
    if case["storage"] == "fp32":
        return [f[n] for n in WAVE] + [s.rec["out"]]
    return [f[n].view(KIND16[case["storage"]]) for n in WAVE] + [s.rec["out"]]


def _launch_step(st):
    """velocity, stress + Q, sources, free surface: pmcl3d's one-grid order."""
    lib, d, m, f, case = st["lib"], st["d"], st["m"], st["f"], st["case"]
    P = lambda t: t.data_ptr()  # noqa: E731
    stream = torch.cuda.current_stream().cuda_stream
    (s_i, e_i), (s_j, e_j) = d.i_range, d.j_range
    sponge = [P(m[n]) for n in ("dcrjx", "dcrjy", "dcrjz")]
    wide = case["storage"] == "fp32"
    more = () if wide else (FMT[case["storage"]], st["sc"])
    vel = lib.dvelcx_H_opt if wide else lib.awp_dvelcx_s16
    vel(*(P(f[n]) for n in VEL + STRESS), *sponge, P(m["d1"]), d.nyt, d.nzt, stream, s_i, e_i, 0,
        1, *more)
    a = [P(f[n]) for n in STRESS + MEM + VEL] + [P(m[n]) for n in ("lam", "mu", "qp", "coeff", "qs")]
    tail = (d.nxt, 0, 0, 0, s_i, e_i, s_j, e_j, 0)
    if case["texture"] == "rule":
        fn = lib.awp_dstrqc_tex if wide else lib.awp_dstrqc_tex_s16
        fn(*a, *sponge, d.nyt, d.nzt, stream, P(m["lam_mu"]), C.addressof(st["tex"]), None, *tail,
           *more)
    else:
        fn = lib.dstrqc_H if wide else lib.awp_dstrqc_s16
        fn(*a, *sponge, d.nyt, d.nzt, stream, P(m["lam_mu"]),
           *(P(m[n]) for n in ("vx1", "vx2", "ww", "wwo")), *tail, *more)
    axx, ayy, azz, axz, ayz, axy = (P(c) for c in st["cols"])
    src = lib.addsrc_H if wide else lib.awp_addsrc_s16
    src(2, NT, 3, P(st["psrc"]), st["nsrc"], stream, axx, ayy, azz, axz, ayz, axy, P(f["xx"]),
        P(f["yy"]), P(f["zz"]), P(f["xy"]), P(f["yz"]), P(f["xz"]), 0, *more)
    top = lib.fstr_H if wide else lib.awp_fstr_s16
    top(P(f["zz"]), P(f["xz"]), P(f["yz"]), stream, s_i, e_i, s_j, e_j, *more)
    _lib.check()
    return [f[n] for n in WAVE]


# --------------------------------------------------------------------------
# What a pass cannot do without

def work(case):
    kind = case["kind"]
    n = case["x"] * case["y"] * case["z"]
    if kind == "points":
        # receivers: 64 stencil values, 12 weights, indices, the sample;
        # sources: each touched value once (64 a source at most), 12 weights
        b = case["nrec"] * (3 * 4 * (64 + 1) + 4 * 16) + case["nsrc"] * (6 * 4 * (2 * 24 + 1) + 4 * 16)
        return dict(bytes=b, flops=3 * case["nrec"] * 64 * 4 + 6 * case["nsrc"] * 64 * 5)
    if kind == "adjoint":
        # a forward, the recompute of all but the last segment, and the
        # adjoint steps (12 adjoint fields read and written, 8 gradient sums
        # read and written, 9 forward fields, 5 medium + 4 texture arrays)
        rec = max(0, case["steps"] - case["every"])
        return dict(bytes=n * ((case["steps"] + rec) * 156 + case["steps"] * 4 * (30 + 16 + 9 + 9)),
                    flops=n * ((case["steps"] + rec) * 300 + case["steps"] * 700))
    if kind == "dm":
        cells = 9 * n + case["x"] * case["y"] * case["zc"]
        # step as below with the texture rule, plus sigma2, cohesion, friction
        # angle, yield factor and plastic strain
        return dict(bytes=cells * case["steps"] * 4 * (15 + 5 + 15 + 3 + 3),
                    flops=cells * case["steps"] * 500)
    w = 4 if case["storage"] == "fp32" else 2
    tex = 16 if case["texture"] == "arrays" else 0
    return dict(bytes=n * case.get("steps", 1) * (30 * w + 20 + tex),
                flops=n * case.get("steps", 1) * (900 if case.get("topo") else 300))


def tolerance(case):
    """About four times the distance from exact().  An anelastic step moves
    with the branch of its Q weight at 1 / (2 q) = 200, which a cell whose
    averaged quality factor rounds to the other side takes differently: a few
    cells in ten million, 1.5e-4 of a memory variable's norm.  The curvilinear
    step differentiates metrics of order 1 kept in 32 bits."""
    kind = case["kind"]
    if kind in ("solver", "launch"):
        if case["storage"] == "bf16":
            return {"rel": 2.0e-2}  # r1..r6: differences of rounded velocities
        if case["storage"] == "fp16":
            return {"rel": 8.0e-3}
        if case.get("q", True) or case.get("topo"):
            return {"rel": 6.0e-4}
    return {"rel": 1.0e-5}


# --------------------------------------------------------------------------
# The same passes in 64 bits with plain torch

C1, C2 = 9.0 / 8.0, -1.0 / 24.0


def _s(A, b, i=0, j=0, k=0):
    return A[b[0][0] + i:b[0][1] + i, b[1][0] + j:b[1][1] + j, b[2][0] + k:b[2][1] + k]


def _put(f, name, b, v):
    """f[name] with v in box b, without touching the old tensor (autograd)."""
    if v.requires_grad or f[name].requires_grad:
        f[name] = f[name].clone()
    _s(f[name], b)[...] = v


class _Grid:
    """One grid in 64 bits: fields f, medium m, position p in a stack of G."""

    def __init__(self, d, DH, DT, m, f, p=0, G=1):
        self.d, self.DH, self.DT = d, _f32(DH), _f32(DT)
        self.m = {k: (v if torch.is_tensor(v) else torch.from_numpy(np.ascontiguousarray(v))).to(DEV)
                  for k, v in m.items()}
        self.m = {k: v.long() if k == "ww" else v.double() for k, v in self.m.items()}
        self.f = {k: v.double() for k, v in f.items()}
        self.p, self.G = p, G
        self.dth, self.dh1 = self.DT / self.DH, 1.0 / self.DH
        self.I, self.J = (10, d.nxt + 10), (10, d.nyt + 10)
        self.top = d.nzt + ALIGN - 1

    def sponge(self, b):
        m = self.m
        return (m["dcrjx"][b[0][0]:b[0][1], None, None] * m["dcrjy"][None, b[1][0]:b[1][1], None] *
                m["dcrjz"][None, None, b[2][0]:b[2][1]])

    def velocity(self, second=False):
        """The 4th-order update, or the 2nd-order one of level align+2."""
        k = (ALIGN + 2, ALIGN + 3) if second else (
            ALIGN + 3 if self.p < self.G - 1 else ALIGN, self.top - (1 if self.p else -1))
        b = (self.I, self.J, k)
        f, rho = self.f, self.m["d1"]

        def back(A, ax):  # derivative at -1/2 .. of index n: n, n-1; n+1, n-2
            e = lambda q: {"i": 0, "j": 0, "k": 0, ax: q}  # noqa: E731
            r = _s(A, b, **e(0)) - _s(A, b, **e(-1))
            return r if second else C1 * r + C2 * (_s(A, b, **e(1)) - _s(A, b, **e(-2)))

        def fwd(A, ax):
            e = lambda q: {"i": 0, "j": 0, "k": 0, ax: q}  # noqa: E731
            r = _s(A, b, **e(1)) - _s(A, b, **e(0))
            return r if second else C1 * r + C2 * (_s(A, b, **e(2)) - _s(A, b, **e(-1)))

        dc = self.sponge(b)
        r0, rj, rk, rjk = _s(rho, b), _s(rho, b, j=-1), _s(rho, b, k=-1), _s(rho, b, j=-1, k=-1)
        ri, rik, rij = _s(rho, b, 1), _s(rho, b, 1, k=-1), _s(rho, b, 1, j=-1)
        t = self.dth
        new = {}
        new["u1"] = (_s(f["u1"], b) + t / (0.25 * (r0 + rj + rk + rjk)) *
                     (back(f["xx"], "i") + back(f["xy"], "j") + back(f["xz"], "k"))) * dc
        new["v1"] = (_s(f["v1"], b) + t / (0.25 * (r0 + ri + rk + rik)) *
                     (fwd(f["xy"], "i") + fwd(f["yy"], "j") + back(f["yz"], "k"))) * dc
        new["w1"] = (_s(f["w1"], b) + t / (0.25 * (r0 + ri + rj + rij)) *
                     (fwd(f["xz"], "i") + back(f["yz"], "j") + fwd(f["zz"], "k"))) * dc
        for n, v in new.items():
            _put(f, n, b, v)

    def ghosts(self, I, J):
        """Velocities one level above the free surface."""
        f, m, t = self.f, self.m, self.top
        at = lambda A, i=0, j=0, k=t: A[I[0] + i:I[1] + i, J[0] + j:J[1] + j, k]  # noqa: E731
        u, v, w = f["u1"], f["v1"], f["w1"]
        gi = torch.arange(*I, device=DEV) - NGSL - 1
        gj = torch.arange(*J, device=DEV) - NGSL - 1
        ug = at(u) - (at(w) - at(w, -1))
        vg = at(v) - (at(w, 0, 1) - at(w))
        vs1 = (gi < self.d.nxt).double()[:, None] * (at(u, 1) - (at(w, 1) - at(w)))
        vs2 = (gj > 1).double()[None, :] * (at(v, 0, -1) - (at(w) - at(w, 0, -1)))
        wg = at(w, k=t - 1) - m["lam_mu"][I[0]:I[1], J[0]:J[1]] * (
            (vs1 - ug) + (at(u, 1) - at(u)) + (vg - vs2) + (at(v) - at(v, 0, -1)))
        b = (I, J, (t + 1, t + 2))
        for n, x in (("u1", ug), ("v1", vg), ("w1", wg)):
            _put(f, n, b, x[:, :, None])

    def stress(self, I=None, J=None, second=False, rates=None):
        """Stresses and memory variables on columns I x J (half-open).
        second: the 2nd-order update of level align+2.  rates: (box, the six
        strain rates) of the curvilinear update."""
        I, J = I or self.I, J or self.J
        if I[0] >= I[1] or J[0] >= J[1]:
            return
        f, m = self.f, self.m
        if rates is None and not second and self.p == 0:
            self.ghosts(I, J)
        if rates is not None:
            b, (N1, N2, N3, E4, E5, E6) = rates
        else:
            b = (I, J, (ALIGN + 2, ALIGN + 3) if second else
                 (ALIGN + 3, self.top - (1 if self.p else -1)))

            def dif(A, ax, fw):
                e = lambda q: {"i": 0, "j": 0, "k": 0, ax: q}  # noqa: E731
                lo = 0 if fw else -1
                r = _s(A, b, **e(lo + 1)) - _s(A, b, **e(lo))
                return r if second else C1 * r + C2 * (_s(A, b, **e(lo + 2)) - _s(A, b, **e(lo - 1)))

            u, v, w = f["u1"], f["v1"], f["w1"]
            N1, N2, N3 = dif(u, "i", 1), dif(v, "j", 0), dif(w, "k", 0)
            E4 = dif(u, "j", 1) + dif(v, "i", 0)
            E5 = dif(u, "k", 1) + dif(w, "i", 0)
            E6 = dif(v, "k", 1) + dif(w, "j", 1)
        DT, dth, dh1 = self.DT, self.dth, self.dh1
        lam, mu, qp, qs = m["lam"], m["mu"], m["qp"], m["qs"]
        eight = lambda A: sum(_s(A, b, i, -j, -k) for i in (0, 1) for j in (0, 1) for k in (0, 1))  # noqa: E731
        vx1, vx2, wwo, ww = (_s(m[n], b) for n in ("vx1", "vx2", "wwo", "ww"))
        ca, cb = m["coeff"][2 * ww - 2], m["coeff"][2 * ww - 1]
        high = 1.0 if second else 2.0  # the level's update has no factor 2 there

        def qw(q):
            return torch.where(1.0 / (2.0 * q) <= 200.0, ca * (2 * q) ** 2 + cb * 2 * q,
                               high * wwo * q) / wwo

        xm = 16.0 / eight(mu)
        xl = 8.0 / eight(lam) + xm
        mid = lambda A, **e: _s(A, b) + _s(A, b, **e)  # noqa: E731
        one = (dict(k=-1), dict(j=-1), dict(i=1))
        xmu = [2.0 / mid(mu, **e) for e in one]
        hs = [-x * qw(0.25 * mid(qs, **e)) * dh1 * vx1 for x, e in zip(xmu, one)]
        h = -xm * qw(0.0625 * eight(qs)) * dh1 * vx1
        qpa = -qw(0.0625 * eight(qp)) * xl * dh1 * vx1
        XM = xm * dth + DT * h
        a1 = qpa * (N1 + N2 + N3)
        tmp = xl * dth * (N1 + N2 + N3) + DT * a1
        vp = DT * (1 + vx2 * vx1)
        dc = self.sponge(b)
        for n, r, part, twice in (("xx", "r1", N2 + N3, 0), ("yy", "r2", N1 + N3, 1),
                                  ("zz", "r3", N1 + N2, 1)):
            fr, rt = _s(f[r], b), -h * part + a1
            t = _s(f[n], b) + tmp - XM * part + vp * fr
            if twice:
                t = t * dc
            new = (t + DT * (rt * (wwo - 1) + vx2 * fr * (1 - vx1))) * dc
            _put(f, r, b, vx2 * fr + wwo * rt)
            _put(f, n, b, new)
        for n, r, E, hh, x in (("xy", "r4", E4, hs[0], xmu[0]), ("xz", "r5", E5, hs[1], xmu[1]),
                               ("yz", "r6", E6, hs[2], xmu[2])):
            fr, rt = _s(f[r], b), hh * E
            t = _s(f[n], b) + (x * dth + DT * hh) * E + vp * fr
            new = (t + DT * (rt * (wwo - 1) + vx2 * fr * (1 - vx1))) * dc
            _put(f, r, b, vx2 * fr + wwo * rt)
            _put(f, n, b, new)

    def source(self, src, sample):
        v = self.DT / self.DH ** 3
        for name, c in (("xx", 0), ("yy", 1), ("zz", 2), ("xz", 3), ("yz", 4), ("xy", 5)):
            a = self.f[name].clone() if self.f[name].requires_grad else self.f[name]
            for (x, y, z), r in zip(src.psrc(self.d), src.rates):
                a[x + 1 + NGSL, y + 1 + NGSL, z + ALIGN - 1] -= v * float(r[sample - 1, c])
            self.f[name] = a

    def image(self):
        """Antisymmetric stresses above the free surface."""
        f, t = self.f, self.top
        at = lambda n, k: f[n][self.I[0]:self.I[1], self.J[0]:self.J[1], k:k + 1]  # noqa: E731
        for n, k, val in (("zz", t + 1, -at("zz", t)), ("zz", t + 2, -at("zz", t - 1)),
                          ("xz", t + 1, -at("xz", t - 1)), ("xz", t + 2, -at("xz", t - 2)),
                          ("yz", t + 1, -at("yz", t - 1)), ("yz", t + 2, -at("yz", t - 2)),
                          ("xz", t, 0.0 * at("xz", t)), ("yz", t, 0.0 * at("yz", t))):
            _put(f, n, (self.I, self.J, (k, k + 1)), val)

    def sample(self, rec):
        idx = torch.from_numpy(rec.array_index(self.d)).to(DEV).long()
        i, j, k = idx.T
        return torch.stack([self.f["u1"][i, j, k], self.f["v1"][i, j, k], self.f["w1"][i, j, k - 1]], 1)

    # plasticity (principal axes along the grid: the rotation of the default
    # strikes and dips, evaluated here)
    def rotated(self, b, pf, i=0, j=0, k=0):
        """Initial stress xx, yy, zz, xy, xz, yz rotated from the principal
        frame, fluid pressure pf."""
        s = _s(self.m["sigma2"], b, i, j, k) + pf
        R = self.R
        ent = lambda p, q: sum(R[c][p] * R[c][q] for c in range(3)) * s  # noqa: E731
        return [ent(0, 0) - pf, ent(1, 1) - pf, ent(2, 2) - pf, ent(0, 1), ent(0, 2), ent(1, 2)]

    def pfluid(self, b, dk=0):
        dep = (self.top - (torch.arange(b[2][0], b[2][1], device=DEV) + dk)).double() * self.DH
        return torch.where(dep > 0, (dep + 0.5 * self.DH) * 9.81e3,
                           torch.full_like(dep, self.DH / 2 * 9.81e3))

    def yield_factor(self, I, J, Tv):
        """Inclusive column ranges I, J."""
        b = ((I[0], I[1] + 1), (J[0], J[1] + 1), (ALIGN, self.top + 1))
        f, m = self.f, self.m
        pf = self.pfluid(b)
        a, n = self.rotated(b, pf), self.rotated(b, pf, 1)
        ii = [0.5 * (p + q) for p, q in zip(a, n)]
        four = lambda A, e, g, h: 0.25 * (_s(A, b) + _s(A, b, *e) + _s(A, b, *g) + _s(A, b, *h))  # noqa: E731
        Sxx, Syy, Szz = (_s(f[c], b) + q for c, q in zip(("xx", "yy", "zz"), ii))
        Sxz = four(f["xz"], (1, 0, 0), (0, 0, -1), (1, 0, -1)) + ii[4]
        Syz = four(f["yz"], (0, -1, 0), (0, 0, -1), (0, -1, -1)) + ii[5]
        Sxy = four(f["xy"], (1, 0, 0), (0, -1, 0), (1, -1, 0)) + ii[3]
        phi = _s(m["phi"], b) * 0.017453292519943295
        sm = (Sxx + Syy + Szz) / 3.0
        D = [Sxx - sm, Syy - sm, Szz - sm]
        J2 = torch.sqrt(0.5 * sum(x * x for x in D) + Sxz ** 2 + Sxy ** 2 + Syz ** 2)
        lim = torch.clamp(_s(m["cohes"], b) * torch.cos(phi) - (sm + pf) * torch.sin(phi), min=0.0)
        hit = J2 > lim
        r = lim / torch.where(hit, J2, torch.ones_like(J2))
        y = torch.where(hit, r + (1.0 - r) * math.exp(-self.DT / Tv), torch.ones_like(r))
        xm = 2.0 / (_s(m["mu"], b) + _s(m["mu"], b, 1))
        d = [x * (y - 1.0) / xm for x in (*D, Sxy, Sxz, Syz)]
        e = torch.sqrt(0.5 * (d[0] ** 2 + d[1] ** 2 + d[2] ** 2) + 2.0 * (d[3] ** 2 + d[4] ** 2 + d[5] ** 2))
        _put(f, "yldfac", b, y)
        _put(f, "neta", b, _s(f["neta"], b) + torch.where(y < 1.0, e, torch.zeros_like(e)))

    def yield_apply(self):
        b = (self.I, self.J, (ALIGN, self.top + 1))
        f = self.f
        Y = f["yldfac"]
        pf, pf1 = self.pfluid(b), self.pfluid(b, -1)
        y0 = _s(Y, b)
        yxz = 0.25 * (_s(Y, b, -1) + y0 + _s(Y, b, -1, 0, 1) + _s(Y, b, 0, 0, 1))
        yyz = 0.25 * (y0 + _s(Y, b, 0, 1) + _s(Y, b, 0, 1, 1) + _s(Y, b, 0, 0, 1))
        yxy = 0.25 * (y0 + _s(Y, b, 0, 1) + _s(Y, b, -1) + _s(Y, b, -1, 1))
        r0 = self.rotated(b, pf)
        rb = self.rotated(b, pf1, 1)
        ii = [0.5 * (r0[c] + rb[c]) for c in range(3)]
        S = [_s(f[n], b) + q for n, q in zip(("xx", "yy", "zz"), ii)]
        sm = sum(S) / 3.0
        for n, x, q in zip(("xx", "yy", "zz"), S, ii):
            _put(f, n, b, torch.where(y0 < 1, (x - sm) * y0 + sm - q, _s(f[n], b)))
        q = 0.5 * (r0[4] + self.rotated(b, pf1, 0, 0, 1)[4])
        _put(f, "xz", b, torch.where(yxz < 1, (_s(f["xz"], b) + q) * yxz - q, _s(f["xz"], b)))
        q = 0.125 * sum(self.rotated(b, pf1 if e[2] else pf, *e)[5]
                        for e in ((i, j, k) for i in (0, 1) for j in (0, 1) for k in (0, 1)))
        _put(f, "yz", b, torch.where(yyz < 1, (_s(f["yz"], b) + q) * yyz - q, _s(f["yz"], b)))
        q = 0.5 * (r0[3] + self.rotated(b, pf, 0, 1)[3])
        _put(f, "xy", b, torch.where(yxy < 1, (_s(f["xy"], b) + q) * yxy - q, _s(f["xy"], b)))


# offsets of each field's sample in the 3:1 coupling: u1 v1 w1 xx yy zz xy xz yz
COUPLED = VEL + STRESS
INTP_OX = (0, 1, 1, 1, 1, 1, 0, 0, 1)
INTP_OY = (0, 1, 0, 0, 0, 0, 1, 0, 1)
SWAP_O = dict(u1=(2, 2), v1=(3, 3), w1=(3, 2), xx=(3, 2), yy=(3, 2), zz=(3, 2), xy=(2, 3),
              xz=(2, 2), yz=(3, 3))


def _interpolate(lo, hi):
    """Coarse level nzt+align-3 onto fine level align+1 (bilinear)."""
    d = lo.d
    ti = torch.arange(3 * (d.nxt + 3) + 4, device=DEV)
    tj = torch.arange(3 * (d.nyt + 3) + 4, device=DEV)
    ir, jr = torch.clamp(ti // 3, max=d.nxt + 3), torch.clamp(tj // 3, max=d.nyt + 3)
    a, b = (1.0 - (ti - 3 * ir) / 3.0).double()[:, None], (1.0 - (tj - 3 * jr) / 3.0).double()[None, :]
    for n, ox, oy in zip(COUPLED, INTP_OX, INTP_OY):
        A = lo.f[n][:, :, d.nzt + ALIGN - 3]
        at = lambda i, j: A[(NGSL + ir + i)[:, None], (NGSL + jr + j)[None, :]]  # noqa: E731,B023
        v = (at(0, 0) * a * b + at(1, 0) * (1 - a) * b + at(0, 1) * a * (1 - b) +
             at(1, 1) * (1 - a) * (1 - b))
        i0, j0 = (NGSL - 10) * 3 + 10 + ox, (NGSL - 10) * 3 + 10 + oy
        hi.f[n][i0:i0 + v.shape[0], j0:j0 + v.shape[1], ALIGN + 1] = v


def _swap(hi, lo):
    """Triangular 5x5x5 averages of the fine grid onto the coarse top levels."""
    d = lo.d
    i = torch.arange(NGSL, d.nxt + NGSL + 5, device=DEV)
    j = torch.arange(NGSL, d.nyt + NGSL + 5, device=DEV)
    w = [(3 - abs(q)) / 9.0 for q in range(-2, 3)]
    for n, (oi, oj) in SWAP_O.items():
        for kc, kh in ((-2, ALIGN + 4),) if n in ("w1", "xz", "yz") else ((-2, ALIGN + 3), (-1, ALIGN + 6)):
            A = sum(w[q + 2] * hi.f[n][:, :, kh + q] for q in range(-2, 3))
            A = sum(w[q + 2] * A[3 * (i - 10) + oi + NGSL + q] for q in range(-2, 3))
            A = sum(w[q + 2] * A[:, 3 * (j - 10) + oj + NGSL + q] for q in range(-2, 3))
            lo.f[n][NGSL:NGSL + len(i), NGSL:NGSL + len(j), d.nzt + ALIGN + kc] = A


def _regions(d):
    """The strips of the plastic step on one rank (inclusive)."""
    xl, xr, yl, yr = 10, d.nxt + 9, 10, d.nyt + 9
    y2, e2 = int(yl + (yr - yl) * 0.25), int(yl + (yr - yl) * 0.75)
    y2, e2 = y2 + y2 % 2, e2 - (1 - e2 % 2)
    return dict(x=(xl, xr), y=(yl, yr), left=(xl, 11), mid=(12, d.nxt + 7), right=(d.nxt + 8, xr),
                y2=max(y2, yl + 10), e2=min(e2, yr - 10))


def _dm_step(g, src, sample, Tv):
    half = lambda a, b: (a, b + 1)  # noqa: E731
    R = [_regions(x.d) for x in g]
    for x in g:
        x.velocity()
    g[0].velocity(second=True)
    _interpolate(g[1], g[0])
    _swap(g[0], g[1])
    for x, r in zip(g, R):
        x.stress(half(*r["mid"]), half(r["y"][0], r["y2"] - 1))
        x.stress(half(*r["mid"]), half(r["e2"] + 1, r["y"][1]))
    for x, r in zip(g, R):
        x.stress(half(*r["left"]), half(*r["y"]))
        x.stress(half(*r["right"]), half(*r["y"]))
    g[0].stress(second=True)
    g[1].source(src, sample)
    _interpolate(g[1], g[0])
    _swap(g[0], g[1])
    for x, r in zip(g, R):
        (a, b), (c, e) = r["x"], r["y"]
        x.yield_factor((a, b), (c, c + 8), Tv)
        x.yield_factor((a, b), (e - 8, e), Tv)
    for x, r in zip(g, R):
        x.stress(half(*r["mid"]), half(r["y2"], r["e2"]))
    for x, r in zip(g, R):
        (a, b), (c, e) = r["x"], r["y"]
        x.yield_factor((a, a + 8), (c, e), Tv)
        x.yield_factor((b - 8, b), (c, e), Tv)
    for x, r in zip(g, R):
        (a, b), (c, e) = r["x"], r["y"]
        x.yield_factor((a + 8, b - 8), (c + 8, e - 8), Tv)
    for x in g:
        x.yield_apply()
    g[0].image()


# Curvilinear operators in z: interior 7- and 4-point rows, and the one-sided
# rows of the top six levels (row r: level nz-1-r, column c: level nz-1-c).
P4 = (-0.0625, 0.5625, 0.5625, -0.0625)
D4 = (1.0 / 24.0, -1.125, 1.125, -1.0 / 24.0)
Z7 = (-0.0026041666666667, 0.09375, -0.6796875, 0.0, 0.6796875, -0.09375, 0.0026041666666667)
TOP = dict(
    v_dhpz=((-1.5373923010673118, -1.1059180740634813, -0.2134752473866528, -0.0352027995732726, -0.0075022330101095, -0.0027918394266035),
            (0.8139439685257414, 0.1273679143938725, -1.1932750007455710, 0.1475120181828087, 0.1125814499297686, -0.0081303502866204),
            (0.1639182541610305, 0.3113839909089030, -0.0536007135209480, -0.3910958927076030, -0.0401741813821989, 0.0095685425408165),
            (0.0171478318814576, -0.0916600077207278, 0.7187220404622645, -0.1434031863528334, -0.5827389738506837, 0.0847863081664324, -0.0028540125859095),
            (-0.0579176640853654, 0.0022069616616207, 0.0108792602269819, 0.6803612607837533, -0.0530169938441240, -0.6736586580761996, 0.09375, -0.0026041666666667),
            (0.0020323834153791, 0.0002106933140862, -0.0013351454085978, -0.0938400881871787, 0.6816971139746001, -0.0002232904416222, -0.6796875, 0.09375, -0.0026041666666667)),
    v_dhz=((0.0, -1.4511412472637157, -1.8534237417911470, 0.3534237417911469, 0.0488587527362844),
           (0.0, 0.8577143189081458, -0.5731429567244373, -0.4268570432755628, 0.1422856810918542),
           (0.0, 0.1674548505882877, 0.4976354482351368, -0.4976354482351368, -0.1674548505882877),
           (0.0, -0.1027061113405124, 0.2624541326469860, 0.8288742701021167, -1.0342864927831414, 0.0456642013745513),
           (0.0, 0.0, 0.0, -0.0416666666666667, 1.125, -1.125, 0.0416666666666667),
           (0.0, 0.0, 0.0, 0.0, -0.0416666666666667, 1.125, -1.125, 0.0416666666666667)),
    v_dphz=((0.0,),
            (0.0, -1.5886075042755421, -2.4835574634505861, 0.0421173406787286, 0.4968761536590695, -0.0228264197210198),
            (0.0, 0.4428256655817484, -0.0574614517751294, -0.2022259589759502, -0.1944663890497050, 0.0113281342190362),
            (0.0, -0.3360140866060758, 1.2113298407847195, -0.3111668377093505, -0.6714462506479002, 0.1111440843153523, -0.0038467501367455),
            (0.0, 0.0338560531369653, -0.0409943223643902, 0.5284757132923059, 0.0115571196122084, -0.6162252315536446, 0.0857115441015996, -0.0023808762250444),
            (0.0, -0.0040378273193044, 0.0064139372778371, -0.0890062133451850, 0.6749219241340761, 0.0002498459192428, -0.6796875, 0.09375, -0.0026041666666667)),
    v_dz=((0.0,),
          (-1.7779989465546753, -1.3337480247900155, -0.7775013168066564, 0.3332503950419969),
          (0.4410217341392059, 0.1730842484889890, -0.4487228323259926, -0.1653831503022022),
          (-0.1798793213882701, 0.2757257254150788, 0.9597948548284453, -1.1171892610431817, 0.0615480021879277),
          (-0.0153911381507088, -0.0568851455503591, 0.1998976464597171, 0.8628231468598346, -1.0285385292191949, 0.0380940196007109),
          (0.0, 0.0, 0.0, -0.0416666666666667, 1.125, -1.125, 0.0416666666666667)),
    s_phdz=((1.5373923010673116, -1.0330083346742178, -0.6211677623382129, -0.0454110758451345, 0.1680934225988761, -0.0058985508086226),
            (0.8713921425924012, -0.1273679143938725, -0.9297550647681331, 0.1912595577524762, -0.0050469052908678, -0.0004818158920039),
            (0.0563333965151294, 0.3996393739211770, 0.0536007135209481, -0.5022638816465500, -0.0083321572725344, 0.0010225549618299),
            (0.0132930497153990, -0.0706942590708847, 0.5596445380498726, 0.1434031863528334, -0.7456356868769503, 0.1028431844156395, -0.0028540125859095),
            (0.0025849423769932, -0.0492307522105194, 0.0524552477068130, 0.5317248489238559, 0.0530169938441240, -0.6816971139746001, 0.09375, -0.0026041666666667),
            (0.0009619461344193, 0.0035553215968974, -0.0124936029037323, -0.0773639466787397, 0.6736586580761996, 0.0002232904416222, -0.6796875, 0.09375, -0.0026041666666667)),
    s_dz=((0.0,), (1.7779989465546748, -1.3337480247900155, -0.7775013168066564, 0.3332503950419969)),
    s_dhz=((0.0, 1.4511412472637157, -1.8534237417911470, 0.3534237417911469, 0.0488587527362844),),
    s_pdhz=((0.0,),
            (0.0, 1.5886075042755419, -2.2801810182668114, 0.8088980291471826, -0.1316830205960989, 0.0143585054401857),
            (0.0, 0.4823226655921295, 0.0574614517751295, -0.5663203488781653, 0.0309656800624243, -0.0044294485515179),
            (0.0, -0.0174954311279016, 0.4325508330649349, 0.3111668377093504, -0.8538512002386446, 0.1314757107290064, -0.0038467501367455),
            (0.0, -0.1277481742492071, 0.2574468839590017, 0.4155794781917712, -0.0115571196122084, -0.6170517361659126, 0.0857115441015996, -0.0023808762250444),
            (0.0, 0.0064191319587820, -0.0164033832904366, -0.0752421418813823, 0.6740179057989464, -0.0002498459192428, -0.6796875, 0.09375, -0.0026041666666667)))
# the stress tables share the velocity tables' other rows
TOP["s_dz"] += TOP["v_dz"][2:]
TOP["s_dhz"] += TOP["v_dhz"][1:]


def _zop(name, nz):
    """The operator as a matrix over the levels; rows below level 3 unused."""
    row, first = ((Z7, -3) if name in ("v_dhpz", "v_dphz", "s_phdz", "s_pdhz") else
                  (D4, -2) if name in ("v_dhz", "s_dhz") else (D4, -1))
    M = np.zeros((nz, nz))
    for k in range(3, nz - 6):
        M[k, k + first:k + first + len(row)] = row
    for r, t in enumerate(TOP[name]):
        for c, x in enumerate(t):
            M[nz - 1 - r, nz - 1 - c] = x
    return torch.from_numpy(M.T.copy()).to(DEV)


class _Topo:
    def __init__(self, g, elev):
        self.g = g
        d, h = g.d, g.DH
        n = d.nzt
        self.Z = {k: _zop(k, n) for k in TOP}
        f = 1.0 + torch.from_numpy(elev).to(DEV) / (h * (n - 2))
        f = F.pad(f[None, None], (4, 4, 4, 4), mode="replicate")[0, 0]  # i = -12 ..

        def op(A, w, ax, first):
            return sum(x * torch.roll(A, -(first + q), ax) for q, x in enumerate(w))

        f_1, f_2 = op(f, P4, 1, -2), op(f, P4, 0, -1)
        f_c = op(f_2, P4, 1, -2)
        M = dict(f=f, f_1=f_1, f_2=f_2, f_c=f_c, f1_1=op(f_c, D4, 0, -2) / h,
                 f1_2=op(f, D4, 0, -1) / h, f1_c=op(f_1, D4, 0, -1) / h, f2_1=op(f, D4, 1, -2) / h,
                 f2_2=op(f_c, D4, 1, -1) / h, f2_c=op(f_2, D4, 1, -2) / h)
        self.M = {k: v[2:, 2:] for k, v in M.items()}  # array index = i + 10
        lev = torch.arange(n, device=DEV).double()
        self.gn = h * lev
        self.gn[-1] = 0.0
        self.gc = lev - 0.5
        self.gc[0], self.gc[-1] = 0.0, n - 2.0
        self.gc *= h

    def _ops(self, I, J):
        kk = slice(ALIGN, ALIGN + self.g.d.nzt)

        def S(A, i=0, j=0):
            return A[I[0] + i:I[1] + i, J[0] + j:J[1] + j, kk]

        def m(n, i=0, j=0):
            return self.M[n][I[0] + i:I[1] + i, J[0] + j:J[1] + j, None]

        def x(w, first, A, met=None, z=None):
            return sum(c * (m(met, first + q) if met else 1.0) * (S(A, first + q) if z is None else S(A, first + q) @ z)
                       for q, c in enumerate(w))

        def y(w, first, A, met=None, z=None):
            return sum(c * (m(met, 0, first + q) if met else 1.0) * (S(A, 0, first + q) if z is None else S(A, 0, first + q) @ z)
                       for q, c in enumerate(w))

        return S, m, x, y

    def velocity(self):
        g, Z = self.g, self.Z
        f, rho = g.f, g.m["d1"]
        I, J = g.I, g.J
        S, m, x, y = self._ops(I, J)
        dc = g.sponge((I, J, (ALIGN, ALIGN + g.d.nzt)))
        r = lambda i=0, j=0, k=0: _s(rho, (I, J, (ALIGN, ALIGN + g.d.nzt)), i, j, k)  # noqa: E731
        r1 = 0.25 * (r() + r(0, -1) + r(0, 0, -1) + r(0, -1, -1))
        r2 = 0.25 * (r() + r(-1) + r(0, 0, -1) + r(-1, 0, -1))
        r3 = 0.25 * (r() + r(-1) + r(0, -1) + r(-1, -1))
        gc, gn = self.gc, self.gn
        a = {}
        a["u1"] = (g.dth / (m("f_1") * r1), x(D4, -2, f["xx"], "f_c") + y(D4, -2, f["xy"], "f") +
                   S(f["xz"]) @ Z["v_dhz"] - m("f1_1") * ((gc * x(P4, -2, f["xx"])) @ Z["v_dhpz"]) -
                   m("f2_1") * ((gc * y(P4, -2, f["xy"])) @ Z["v_dhpz"]))
        a["v1"] = (g.dth / (m("f_2") * r2), S(f["yz"]) @ Z["v_dhz"] + x(D4, -1, f["xy"], "f") +
                   y(D4, -1, f["yy"], "f_c") - m("f1_2") * ((gc * x(P4, -1, f["xy"])) @ Z["v_dhpz"]) -
                   m("f2_2") * ((gc * y(P4, -1, f["yy"])) @ Z["v_dhpz"]))
        a["w1"] = (g.dth / (m("f_c") * r3), y(D4, -2, f["yz"], "f_2") + x(D4, -1, f["xz"], "f_1") +
                   S(f["zz"]) @ Z["v_dz"] - m("f1_c") * ((gn * x(P4, -1, f["xz"])) @ Z["v_dphz"]) -
                   m("f2_c") * ((gn * y(P4, -2, f["yz"])) @ Z["v_dphz"]))
        b = (I, J, (ALIGN + 3, ALIGN + g.d.nzt))
        for n, (c, s) in a.items():
            _put(f, n, b, ((S(f[n]) + c * s) * dc)[:, :, 3:])

    def stress(self):
        g, Z = self.g, self.Z
        f = g.f
        u, v, w = f["u1"], f["v1"], f["w1"]
        I, J = (g.I[0] + 4, g.I[1] - 4), (g.J[0] + 4, g.J[1] - 4)
        S, m, x, y = self._ops(I, J)
        Zh, Zn = Z["s_phdz"], Z["s_pdhz"]
        gc, gn = self.gc, self.gn
        N1 = x(D4, -1, u) - gc / m("f_c") * x(P4, -1, u, "f1_1", Zh)
        N2 = y(D4, -2, v) - gc / m("f_c") * y(P4, -2, v, "f2_2", Zh)
        N3 = (S(w) @ Z["s_dhz"]) / m("f_c")
        E4 = (y(D4, -1, u) + x(D4, -2, v) -
              gc / m("f") * (y(P4, -1, u, "f2_1", Zh) + x(P4, -2, v, "f1_2", Zh)))
        E5 = ((S(u) @ Z["s_dz"]) / m("f_1") + x(D4, -2, w) - gn / m("f_1") * x(P4, -2, w, "f1_c", Zn))
        E6 = ((S(v) @ Z["s_dz"]) / m("f_2") + y(D4, -1, w) - gn / m("f_2") * y(P4, -1, w, "f2_c", Zn))
        g.stress(I, J, rates=((I, J, (ALIGN + 3, ALIGN + g.d.nzt)),
                              [t[:, :, 3:] for t in (N1, N2, N3, E4, E5, E6)]))


def _lagrange(x, q):
    """Degree-3 weights at q (n) and first node, on the axis x, in 64 bits."""
    x = torch.from_numpy(x).to(DEV).double()
    q = torch.from_numpy(q).to(DEV).double()
    h = x[1] - x[0]
    near = torch.round(q / h).long()
    first = torch.clamp(near - torch.where(x[near] > q, 2, 1), 0, len(x) - 4)
    n = x[first[:, None] + torch.arange(4, device=DEV)]
    w = torch.ones_like(n)
    for a in range(4):
        for b in range(4):
            if a != b:
                w[:, a] = w[:, a] * (q - n[:, b]) / (n[:, a] - n[:, b])
    return w, first


def exact(case, seed):
    kind = case["kind"]
    if kind == "points":
        d, h, DT, ax, rec, src = _point_inputs(case, seed)
        f = {n: a.double() for n, a in _wave(d, seed).items()}
        val = (torch.randn((6, case["nsrc"]), generator=_gen(seed, 3), device=DEV) * 1.0e12).double()
        a4 = torch.arange(4, device=DEV)

        def stencil(q):
            (wx, ix), (wy, iy), (wz, iz) = (_lagrange(a, p) for a, p in zip(ax, q))
            W = wx[:, :, None, None] * wy[:, None, :, None] * wz[:, None, None, :]
            pos = (((ix[:, None] + a4 + 2) * d.shape[1])[:, :, None, None] +
                   (iy[:, None] + a4 + 2)[:, None, :, None]) * d.shape[2] + (iz[:, None] + a4 + ALIGN)[:, None, None, :]
            return W, pos

        W, pos = stencil(rec)
        out = torch.stack([(W * f[n].view(-1)[pos]).sum((1, 2, 3)) for n in VEL])
        W, pos = stencil(src)
        for c, n in enumerate(STRESS):
            f[n].view(-1).index_add_(0, pos.view(-1), (W * val[c][:, None, None, None]).view(-1),
                                     alpha=-_f32(DT) / h ** 3)
        return [out] + [f[n] for n in STRESS]
    if kind == "dm":
        DT, DHs, ds, meds, pls, waves, src = _dm_inputs(case, seed)
        g = []
        for p, d in enumerate(ds):
            m = dict(meds[p].arrays(), **pls[p])
            waves[p].update(yldfac=torch.ones(d.shape, device=DEV), neta=torch.zeros(d.shape, device=DEV))
            g.append(_Grid(d, DHs[p], DT, m, waves[p], p, 2))
            # principal axes: strikes 0, 0, 90 and dips 0, 90, 0 degrees
            g[p].R = ((1.0, 0.0, 0.0), (0.0, 0.0, 1.0), (0.0, 1.0, 0.0))
        rec = _receivers(ds[0], seed)
        tr = torch.zeros((NT, len(rec.xy), 3), dtype=torch.float64, device=DEV)
        for n in range(2, 2 + case["steps"]):
            _dm_step(g, src, n + 1, 0.01)
            tr[n - 1] = g[0].sample(rec)
        return [x.f[n] for x in g for n in WAVE + ("yldfac", "neta")] + [tr]
    d = Dims(case["x"], case["y"], case["z"])
    DH, DT = _spacing(case)
    if kind == "adjoint":
        return _exact_gradient(case, seed, d, DH, DT)
    storage = case["storage"]
    src = _sources(d, seed, 4, 1.0e13, DT)
    m, _, _ = _medium(d, DH, DT, seed, q=case.get("q", True))
    scales = {n: 1.0 for n in WAVE}
    if storage == "fp32":
        wave = _wave(d, seed)
    else:
        scales = _unit_scales(d, m, storage, src, DH, DT)
        wave = {n: a.double() * scales[n] for n, a in _wave16(d, seed, storage, scales).items()}
    if not case.get("q", True):
        for n in MEM:
            wave[n].zero_()
    g = _Grid(d, DH, DT, m, wave)
    del wave, m
    if kind == "launch":
        g.velocity()
        g.stress()
        g.source(src, 2)
        g.image()
        return [g.f[n] / scales[n] for n in WAVE]
    rec = _receivers(d, seed)
    tr = torch.zeros((NT, len(rec.xy), 3), dtype=torch.float64, device=DEV)
    T = _Topo(g, _topography(d, DH, seed)) if case["topo"] else None
    n0 = 0 if storage == "fp16" else 1
    if n0 == 0:
        g.source(src, 1)
    for n in range(n0 + 1, n0 + 1 + case["steps"]):
        (T or g).velocity()
        (T or g).stress()
        g.source(src, n + 1)
        g.image()
        tr[n - 1] = g.sample(rec)
    return [g.f[n] / scales[n] for n in WAVE] + [tr]


def _exact_gradient(case, seed, d, DH, DT):
    m, _, _ = _medium(d, DH, DT, seed)
    src, rec = _adjoint_points(d, DT, seed)
    g = _Grid(d, DH, DT, m, {n: torch.zeros(d.shape, device=DEV) for n in WAVE})
    p = {n: g.m[n].requires_grad_() for n in ("lam", "mu", "d1")}
    I, J, _ = d.interior()
    xl = 1.0 / p["lam"][I, J, d.ktop]
    g.m["lam_mu"] = torch.zeros(d.shape[:2], dtype=torch.float64, device=DEV)
    g.m["lam_mu"][I, J] = xl / (2.0 / p["mu"][I, J, d.ktop] + xl)
    g.source(src, 1)
    tr = []
    for n in range(1, case["steps"] + 1):
        g.velocity()
        g.stress()
        g.source(src, n + 1)
        g.image()
        tr.append(g.sample(rec))
    J_ = 0.5 * torch.stack(tr).square().sum()
    return [J_.item(), *torch.autograd.grad(J_, [p["lam"], p["mu"], p["d1"]])]
