"""Kernels and host paths at the sizes where their tiles, chunks and launches
change: plasticity tiles, curvilinear marches and columns, the adjoint's
surface band and moved fields, the 16-bit magnitude check, and the native step
loop.  Against the oracle or the step-by-step path bit for bit (the same
arithmetic: the tolerance is zero); the adjoint against the float64 reference
at the bound its other tests use."""
import ctypes as C

import numpy as np
import pytest

from awp_amd import configs
from awp_amd.grid import Dims
from tests._fields import first_mismatch, random_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awp_amd import _lib
    return torch, _lib


@pytest.mark.parametrize("nz", [36, 48, 65, 101, 128, 129, 150, 193, 256, 257])
def test_plasticity_tiles(gpu, oracle_lib, nz):
    from awp_amd.plasticity import PlasticParams
    from tests.test_gpu_parity import _plastic_state
    torch, _lib = gpu
    lib, o = _lib.load(), oracle_lib.load()
    d = Dims(10, 11, nz)
    st, med = _plastic_state(d, nz)
    pp = PlasticParams(fmajor=1.2, fminor=0.8, strike=(30.0, 0.0, 120.0))
    Rz, RzT = pp.rotation()
    F, I = C.c_float, C.c_int
    lib.SetDeviceConstValue((F * 1)(75.0), F(0.004), (I * 1)(d.nxt), (I * 1)(d.nyt),
                            (I * 1)(d.nzt), 1, pp.fmajor, pp.fminor, (F * 9)(*Rz.tolist()),
                            (F * 9)(*RzT.tolist()))
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in {**st, **med}.items()}
    host = {k: v.copy() for k, v in st.items()}
    p = lambda n: dev[n].data_ptr()  # noqa: E731
    q = lambda n: (host[n] if n in host else med[n]).ctypes.data  # noqa: E731
    s = torch.cuda.current_stream().cuda_stream
    S = ("xx", "yy", "zz", "xy", "xz", "yz")
    box = (10, d.nxt + 9, 10, d.nyt + 9)
    lib.drprecpc_calc_H_opt(*map(p, S + ("mu", "d1", "sigma2", "yldfac", "cohes", "phi", "neta")),
                            d.nzt, *box, s, 0)
    lib.drprecpc_app_H(*map(p, S + ("mu", "sigma2", "yldfac")), d.nzt, *box, s, 0)
    _lib.check()
    pl = np.ascontiguousarray(pp.packed())
    o.awp_oracle_drprecpc_calc_f32(
        *map(q, S + ("mu", "d1", "sigma2", "yldfac", "cohes", "phi", "neta")), d.nxt, d.nyt,
        d.nzt, 75.0, 0.004, *box, pl.ctypes.data, 0.0)
    o.awp_oracle_drprecpc_app_f32(*map(q, S + ("sigma2", "yldfac")), d.nxt, d.nyt, d.nzt, 75.0,
                                  *box, pl.ctypes.data)
    torch.cuda.synchronize()
    assert (host["yldfac"] < 1).sum() > 100
    for n in S + ("yldfac", "neta"):
        mm = first_mismatch(dev[n].cpu().numpy(), host[n])
        assert mm is None, f"nz={nz}: {n} differs: {mm}"


# columns around one, two, three, four and eight waves (the velocity takes one-wave
# segments above four); odd planes; few planes
@pytest.mark.parametrize("nx,ny,nz", [(20, 21, 18), (33, 18, 63), (18, 19, 64), (17, 34, 65),
                                      (21, 20, 127), (19, 18, 130), (18, 17, 193),
                                      (17, 18, 256), (18, 17, 257), (17, 18, 520)])
def test_curvilinear_columns(gpu, oracle_lib, nx, ny, nz):
    torch, _lib = gpu
    from awp_amd.solver import FIELDS, Solver
    from oracle.oracle import OracleSolver
    w = configs.topography_hills(nx=nx, ny=ny, nz=nz, nt=4, DH=100.0, DT=0.005, nhills=3,
                                 hmax=300.0, wmin=700.0, wmax=1800.0, nrec=2)
    med, topo = w.medium(), w.params["topography"]
    g = Solver(med, None, None, topography=topo)
    o = OracleSolver(med, None, None, topography=topo)
    rng = np.random.default_rng(nz)
    for n in FIELDS:
        a = rng.standard_normal(o.f[n].shape).astype(np.float32)
        o.f[n][...] = a
        g.f[n].copy_(torch.from_numpy(a))
    for s in (g, o):
        s.velocity(0)
        s.stress_region(0, *med.dims.i_range, *med.dims.j_range)
    _lib.check()
    for n in FIELDS:
        mm = first_mismatch(g.field(n), o.f[n])
        assert mm is None, f"{nx}x{ny}x{nz}: {n} differs: {mm}"


# nz - 3 stress levels and nz - 2 velocity levels around one wave, 3 ny band
# cells around a block; nz = 5, 6: fstr^T in a launch of its own, in the kernel
@pytest.mark.parametrize("nx,ny,nz", [(20, 21, 5), (21, 20, 6), (20, 85, 66), (20, 86, 67),
                                      (21, 22, 68)])
def test_adjoint_band(gpu, nx, ny, nz):
    from awp_amd.adjoint import AdjointProblem
    from oracle.torch_ref import TorchForward
    torch, _lib = gpu
    nt = 12
    bg, _, src, rec = configs.adjoint_pair(nx=nx, ny=ny, nz=nz, nt=nt, DH=100.0, DT=0.005,
                                           nsrc=2, nrec_side=2, f0=20.0, M0=1.0e22)
    # near the surface, the receivers beside them: a dozen steps reach far enough
    cells = np.array(src.cells)
    cells[:, 2] = 1
    src = type(src)(cells, src.rates)
    rec = type(rec)(cells[:, :2] + 1)
    arrays = lambda m: [torch.from_numpy(a.copy()) for a in (m.lam, m.mu, m.d1)]  # noqa: E731
    leaves = [a.requires_grad_(True) for a in arrays(bg)]
    d = TorchForward(bg, src, rec, nt).run(*leaves)  # observed: silence
    (0.5 * (d ** 2).sum()).backward()
    P = AdjointProblem(bg, src, rec, nt, np.zeros(d.shape, np.float32), checkpoint_every=5,
                       resident_steps=0)
    P.forward()
    for n, a, b in zip(("lam", "mu", "rho"), P.backward(), (x.grad for x in leaves)):
        a = a.cpu()
        err = float(torch.linalg.norm((a - b).flatten()) / torch.linalg.norm(b.flatten()))
        assert err < 2e-3, (n, err)


@pytest.mark.parametrize("nx,ny,nz", [(9, 7, 4), (21, 18, 64), (12, 13, 70)])
def test_adjoint_flush_of_the_grid(gpu, nx, ny, nz):
    """awp_adjoint_flush_grid as awp_adjoint_flush of each array, which are zero
    outside the cells that awp_adjoint_step writes."""
    torch, _lib = gpu
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    d = Dims(nx, ny, nz)
    F, I = C.c_float, C.c_int
    lib.SetDeviceConstValue((F * 1)(50.0), F(0.0025), (I * 1)(nx), (I * 1)(ny), (I * 1)(nz), 1, 0.0,
                            0.0, (F * 9)(), (F * 9)())
    gen = torch.Generator(device="cuda").manual_seed(nz)
    (xs, xe), (ys, ye) = d.i_range, d.j_range
    g32 = [torch.zeros(d.shape, device="cuda") for _ in range(8)]
    for t in g32:
        box = t[xs:xe + 1, ys:ye + 1, 32:d.ktop + 1]
        box.copy_(torch.randn(box.shape, generator=gen, device="cuda"))
    l32 = torch.zeros(d.shape[:2], device="cuda")
    l32[xs:xe + 1, ys:ye + 1] = torch.randn((nx, ny), generator=gen, device="cuda")
    r64 = lambda sh: torch.randn(sh, generator=gen, device="cuda", dtype=torch.float64)  # noqa: E731
    g64, l64 = [r64(d.shape) for _ in range(8)], r64(d.shape[:2])
    a32, a64 = [t.clone() for t in g32 + [l32]], [t.clone() for t in g64 + [l64]]
    for a, b in zip(a32, a64):
        lib.awp_adjoint_flush(a.data_ptr(), b.data_ptr(), a.numel(), st)
    pp = lambda ts: (C.c_void_p * 8)(*[t.data_ptr() for t in ts])  # noqa: E731
    lib.awp_adjoint_flush_grid(pp(g32), pp(g64), l32.data_ptr(), l64.data_ptr(), st)
    _lib.check()
    for got, want in zip(g32 + [l32] + g64 + [l64], a32 + a64):
        assert torch.equal(got, want)


@pytest.mark.parametrize("off,size", [(0, 1), (0, 16), (0, 4099), (1, 4099), (4, 65537)])
def test_move_fields(gpu, off, size):
    """Copies and clears over unaligned starts and ragged ends, nothing beyond."""
    torch, _lib = gpu
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    src = [torch.randint(0, 255, (size + 64,), dtype=torch.uint8, device="cuda") for _ in range(5)]
    dst = [torch.full_like(t, 7) for t in src]
    pp = lambda ts: (C.c_void_p * len(ts))(*[t.data_ptr() + off for t in ts])  # noqa: E731
    want = [t.clone() for t in dst]
    for copy in (True, False):
        lib.awp_move_fields(pp(dst), pp(src) if copy else None, len(dst), size, st)
        _lib.check()
        for w, s, t in zip(want, src, dst):
            w[off:off + size] = s[off:off + size] if copy else 0
            assert torch.equal(w, t)


@pytest.mark.parametrize("fmt", [1, 2], ids=["bf16", "fp16"])
def test_absmax_of_several_fields(gpu, fmt):
    """awp_s16_absmax_fields field by field as awp_s16_absmax: ragged lengths,
    one unaligned array among aligned ones, NaN in one of them."""
    torch, _lib = gpu
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    dt = torch.bfloat16 if fmt == 1 else torch.float16
    gen = torch.Generator(device="cuda").manual_seed(fmt)
    for n, off in ((1, 0), (4097, 0), (4097, 1), (300001, 3)):
        q = [torch.randn(n + 8, generator=gen, device="cuda").mul_(10.0 ** c).to(dt)
             for c in range(4)]
        q[2][n // 2 + off] = float("nan")
        at = [t.data_ptr() + (2 * off if c == 1 else 0) for c, t in enumerate(q)]
        out = torch.full((4,), -1.0, device="cuda")
        one = torch.zeros(4, device="cuda")
        lib.awp_s16_absmax_fields((C.c_void_p * 4)(*at), 4, n, fmt, out.data_ptr(), st)
        for c in range(4):
            lib.awp_s16_absmax(at[c], n, fmt, one[c:].data_ptr(), st)
        _lib.check()
        assert torch.equal(out.view(torch.int32), one.view(torch.int32)), (n, off)
        want = q[0][:n].float().abs().max()
        assert out[0] == want


@pytest.mark.parametrize("kw", [{}, {"variant": "dstrqc_new", "NPC": 2}, {"texture": "table"},
                                {"texture": "rule"}, {"sources": False}, {"receivers": False}],
                         ids=lambda k: "-".join(map(str, k)) or "plain")
def test_native_steps_match_single_steps(gpu, kw):
    """run (awp_run_steps) and a loop over step: sources that end and traces
    that fill up within the run, chunks of check_every."""
    torch, _lib = gpu
    from awp_amd.solver import FIELDS, Solver
    kw = dict(kw)
    w = configs.anelastic(nx=24, ny=21, nz=20, nt=12, DH=200.0, DT=0.01)
    med = w.medium()
    src = w.sources if kw.pop("sources", True) else None
    rec = w.receivers if kw.pop("receivers", True) else None
    a, b = (Solver(med, src, rec, nt_record=9, **kw) for _ in range(2))
    assert a._native()
    a.run(10, check_every=4)
    a.run(6)
    b.start()
    for _ in range(16):
        b.step()
    _lib.check()
    assert a.cur_step == b.cur_step == 16
    assert np.array_equal(a.traces(), b.traces())
    for n in FIELDS:
        mm = first_mismatch(a.field(n), b.field(n))
        assert mm is None, f"{n} differs: {mm}"


def test_replaced_steps_are_called(gpu, monkeypatch):
    """A part of the step replaced on the object or the class runs."""
    torch, _lib = gpu
    from awp_amd.solver import Solver
    w = configs.anelastic(nx=24, ny=21, nz=20, nt=4, DH=200.0, DT=0.01)
    s = Solver(w.medium(), w.sources, w.receivers, nt_record=4)
    seen = []
    s.record = seen.append
    assert not s._native()
    s.run(2)
    assert seen == [0, 1]
    del s.record
    monkeypatch.setattr(Solver, "free_surface", lambda self: seen.append("top"))
    assert not s._native()
    s.run(1)
    assert seen[2:] == ["top"]
