"""The (k, j) tiles of the marching Cartesian kernels (awp_pick_tile) at the
column heights where the rule changes: one wave and less, 64 m levels, one row
per workgroup of 2, 3 and 4 waves, 64-level runs beyond 256 and 32-level runs up to 32 (in 16-bit
storage up to 96); and the two routes of the free-surface velocity ghosts.  Bit for bit against the oracle: the arithmetic
is the same expression by expression, so the tolerance is zero."""
import ctypes as C

import numpy as np
import pytest

from awp_amd.grid import Dims
from tests._fields import WAVE, first_mismatch, random_state

pytestmark = pytest.mark.gpu

DH, DT = 50.0, 0.0025
VEL = ("u1", "v1", "w1", "xx", "yy", "zz", "xy", "xz", "yz")
STR = ("xx", "yy", "zz", "xy", "xz", "yz", "r1", "r2", "r3", "r4", "r5", "r6", "u1", "v1", "w1")


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awp_amd import _lib
    return torch, _lib.load(), _lib


@pytest.mark.parametrize("nz", [4, 5, 31, 32, 33, 36, 61, 64, 65, 101, 128, 130, 191, 193, 255, 256, 257, 300])
def test_column_heights_bit_exact(gpu, oracle_lib, nz):
    _velocity_stress(gpu, oracle_lib, Dims(11, 9, nz))


@pytest.mark.parametrize("nx,ny,nz", [(256, 256, 4), (257, 256, 5), (512, 256, 4), (513, 256, 4)])
def test_surface_ghosts_bit_exact(gpu, oracle_lib, nx, ny, nz):
    """The velocity ghosts in the stress kernel (up to 2^17 columns) and in
    their own launch (more)."""
    _velocity_stress(gpu, oracle_lib, Dims(nx, ny, nz))


@pytest.mark.parametrize("variant,NPC", [("dstrqc", 2), ("dstrqc_new", 0), ("dstrqc_new", 2)])
@pytest.mark.parametrize("nx,nz", [(60, 6), (513, 5)])
def test_surface_ghost_bounds_bit_exact(gpu, oracle_lib, nx, nz, variant, NPC):
    """Where vs1 and vs2 exist, in both routes of the ghosts: dstrqc_new keeps
    vs1 on periodic boundaries, both keep vs2."""
    _velocity_stress(gpu, oracle_lib, Dims(nx, 256, nz), variant, NPC)


# 16-bit storage: the ghosts in the stress kernel up to 2^16 columns and in
# their own launch beyond; columns of 32-level runs (up to 32, 65 to 96 levels),
# one row per workgroup, and 514 waves per velocity chunk
@pytest.mark.parametrize("storage", ["bf16", "fp16"])
@pytest.mark.parametrize("nx,ny,nz,texture", [(256, 256, 5, "arrays"), (257, 256, 4, "arrays"),
                                              (257, 256, 6, "rule"), (20, 17, 31, "table"),
                                              (21, 18, 66, "arrays"), (20, 19, 96, "rule"),
                                              (20, 18, 97, "arrays"), (274, 258, 97, "arrays")])
def test_16bit_surfaces_and_columns_bit_exact(gpu, oracle_lib, nx, ny, nz, texture, storage):
    torch, _, _lib = gpu
    from awp_amd import configs
    from awp_amd.solver import Solver16
    from awp_amd.storage import FIELDS16
    from oracle.oracle import OracleSolver16
    med = configs.anelastic(nx=nx, ny=ny, nz=nz, nt=2, DH=100.0, DT=0.005).medium()
    g = Solver16(med, None, None, storage=storage, texture=texture)
    o = OracleSolver16(med, None, None, storage=storage)
    rng = np.random.default_rng(nz)
    dt = torch.bfloat16 if storage == "bf16" else torch.float16
    for n in FIELDS16:
        # moderate stored values: no stress leaves the range of binary16
        x = rng.standard_normal(med.dims.shape, dtype=np.float32)
        q = torch.from_numpy(x * np.float32(0.01 if n in VEL[:3] else 1.0)).to(dt)
        g.f[n].copy_(q.view(torch.int16))
        o.levels[0].q[n][...] = q.view(torch.int16).numpy().view(np.uint16)
    for s in (g, o):
        s.velocity(0)
        s.stress_region(0, *med.dims.i_range, *med.dims.j_range)
    _lib.check()
    for n in FIELDS16:
        a, b = g.raw(n), o.levels[0].q[n]
        bad = np.argwhere(a != b)
        assert len(bad) == 0, (n, len(bad), tuple(bad[0]))
    top = o.field("w1")[..., med.dims.ktop + 1]
    assert np.isfinite(top).all() and np.abs(top).max() > 0


# ten arrays of 253 and 259 MiB, chunks of 510, 514 and 516 waves; 257 and 129
# tiles are no multiple of the XCDs
@pytest.mark.parametrize("nx,ny,nz", [(186, 257, 65), (190, 257, 65), (192, 255, 65),
                                      (99, 515, 64)])
def test_velocity_block_orders_bit_exact(gpu, oracle_lib, nx, ny, nz):
    """XCDs with i-chunks of their own and (arrays beyond 256 MiB, chunks of 512
    waves and more) side by side in one chunk."""
    _velocity_stress(gpu, oracle_lib, Dims(nx, ny, nz))


def _velocity_stress(gpu, oracle_lib, d, variant="dstrqc", NPC=0):
    torch, lib, _lib = gpu
    st, med = random_state(d, seed=3 + d.nzt)
    F, I = C.c_float, C.c_int
    z9 = (F * 9)()
    lib.SetDeviceConstValue((F * 1)(DH), F(DT), (I * 1)(d.nxt), (I * 1)(d.nyt), (I * 1)(d.nzt),
                            1, 0.0, 0.0, z9, z9)
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in {**st, **med}.items()}
    host = {k: v.copy() for k, v in st.items()}
    p = lambda n: dev[n].data_ptr()  # noqa: E731
    q = lambda n: (host[n] if n in host else med[n]).ctypes.data  # noqa: E731
    s = torch.cuda.current_stream().cuda_stream
    (s_i, e_i), (s_j, e_j) = d.i_range, d.j_range
    sp = ("dcrjx", "dcrjy", "dcrjz")
    lib.dvelcx_H_opt(*map(p, VEL + sp), p("d1"), d.nyt, d.nzt, s, s_i, e_i, 0, 1)
    stress = lib.dstrqc_H if variant == "dstrqc" else lib.dstrqc_H_new
    stress(*map(p, STR), *map(p, ("lam", "mu", "qp", "coeff", "qs") + sp), d.nyt, d.nzt, s,
           *map(p, ("lam_mu", "vx1", "vx2", "ww", "wwo")), d.nxt, NPC, 0, 0, s_i, e_i, s_j, e_j,
           0)
    _lib.check()
    o = oracle_lib.load()
    o.awp_oracle_dvelcx_f32(*map(q, VEL + sp), q("d1"), d.nxt, d.nyt, d.nzt, DH, DT, s_i, e_i, 0,
                            1)
    getattr(o, f"awp_oracle_{variant}_f32")(
        *map(q, STR), *map(q, ("lam", "mu", "qp", "coeff", "qs") + sp),
        *map(q, ("lam_mu", "vx1", "vx2", "ww", "wwo")), d.nxt, d.nyt, d.nzt, DH, DT, d.nxt, NPC, 0,
        0, s_i, e_i, s_j, e_j, 0)
    torch.cuda.synchronize()
    for n in WAVE:
        mm = first_mismatch(dev[n].cpu().numpy(), host[n])
        assert mm is None, f"nz={nz}: {n} differs: {mm}"
