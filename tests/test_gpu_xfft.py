"""The x transforms of the plane kernels at every compiled line length (48,
96, 144, 192, 288, 384 points: six factorisations into two register passes,
one to five lines a wavefront, with partial last batches for the 6 and 9 in,
3 and 4 out fields of the Navier-Stokes plane, the 21 and 6 of the polymer
plane and the 4 of the gradient plane) against the oracle's transforms."""
import functools

import numpy as np
import pytest

from oracle import kmm_oracle as O
from tests._cases import params, poly_state, rel, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

GRIDS = [(32, 32), (64, 32), (96, 96), (128, 64), (192, 192), (256, 128)]


@functools.lru_cache(maxsize=1)
def evaluation(nx, nz):
    """Inputs and the oracle's evaluation of one state, with and without the scalar."""
    p = params(nx, 32, nz, scalar=True, dt=0.005, polymer=True, tpoly=0.5, zlmax=30.0, qbeta=0.9, src_start=0)
    st = seeded(p, 44, amp=0.3)
    C = poly_state(p, 45, amp=0.05)
    C = {ij: C["c" + ij] for ij in O.POLY}
    u, v, w = O.veloc(st["v"], st["omy"], st["u0"], st["w0"], p)
    omx, omz = O.vort(u, v, w, p)
    grad = list(O.gradscl(st["scalar"], p))
    for a in [u, v, w, omx, omz] + grad:
        O.norm(a)
    gv, dC = O.gradv(u, v, w, p), O.derivscji(C, p)
    fields = dict(u=u, v=v, w=w, omx=omx, omy=st["omy"], omz=omz, C=C, dC=dC, gradv=gv, sclx=grad[0], scly=grad[1],
                  sclz=grad[2])
    z = np.zeros((p.mx, p.mz, p.nyp))
    gn, fn, oz, scn, phys = O.vcw3dp(dict(fxintg=z, fyintg=z, fzintg=z), p, 1, fields)
    gp = [[O.to_physical(gv[f"u{i}{k}"], p) for k in (1, 2, 3)] for i in (1, 2, 3)]
    return p, st, fields, [O.norm(a) for a in (gn, fn, oz, scn)], phys, O.swirl_eig(gp)


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("precision", [0, 1])
def test_plane_transforms_at_every_line_length(grid, precision):
    """FP64: 1e-11 of the largest value, the bound of the other evaluation
    tests.  Mixed: FP32 transforms of two directions and a product of two
    fields, about ten roundings of 2^-24 growing with sqrt(log2(points)) ~ 4
    and the 100-fold scale between a term's factors and the sum: 2e-5.  The swirl
    strength, the imaginary part of an eigenvalue pair, grows like the square
    root of the gradient's rounding near a vanishing discriminant: 1e-7, 1e-3."""
    p, st, f, want, phys, swirl = evaluation(*grid)
    tol, tol_swirl = (1e-11, 1e-7) if precision == 0 else (2e-5, 1e-3)
    print(f"grid {grid[0]} x {grid[1]}, precision {precision}", flush=True)
    base = dict(xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, precision=precision)
    full = [f["C"][O._CIDX[(i, j)]] for i in range(3) for j in range(3)]
    dc = [None] * 27
    for i in range(3):
        for j in range(3):
            for k in range(3):
                dc[9 * j + 3 * i + k] = f["dC"][O._CIDX[(i, j)]][k]
    args = (f["u"], f["v"], f["w"], f["omx"], f["omy"], f["omz"])
    with kmm.Channel(kmm.make_config(p.nx, p.ny, p.nz, scalar=1, **base)) as ch:
        # 9 fields in, 4 out
        for name, a, b in zip(("gn", "fn", "omz", "scn"), ch.vcw3dp(*args, f["sclx"], f["scly"], f["sclz"]), want):
            assert rel(a, b) < tol, (name, rel(a, b))
    with kmm.Channel(kmm.make_config(p.nx, p.ny, p.nz, polymer=1, tpoly=p.tpoly, zlmax=p.zlmax, qbeta=p.qbeta, crstrt=1,
                                     src_start=0, **base)) as ch:
        # 6 fields in, 3 out, and the polymer plane
        gn, fn, oz, cn, sn, _ = ch.vcw3dp_poly(*args, [f["gradv"][f"u{i}{k}"] for i in (1, 2, 3) for k in (1, 2, 3)],
                                               full, dc)
        for name, a, b in zip(("gn", "fn", "omz"), (gn, fn, oz), want):
            assert rel(a, b) < tol, (name, rel(a, b))
        for ij in O.POLY:
            for got, key in ((cn, "cn"), (sn, "str")):
                b = O.norm(phys["poly"][key][ij].copy())
                assert rel(got[ij], b) < tol, (key, ij, rel(got[ij], b))
        # the velocity capture and the gradient plane, at 500 tracers
        for k in ("v", "omy", "u0", "w0"):
            ch.put(k, st[k])
        for ij in O.POLY:
            ch.put("c" + ij, f["C"][ij])
        rng = np.random.default_rng(7)
        x, y, z = rng.uniform(0, p.xl, 500), rng.uniform(-0.95, 0.95, 500), rng.uniform(0, p.zl, 500)
        ch.set_particles(x, y, z)
        ch.startup()
        got = ch.particles()
    ref = O.fluid_interp(x, y, z, [phys["up"], phys["vp"], phys["wp"], swirl], p)
    for k, b in zip(("u", "v", "w", "swirl"), ref):
        t = tol if k != "swirl" else tol_swirl
        assert rel(got[k], b) < t, (k, rel(got[k], b))
