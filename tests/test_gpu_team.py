"""The step kernel's two forms, four wavefronts on the same four pencils (few
pencils) and a wavefront each (many; the tuning's other variant runs it at any
size): the same steps on one channel, with and without the scalar, at constant
mass flux, through a step that starts from the stored nonlinear terms, and with
the polymer's force and velocity gradients."""
import numpy as np
import pytest

from tests._cases import params, poly_state, rel, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

POLY = dict(zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9, crstrt=1, src_start=0)


def run(p, st, variant, **kw):
    cfg = kmm.make_config(p.nx, p.ny, p.nz, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, cmf=1, **kw)
    with kmm.Channel(cfg) as ch:
        for k, v in st.items():
            ch.put(k, v)
        ch.startup()
        ch.set_tuning(variant, 0)
        ch.step(2)
        ch.put("fn", ch.get("fn"))   # the next step loads fn, gn, scn
        ch.step(2)
        keys = ["v", "omy", "u0", "w0", "fn", "gn", "fnm1", "gnm1", "h1n", "h3n"]
        keys += ["scalar", "scn", "scnm1"] if kw.get("scalar") else []
        keys += ["c12", "c22"] if kw.get("polymer") else []
        return {k: ch.get(k) for k in keys}


@pytest.mark.parametrize("ny,kind", [(32, "flow"), (48, "scalar"), (64, "poly"), (80, "flow"), (96, "scalar"),
                                     (128, "scalar"), (192, "flow"), (192, "scalar")])
@pytest.mark.parametrize("precision", [0, 1])
def test_team_and_rows_agree(ny, kind, precision):
    """Bit for bit: the two forms write the same expressions, and products are
    contracted with additions within an expression only.  (A member of an
    ensemble, whose launches take the rows' form, equals the channel alone.)"""
    p = params(32, ny, 32, dt=0.002, scalar=kind == "scalar")
    st = seeded(p, 23, amp=0.2)
    if kind != "scalar":
        st = {k: st[k] for k in ("v", "omy", "u0", "w0")}
    else:
        st = {k: st[k] for k in ("v", "omy", "u0", "w0", "scalar")}
    kw = dict(precision=precision)
    if kind == "scalar":
        kw.update(scalar=1, diff=0.71, scl_flag=6, deltaT=0.3)
    if kind == "poly":
        kw.update(polymer=1, **POLY)
        st.update(poly_state(p, 24, amp=0.05))
    print(f"case: step forms, 32 x {ny + 1} x 32, {kind}, precision {precision}", flush=True)
    a, b = run(p, st, 0, **kw), run(p, st, 1, **kw)
    for k in a:
        assert np.isfinite(a[k]).all() and np.array_equal(a[k], b[k]), (k, rel(a[k], b[k]))
