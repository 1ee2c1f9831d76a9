"""The step kernel's rows of 16 lanes (four pencils a wavefront) where they can
go wrong: pencil lengths that fill a row's lanes and lengths that leave some
without a coefficient pair (48, 80), the longest, the (0,0) pencil (which
carries the mean flow, with the constant-mass-flux correction) and the
z-Nyquist pencil beside ordinary ones of the same wavefront, with values that
the start has to drop in both."""
import numpy as np
import pytest

from oracle import kmm_oracle as O
from tests._cases import params, rel, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

KEYS = ("v", "omy", "fn", "gn", "u0", "w0", "h1n", "h3n", "scalar", "scn")


@pytest.mark.parametrize("ny", [32, 48, 80, 96, 128, 192])
@pytest.mark.parametrize("precision", [0, 1])
def test_special_pencils(ny, precision):
    """FP64 1e-10 as the other step tests.  Mixed: FP32 transforms leave the
    state within 1e-6; the nonlinear terms' second derivatives in y magnify the
    FP32 rounding of a field by up to (ny/2)^2 of its own scale, and are small
    here: 5e-3 of their largest value."""
    p = params(32, ny, 32, scalar=True, diff=0.71, scl_flag=6, deltaT=0.3, cmf=True)
    st = seeded(p, 17, amp=0.2)
    rng = np.random.default_rng(ny)
    for k in ("v", "omy"):
        st[k][0, 0, :5] += rng.standard_normal(5)
        st[k][:, p.nzh, :5] += rng.standard_normal((p.nxh, 5))
    print(f"case: special pencils, 32 x {ny + 1} x 32, precision {precision}", flush=True)
    cfg = kmm.make_config(p.nx, ny, p.nz, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, scalar=1, diff=0.71,
                          scl_flag=6, deltaT=0.3, cmf=1, precision=precision)
    sol = O.Solver(p)
    ost = {k: v.copy() for k, v in st.items()}
    with kmm.Channel(cfg) as ch:
        for k in ("v", "omy", "u0", "w0", "scalar"):
            ch.put(k, st[k])
        ch.startup()
        sol.startup(ost)
        for _ in range(2):
            sol.step(ost)
        ch.step(2)
        err = {k: rel(ch.get(k), ost[k]) for k in KEYS}
        bulk = float(O.bulk(ch.get("u0")))
        nyquist = [np.abs(ch.get(k)[:, p.nzh]).max() for k in ("v", "omy", "fn", "gn", "scalar", "scn")]
        zero = [np.abs(ch.get(k)[0, 0]).max() for k in ("v", "omy", "fn", "gn")]
    print({k: f"{e:.1e}" for k, e in err.items()}, flush=True)
    derived = ("fn", "gn", "scn", "h1n", "h3n")
    for k, e in err.items():
        assert e < (1e-10 if precision == 0 else 5e-3 if k in derived else 1e-6), (k, e)
    assert abs(bulk - p.ubulk) < 1e-12 * abs(p.ubulk)
    assert max(nyquist) == 0.0 and max(zero) == 0.0
