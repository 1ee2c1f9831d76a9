"""The conformation tensor's rows of 16 lanes (four pencils a wavefront):
pencil lengths that fill a row's lanes and lengths that leave some without a
coefficient pair, on both sides of the register split (192 and below), through
the release of the polymer (initialisation, the unsmoothed n -> n-1 copy, the
solve), and the n terms, which a step keeps only as the next step's n-1 terms,
read back before and after further steps."""
import numpy as np
import pytest

from oracle import kmm_oracle as O
from tests._cases import params, poly_state, rel, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

TERMS = [f"{k}{q}{t}" for k in ("c", "str") for q in O.POLY for t in ("n", "nm1")]
CONF = ["c" + q for q in O.POLY]


def make(p, precision):
    return kmm.Channel(kmm.make_config(
        p.nx, p.ny, p.nz, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, polymer=1, zlmax=p.zlmax, tpoly=p.tpoly,
        diffpoly=p.diffpoly, qbeta=p.qbeta, c11z=p.c11z, c22z=p.c22z, c33z=p.c33z, ipeter=p.ipeter, itarget=0,
        src_start=p.src_start, irstrt=p.irstrt, crstrt=p.crstrt, precision=precision))


@pytest.mark.parametrize("ny", [32, 48, 80, 96, 128, 192])
@pytest.mark.parametrize("precision,crstrt", [(0, 1), (0, 0), (1, 1)])
def test_polymer_steps(ny, precision, crstrt):
    """FP64 1e-10, mixed 1e-4 for the velocity and 1e-5 for the conformation,
    as the other polymer step tests."""
    p = params(32, ny, 32, dt=0.002, polymer=True, zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9, crstrt=crstrt,
               irstrt=1, src_start=0)
    print(f"case: FENE-P rows 32 x {ny + 1} x 32, precision {precision}, crstrt {crstrt}", flush=True)
    st = seeded(p, 51, amp=0.2)
    if crstrt:
        st.update(poly_state(p, 52, amp=0.05))
    sol = O.Solver(p)
    with make(p, precision) as ch:
        for k in ("v", "omy", "u0", "w0") + (tuple(CONF) if crstrt else ()):
            ch.put(k, st[k])
        ch.startup()
        ost = {k: v.copy() for k, v in st.items()}
        sol.startup(ost)
        for n in (1, 2):
            ch.step(n)
            for _ in range(n):
                sol.step(ost)
            err = {k: rel(ch.get(k), ost[k]) for k in ["v", "omy"] + CONF + (TERMS if precision == 0 else [])}
            print({k: f"{e:.1e}" for k, e in err.items() if e == max(err.values())}, flush=True)
            for k, e in err.items():
                assert e < (1e-10 if precision == 0 else 1e-5 if k in CONF else 1e-4), (k, e)
        assert max(np.abs(ch.get(k)[:, p.nzh]).max() for k in CONF + TERMS) == 0.0
