"""Inertial particles, four lanes each: the corner values that a particle keeps
while it stays in a cell (slow particles) and reads again in the next (fast
ones cross cells within a step), and the two forms of the fluid's rates, at the
corners for few particles and at every grid point for many.  Particles do not
act on one another, so the same particles among many others move the same to
the last bit."""
import numpy as np
import pytest

from oracle import kmm_oracle as O
from tests._cases import params, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

MR = dict(particle_flag=1, cd_switch=2, ap=0.01, ratio=2.0, gravity=0.5, c_mu=1.0)


def run(p, st, x, y, z, steps):
    cfg = kmm.make_config(p.nx, p.ny, p.nz, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, **MR)
    with kmm.Channel(cfg) as ch:
        for k in ("v", "omy", "u0", "w0"):
            ch.put(k, st[k])
        ch.set_particles(x, y, z)
        ch.startup()
        ch.step(steps)
        return ch.particles()


@pytest.mark.parametrize("few", [1, 5, 1601])
def test_few_particles_move_as_among_many(few):
    """48 x 33 x 48 points: up to 2534 particles take the corner form."""
    p = params(32, 32, 32, dt=0.01)
    st = seeded(p, 31, amp=0.2)
    rng = np.random.default_rng(7)
    n = 6007
    x, z = rng.uniform(0, p.xl, n), rng.uniform(0, p.zl, n)
    y = rng.uniform(-0.95, 0.95, n) * p.yl / 2
    print(f"case: inertial particles, {few} alone and among {n}", flush=True)
    a = run(p, st, x[:few], y[:few], z[:few], 4)
    b = run(p, st, x, y, z, 4)
    for k in "xyzuvw":
        assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k][:few]), k


@pytest.mark.parametrize("dt", [0.002, 0.05])
def test_particles_that_cross_cells_match_oracle(dt):
    """1e-10 as the other particle tests; at dt = 0.05 two particles
    in three change their cell of the 3/2 grid within the steps."""
    p = params(32, 32, 32, dt=dt)
    st = seeded(p, 33, amp=0.05)
    rng = np.random.default_rng(8)
    n = 203
    x, z = rng.uniform(0, p.xl, n), rng.uniform(0, p.zl, n)
    y = rng.uniform(-0.9, 0.9, n) * p.yl / 2
    print(f"case: inertial particles crossing cells, dt {dt}", flush=True)
    got = run(p, st, x, y, z, 3)
    sol = O.Solver(p)
    sol.swirl_fn = O.swirl_eig
    sol.set_particles(x, y, z, **MR)
    ost = {k: v.copy() for k, v in st.items()}
    sol.startup(ost)
    for _ in range(3):
        sol.step(ost)
    for k in "xyzuvw":
        e = np.abs(got[k] - sol.particles[k]).max()
        print(k, f"{e:.1e}", flush=True)
        assert e < 1e-10 * max(1.0, np.abs(sol.particles[k]).max()), (k, e)
