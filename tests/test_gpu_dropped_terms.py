"""FENE-P channels whose pending evaluation is dropped by kmm_vcw3dp or
kmm_read_restart: a step that solves leaves the terms it used as both the n
and the n-1 terms, whichever of the two copies it stored, and the channel
steps on like one given that state field by field."""
import numpy as np
import pytest

from tests._cases import params, poly_state, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

Q = ("11", "12", "13", "22", "23", "33")
STATE = (["v", "fn", "fnm1", "omy", "gn", "gnm1", "u0", "h1n", "h1nm1", "w0", "h3n", "h3nm1"] + ["c" + q for q in Q]
         + ["c%sn" % q for q in Q] + ["c%snm1" % q for q in Q] + ["str%sn" % q for q in Q] + ["str%snm1" % q for q in Q])


def make(ny, precision):
    p = params(32, ny, 32, dt=0.002, polymer=True, crstrt=1, src_start=0, zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9)
    return p, kmm.Channel(kmm.make_config(32, ny, 32, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, precision=precision,
                                          polymer=1, zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9, crstrt=1, src_start=0))


@pytest.mark.parametrize("graph", [0, 2])
@pytest.mark.parametrize("drop", ["vcw3dp", "restart"])
@pytest.mark.parametrize("ny,precision", [(32, 0), (48, 1), (192, 0)])
def test_dropped_evaluation(tmp_path, ny, precision, drop, graph):
    p, ch = make(ny, precision)
    st = seeded(p, 71, amp=0.2)
    st.update(poly_state(p, 72, amp=0.05))
    for k, v in st.items():
        ch.put(k, v)
    ch.startup()
    path = tmp_path / "restart"
    ch.write_restart(path)
    ch.set_graph(graph)
    ch.step(1)
    ch.step(4)          # with graph = 2: two replays
    before = {k: ch.get(k) for k in ("v", "c11")}
    if drop == "vcw3dp":
        z = np.zeros((p.nxh, p.nz, p.nyp), dtype=np.complex128)
        ch.vcw3dp(z, z, z, z, z, z)
    else:
        ch.read_restart(path)
    for q in Q:
        for t in ("c%sn", "str%sn"):
            n, nm1 = ch.get(t % q), ch.get((t + "m1") % q)
            assert np.abs(n).max() > 0 and np.array_equal(n, nm1), t % q
    state = {k: ch.get(k) for k in STATE}
    assert np.array_equal(state["c11"], before["c11"])
    assert np.array_equal(state["v"], before["v"]) == (drop == "vcw3dp")
    _, other = make(ny, precision)
    for k, v in state.items():
        other.put(k, v)
    for c in (ch, other):
        c.set_graph(0)
        c.step(2)
    assert [k for k in STATE if not np.array_equal(ch.get(k), other.get(k))] == []
    ch.close()
    other.close()
