"""One closure network serving two channels of an ensemble, one of which
retrains it: the other channel's steps, queued before on its own stream, run
with the weights of their time."""
import numpy as np
import pytest

from tests._cases import params, poly_state, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

FIELDS = ["v", "omy", "u0"]
STEPS = 20


def channel(n, seed):
    p = params(n, 32, n, dt=0.002, polymer=True, crstrt=1, src_start=0, zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9)
    st = seeded(p, seed, amp=0.2)
    st.update(poly_state(p, seed + 1, amp=0.05))
    ch = kmm.Channel(kmm.make_config(n, 32, n, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, polymer=1, zlmax=30.0,
                                     tpoly=0.5, diffpoly=0.5, qbeta=0.9, crstrt=1, src_start=0))
    for k, v in st.items():
        ch.put(k, v)
    ch.startup()
    ch.set_poly_capture(True)
    ch.step(3)
    return ch


def run(together):
    """Channel a (64 x 33 x 64) only uses the network, b (32 x 33 x 32) also
    trains it at the end of every audit window."""
    net = kmm.Mlp(seed=51)
    net.set_activation("gelu_poly")
    net.set_norm(np.zeros(22), np.ones(22), np.zeros(6), np.full(6, 1e-3))
    a, b = channel(64, 52), channel(32, 54)
    for ch in (a, b):
        ch.set_closure(net)
    b.set_closure_audit(5, window=3, gate=1e30)
    b.set_closure_retrain(8, batch=256, lr=1e-2, seed=3)
    w0 = net.params()
    if together:
        kmm.ensemble_step([a, b], STEPS)
    else:
        a.step(STEPS)
        b.step(STEPS)
    out = {(m, k): ch.get(k) for m, ch in (("a", a), ("b", b)) for k in FIELDS}
    out.update({("a", "stress"): a.poly_stress(1), ("b", "stress"): b.poly_stress(1)})
    out[("net", "params")] = net.params()
    assert b.closure_status()["audits"] >= 2 and not np.array_equal(out[("net", "params")], w0)
    for ch in (a, b):
        ch.close()
    net.close()
    return out


def test_retraining_waits_for_the_other_channels_steps():
    """The ensemble queues a's steps, then b's: the same as a's steps first,
    then b's, bit for bit."""
    one, two = run(False), run(True)
    assert all(np.isfinite(v).all() for v in one.values())
    assert [k for k in one if not np.array_equal(one[k], two[k])] == []
