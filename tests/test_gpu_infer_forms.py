"""Closure inference (kmm_mlp_infer and the closure's step) at the edges of its
16-point tiles, 64-point passes and the passes that are resident at once, for
the three activations, and the field kernel against the row kernel."""
import numpy as np
import pytest

from oracle import mlp_oracle as M
from tests._cases import params, poly_state, seeded

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")

RESIDENT = 256 * 8 * 64   # points of one pass of every wavefront


def make_net(act, seed, sd_y):
    net = kmm.Mlp(seed=seed)
    net.set_activation(act)
    rng = np.random.default_rng(seed)
    nm = [a.astype(np.float32) for a in (0.1 * rng.standard_normal(22), 1.0 + rng.uniform(0, 1, 22),
                                         0.1 * rng.standard_normal(6), np.full(6, sd_y))]
    p = net.params()
    W, b = net.unpack(p)
    for x in b:
        x[:] = 0.05 * rng.standard_normal(x.shape)
    net.set_params(p)
    net.set_norm(*nm)
    return net, nm, net.unpack()


@pytest.mark.parametrize("act", ["relu", "gelu", "gelu_poly"])
def test_inference_at_tile_edges(act):
    """Every size gives the rows of the largest bit for bit (a row's sums do
    not depend on its tile), and the largest the oracle's bf16 forward: sums
    in another order (2^-24) flip a bf16 rounding (2^-8) in about one of
    10^4 activations, and a flip reaches the outputs through weights of about
    1/sqrt(128), so that half of the rows agree to FP32 and none is off by
    more than a few flips of large activations."""
    net, nm, (W, b) = make_net(act, 31, 1.0)
    rng = np.random.default_rng(32)
    n = RESIDENT + 65
    X = rng.standard_normal((n, 22)).astype(np.float32)
    Y = net.infer(X)
    M.ACT = act
    try:
        Yr = M.forward(W, b, X, *nm, mode="bf16")
    finally:
        M.ACT = "relu"
    err = np.abs(Y - Yr) / np.abs(Yr).max()
    print(f"{act}: median {np.median(err):.1e}, max {err.max():.1e}", flush=True)
    assert np.median(err) < 1e-3 and err.max() < 3e-2
    for k in (1, 15, 16, 17, 63, 64, 65, 511, 512, 513, RESIDENT - 1, RESIDENT, RESIDENT + 1):
        assert np.array_equal(net.infer(X[:k]), Y[:k]), k
    net.close()


@pytest.mark.parametrize("act", ["relu", "gelu", "gelu_poly"])
@pytest.mark.parametrize("n,precision", [(32, 0), (64, 0), (64, 1)])
def test_field_inference_equals_row_inference(act, n, precision):
    """The stress a closure step leaves is 2 h1 - h2 + y of its captured
    features: t - h1 - (h1 - h2) gives y back up to the four roundings on the
    way, 2^-24 of the sums each (a factor of two is left)."""
    p = params(n, 32, n, dt=0.002, polymer=True, crstrt=1, src_start=0, zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9)
    st = seeded(p, 41, amp=0.2)
    st.update(poly_state(p, 42, amp=0.05))
    cfg = kmm.make_config(n, 32, n, xl=p.xl, zl=p.zl, re=p.re, dt=p.dt, r_tau=p.R_tau, precision=precision, polymer=1,
                          zlmax=30.0, tpoly=0.5, diffpoly=0.5, qbeta=0.9, crstrt=1, src_start=0)
    net, _, _ = make_net(act, 43, 0.5)
    with kmm.Channel(cfg) as ch:
        for k, v in st.items():
            ch.put(k, v)
        ch.startup()
        ch.set_poly_capture(True)
        ch.step(3)
        ch.set_closure(net)
        ch.step(1)
        X, T = ch.poly_samples(20000, seed=44)
        y = net.infer(X).astype(np.float64)
        h1, d = X[:, 10:16].astype(np.float64), X[:, 16:22].astype(np.float64)
        bound = 2.0 ** -23 * (np.abs(h1 + d) + np.abs(h1 + d + y) + np.abs(d + y) + np.abs(T))
        worst = (np.abs(T - y) / bound).max()
        print(f"{act} {n} {precision}: {worst:.2f} of the bound, |y| {np.abs(y).max():.2f}", flush=True)
        assert np.abs(y).max() > 0.1 and worst <= 1.0
    net.close()
