"""The weight gradient at the edges of its pipeline: k_mlp_wgrad walks groups
of 16 samples, eight groups in flight."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")


@pytest.mark.parametrize("n", [112, 113, 127, 128, 129, 144, 145, 256, 257])
def test_gradient_at_group_edges(n):
    """Seven to nine and sixteen to seventeen groups, full and with one
    sample in the last, FP32 against the oracle's FP64 gradient: sums of FP32
    products over at most 128 inputs per layer and the n samples, rounding
    errors adding up like a random walk through five layers forward and back,
    sqrt(10 * 128) * 2^-24 = 2e-6 of the gradient's norm, with a factor of
    five left."""
    net = kmm.Mlp(seed=81)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 22)).astype(np.float32)
    T = rng.standard_normal((n, 6)).astype(np.float32)
    nm = [np.zeros(22), np.ones(22), np.zeros(6), np.ones(6)]
    net.set_norm(*nm)
    W, b = net.unpack()
    loss, g = net.grad(X, T, mode=0)
    l_ref, gW, gb = M.loss_and_grads([w.astype(np.float64) for w in W], [x.astype(np.float64) for x in b],
                                     X.astype(np.float64), T.astype(np.float64), *nm, mode="fp64")
    gr = np.concatenate([np.concatenate([w.ravel(), x]) for w, x in zip(gW, gb)])
    print(f"n {n}: loss {abs(loss - l_ref) / l_ref:.1e}, gradient {np.linalg.norm(g - gr) / np.linalg.norm(gr):.1e}", flush=True)
    assert abs(loss - l_ref) < 1e-5 * l_ref
    assert np.linalg.norm(g - gr) < 1e-5 * np.linalg.norm(gr)
    net.close()
