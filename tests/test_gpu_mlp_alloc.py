"""A network call whose buffers do not fit the card is refused and leaves the
network as it was for the calls after it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

kmm = pytest.importorskip("polymer_dns_amd.kmm")


def test_calls_after_a_failed_allocation():
    """10^8 samples need 429 GB of training workspace (4.3 KB each), more than
    the card holds; their arrays are never read."""
    net = kmm.Mlp(seed=61)
    rng = np.random.default_rng(62)
    X = rng.standard_normal((300, 22)).astype(np.float32)
    T = rng.standard_normal((300, 6)).astype(np.float32)
    loss, g = net.grad(X, T, mode=1)
    n = 10 ** 8
    with pytest.raises(kmm.KmmError):
        net.grad(np.zeros((n, 22), np.float32), np.zeros((n, 6), np.float32), mode=1)
    loss2, g2 = net.grad(X, T, mode=1)
    assert loss2 == loss and np.array_equal(g2, g)
    losses = net.train(X, T, steps=3, batch=100)
    assert np.isfinite(losses).all()
    net.close()
