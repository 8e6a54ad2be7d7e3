"""The shapes of inputs a surrogate is called with: whatever standardising
them by the input means broadcasts to rows of n_in numbers, one uncertain input
given as a plain vector among them."""
import numpy as np
import pytest

from tensum_amd.surrogate import Surrogate

pytestmark = pytest.mark.gpu


def test_one_input_as_a_vector():
    rng = np.random.default_rng(3)
    u = rng.random(40)
    q = np.stack([np.sin(3 * u), u ** 2], 1)
    net = Surrogate(1, 2, hidden=(16,), max_batch=64, seed=1)
    net.fit(u[:, None], q, epochs=2, batch=20)
    want = net(u[:, None])
    assert want.shape == (40, 2)
    assert np.array_equal(net(u), want)
    assert np.array_equal(net(list(u)), want)
    assert np.array_equal(net(u[:1]), want[:1])
    assert np.array_equal(net(u[:, None, None]), want)


def test_a_fit_to_vectors():
    rng = np.random.default_rng(4)
    u = rng.random(40)
    a, b = (Surrogate(1, 1, hidden=(16,), max_batch=64, seed=1) for _ in range(2))
    la = a.fit(u, u ** 2, epochs=2, batch=20)
    lb = b.fit(u[:, None], (u ** 2)[:, None], epochs=2, batch=20)
    assert np.allclose(la, lb, rtol=1e-6, atol=0)
    assert a(u).shape == (40, 1)
    assert np.array_equal(a(u), a(u[:, None]))


def test_rows_of_the_wrong_width_are_refused():
    net = Surrogate(3, 2, hidden=(16,), max_batch=64, seed=1)
    with pytest.raises(ValueError):
        net(np.zeros((5, 2)))
    with pytest.raises(ValueError):
        net(np.zeros(3))
    assert net(np.zeros((5, 1))).shape == (5, 2)   # one number a row is every input's
    assert net(np.zeros((0, 3))).shape == (0, 2)


def test_moments_of_every_shape():
    rng = np.random.default_rng(5)
    net = Surrogate(3, 2, hidden=(16,), max_batch=64, seed=1)
    u = rng.random((5, 3))
    net.mu_x, net.sd_x = u.mean(0), u.std(0)
    net.mu_y, net.sd_y = np.array([1.0, 2.0]), np.array([3.0, 4.0])
    want = net(u)
    assert np.array_equal(want, net.net((u - net.mu_x) / net.sd_x).astype(np.float64) * net.sd_y + net.mu_y)
    for name in ("mu_x", "sd_x", "mu_y", "sd_y"):
        setattr(net, name, getattr(net, name)[None, :])
        assert np.array_equal(net(u), want), name
    for name in ("mu_x", "mu_y"):  # one of each per row
        setattr(net, name, np.repeat(getattr(net, name), 5, 0))
        assert np.array_equal(net(u), want), name
