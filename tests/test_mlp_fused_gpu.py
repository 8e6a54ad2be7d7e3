"""The fused surrogate kernels at odd widths, row counts and batches: gradients
against the FP64 oracle with the same bf16 rounding points (tolerances as in
test_surrogate_gpu.py), training against the same steps taken one by one
through the gradient call with Adam in numpy (FP32, the same expressions: the
weights agree to a few FP32 roundings), the FP64 evaluation against the FP32 one
to the bit, and nets wider than the fused kernels take."""
import numpy as np
import pytest

import mlp_oracle as MO
from tensum_amd.surrogate import MLP

pytestmark = pytest.mark.gpu

WIDTHS = [[1, 1], [3, 7], [6, 256, 256, 256, 66], [5, 200, 33, 64, 7], [17, 512, 40], [6, 600, 20]]


def _data(widths, n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, widths[0])).astype(np.float32),
            rng.standard_normal((n, widths[-1])).astype(np.float32))


@pytest.mark.parametrize("widths", WIDTHS)
@pytest.mark.parametrize("n", [1, 31, 32, 33, 100])
def test_forward_and_gradient_match_oracle(widths, n):
    print(widths, n, flush=True)
    net = MLP(widths, max_batch=100, seed=3)
    x, t = _data(widths, n, 11)
    ref, _ = MO.forward(net.params.astype(np.float64), widths, x.astype(np.float64), bf=True)
    y = net(x)
    assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref)
    loss, g = net.gradient(x, t)
    lo, go = MO.loss_and_grad(net.params.astype(np.float64), widths, x.astype(np.float64),
                              t.astype(np.float64), bf=True)
    assert abs(loss - lo) <= 1e-4 * lo
    assert np.linalg.norm(g - go) <= 3e-2 * np.linalg.norm(go)


@pytest.mark.parametrize("widths", WIDTHS)
@pytest.mark.parametrize("n,batch", [(70, 32), (100, 100), (65, 64), (9, 4)])
def test_training_is_gradient_steps(widths, n, batch):
    print(widths, n, batch, flush=True)
    x, t = _data(widths, n, 5)
    net, ref = MLP(widths, max_batch=100, seed=4), MLP(widths, max_batch=100, seed=4)
    losses = net.train(x, t, 1, batch=batch, lr=1e-2, seed=9)
    mask, z, perm = (1 << 64) - 1, 9 ^ 0x5851f42d4c957f2d, list(range(n))
    for i in range(n - 1, 0, -1):  # the shuffle: a splitmix64 stream, last index first
        z = (z + 0x9e3779b97f4a7c15) & mask
        h = ((z ^ (z >> 30)) * 0xbf58476d1ce4e5b9) & mask
        h = ((h ^ (h >> 27)) * 0x94d049bb133111eb) & mask
        j = (h ^ (h >> 31)) % (i + 1)
        perm[i], perm[j] = perm[j], perm[i]
    f = np.float32
    p = ref.params
    m, v, total = np.zeros_like(p), np.zeros_like(p), 0.0
    for k, b in enumerate(range(0, n, batch), 1):
        rows = perm[b:b + batch]
        ref.params = p
        loss, g = ref.gradient(x[rows], t[rows])
        total += loss * len(rows) / n
        m = f(0.9) * m + (f(1) - f(0.9)) * g
        v = f(0.999) * v + (f(1) - f(0.999)) * g * g
        c1, c2 = f(1) - f(0.9) ** f(k), f(1) - f(0.999) ** f(k)
        p = p - f(1e-2) * (m / c1) / (np.sqrt(v / c2) + f(1e-8))
    assert abs(losses[0] - total) <= 1e-6 * total
    assert np.abs(net.params - p).max() <= 1e-6


@pytest.mark.parametrize("widths", WIDTHS)
@pytest.mark.parametrize("n", [1, 33, 4097, 40000])
def test_standardised_evaluation_is_the_plain_one(widths, n):
    rng = np.random.default_rng(2)
    net = MLP(widths, max_batch=64, seed=5)
    u = rng.random((n, widths[0]))
    a, b = rng.random(widths[0]), 0.5 + rng.random(widths[0])
    c, d = rng.standard_normal(widths[-1]), 0.5 + rng.random(widths[-1])
    want = net((u - a) / b).astype(np.float64) * d + c
    assert np.array_equal(net.affine(u, a, b, c, d), want)


@pytest.mark.parametrize("width", [256, 257])
def test_deepest_net(width):
    """Sixteen layers, the most a net may have, on both sides of the width up to
    which pre-activations stay on chip: the minibatch kernel's loss is that of the
    evaluation (the same bits; 60 squares added in FP32, 60 eps = 4e-6)."""
    widths = [4] + [width] * 15 + [3]
    print(widths, flush=True)
    net = MLP(widths, max_batch=32, seed=5)
    x, t = _data(widths, 20, 2)
    loss, grad = net.gradient(x, t)
    assert np.all(np.isfinite(grad)) and np.any(grad != 0.0)
    want = np.mean((net(x).astype(np.float64) - t) ** 2)
    np.testing.assert_allclose(loss, want, rtol=2e-5, atol=0)
