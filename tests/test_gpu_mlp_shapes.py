"""Training kernels at the edges of their blocks: gradients of batches around
multiples of 16 and 64 samples against the oracle, output scales against a
partial sort, and training batches gathered from the set against gradients of
the same rows."""
import numpy as np
import pytest

from nemo_amd import engine as E
from oracle import mlp_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 130, 2113])
def test_gradient_shapes(eng, n):
    eng.mlp_init(seed=4)
    p, _ = eng.mlp_get()
    r = np.random.default_rng(n)
    x = r.normal(size=(n, 12)).astype(np.float32)
    t = (0.3 * r.normal(size=(n, E.MLP_OUT))).astype(np.float32)
    g, loss = eng.mlp_grad(x, t)
    gref, lref = mlp_oracle.grad(p, x, t)
    assert abs(loss - lref) / lref < 1e-2
    k = 0
    for s in mlp_oracle.SIZES:
        m = int(np.prod(s))
        a, b = g[k:k + m], gref[k:k + m]
        assert np.linalg.norm(a - b) <= 3e-2 * np.linalg.norm(b) + 1e-7, s
        k += m


def _collect(eng, n, seed):
    m, x, _ = E.mkplummer(n, seed, with_vel=False)
    eng.upload(m, x)
    eng.mlp_clear_samples()
    eng.mlp_collect(E.default_params(tol=1.1, eps=0.01, usequad=1, group_size=192, nleaf=1), rlo=0.45, rhi=1.5)
    return eng.mlp_samples()


@pytest.mark.parametrize("n", [3000, 40000])
def test_output_scales(eng, n):
    eng.mlp_init(seed=1)
    _, Y = _collect(eng, n, 21)
    eng.mlp_train(epochs=1, batch=64, lr=1e-3)
    _, norm = eng.mlp_get()
    for got, blk in ((norm[0], Y[:, :3]), (norm[3], Y[:, 3:])):
        a = np.abs(blk).ravel()
        lim = np.partition(a, int(0.99 * (len(a) - 1)))[int(0.99 * (len(a) - 1))]
        ref = np.sqrt(np.mean(a[a <= lim].astype(np.float64) ** 2))
        assert abs(got - ref) <= 2e-7 * ref      # one rounding to FP32


@pytest.mark.parametrize("batch", [64, 100, 1000])
def test_epoch_is_the_permuted_rows(eng, batch):
    """The loss of an epoch is that of its rows (a i + c) mod n, scaled and
    clipped, at the starting weights (learning rate ~ 0)."""
    X, Y = _collect(eng, 3000, 22)
    n = len(X)
    assert n >= batch
    eng.mlp_init(seed=9)
    p, _ = eng.mlp_get()
    seed = 5
    mask = (1 << 64) - 1
    rs = (seed * 0x9e3779b97f4a7c15 + 7) & mask

    def rnd():
        nonlocal rs
        rs ^= (rs << 13) & mask
        rs ^= rs >> 7
        rs ^= (rs << 17) & mask
        return rs

    a = (rnd() % n) | 1
    while np.gcd(a, n) != 1:
        a = (a + 2) % n
    c = rnd() % n
    loss = eng.mlp_train(epochs=1, batch=batch, lr=1e-30, seed=seed)
    _, norm = eng.mlp_get()
    used = n - n % batch
    rows = [(a * i + c) % n for i in range(used)]
    y = np.clip(Y[rows] / np.where(np.arange(9) < 3, norm[0], norm[3]), -10.0, 10.0)
    ref = mlp_oracle.forward(p, X[rows])
    assert abs(loss[0] - ((ref - y) ** 2).sum() / used) < 1e-2 * loss[0]
