"""A leapfrog step's closing pass at the edges of its blocks (256 threads, at
most 512 blocks): run() in one launch per step equals force() and drift() bit
for bit, eager and replayed, and the diagnostics equal the sums over the
downloaded state."""
import numpy as np
import pytest

from nemo_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


def terms(m, x, v, a, phi):
    """The 36 terms of every body (code_io.c:351-388 before the closing steps)."""
    t = np.empty((len(m), 36), np.longdouble)
    m, phi = m.astype(np.longdouble), phi.astype(np.longdouble)
    x, v, a = (q.astype(np.longdouble) for q in (x, v, a))
    t[:, 0], t[:, 1], t[:, 2] = m, 0.5 * m * (v * v).sum(1), 0.5 * m * phi
    for i in range(3):
        for j in range(3):
            t[:, 3 + 3 * i + j] = 0.5 * m * v[:, i] * v[:, j]
            t[:, 12 + 3 * i + j] = m * x[:, i] * a[:, j]
            t[:, 21 + 3 * i + j] = m * x[:, i] * v[:, j]
    t[:, 30:33], t[:, 33:36] = m[:, None] * x, m[:, None] * v
    return t


def closed(s, size):
    """Sums and the bound of their error, through the closing steps."""
    am = s[21:30].reshape(3, 3)
    o = np.concatenate([[s[1] + s[2], s[1], s[2]], s[3:21], (am - am.T).ravel(), s[30:36] / s[0]])
    b = size[21:30].reshape(3, 3)
    return o, np.concatenate([[size[1] + size[2], size[1], size[2]], size[3:21], (b + b.T).ravel(), size[30:36] / s[0]])


@pytest.mark.parametrize("n", [2, 255, 256, 257, 511, 513, 10000, 131071, 131072, 131073, 200001])
def test_step_in_one_launch_equals_its_parts(eng, n):
    m, x, v = E.mkplummer(n, seed=n)
    steps, kw = 4, dict(tol=1.0, eps=0.05, mode="strict" if n < 3 else "fast")
    a = E.Leapfrog(eng, m, x, v, 1.0 / 32.0, **kw)
    diag, n2b, nbc = [], [], []
    for k in range(steps):
        b, c = a.force()
        diag.append(a.diagnostics())
        n2b.append(b)
        nbc.append(c)
        if k in (0, steps - 1):
            pos, vel, acc, phi, _ = a.state()
            t = terms(m, pos, vel, acc, phi)
            want, size = closed(t.sum(0), np.abs(t).sum(0))
            # n additions and a few products per term
            assert (np.abs(diag[-1] - want) <= (n + 8) * 2.0 ** -53 * size).all()
        a.drift()
    end = a.state()
    for graph in (False, True):
        b = E.Leapfrog(eng, m, x, v, 1.0 / 32.0, **kw)
        d, p, q = b.run(steps, graph=graph)
        assert np.array_equal(d, diag) and np.array_equal(p, n2b) and np.array_equal(q, nbc)
        for u, w in zip(b.state(), end):
            assert np.array_equal(u, w)
