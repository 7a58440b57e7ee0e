"""The FP64 direct sum over its block shapes, against the oracle bit for bit:
remainders of a stage of sources and of a block of targets, every number of
targets per block, self pairs, massless bodies, no softening, and magnitudes
outside the short form of the quotients (near overflow, underflow and zero)."""
import numpy as np
import pytest

from nemo_amd import engine as E
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


def _same(eng, m, x, eps, idx):
    eng.upload(m, x)
    phi, acc = eng.direct(eps, idx)
    rphi, racc = oracle.direct(m, x, eps, idx)
    assert np.array_equal(phi, rphi, equal_nan=True) and np.array_equal(acc, racc, equal_nan=True)


@pytest.mark.parametrize("n", [1, 2, 23, 24, 25, 191, 192, 193, 385, 1000])
@pytest.mark.parametrize("nidx", [1, 9, 2049, 4100, 9000])     # 8, 8, 16, 32 and 64 targets per block on 256 CUs
def test_direct_shapes(eng, n, nidx):
    r = np.random.default_rng(1000 * n + nidx)
    m = r.uniform(0.5, 1.5, n) * (r.uniform(size=n) > 0.1)
    m[0] = 1.0
    _same(eng, m, r.normal(size=(n, 3)), 0.0 if n % 2 else 0.03, r.integers(0, n, nidx))


@pytest.mark.parametrize("scale,mscale", [(1e-130, 1.0), (1e130, 1.0), (1.0, 1e-130), (1.0, 1e140), (1e-160, 1e-160)])
def test_direct_magnitudes(eng, scale, mscale):
    r = np.random.default_rng(5)
    m, x = r.uniform(0.5, 1.5, 300), r.normal(size=(300, 3))
    big = r.uniform(size=300) < 0.05
    _same(eng, np.where(big, m * mscale, m), np.where(big[:, None], x * scale, x), 0.0, np.arange(300))


def test_direct_coincident_and_nonfinite(eng):
    r = np.random.default_rng(6)
    m, x = r.uniform(0.5, 1.5, 100), r.normal(size=(100, 3))
    x[7] = x[50]
    _same(eng, m, x, 0.0, np.arange(100))
    _same(eng, m, x, 0.01, np.arange(100))
    _same(eng, m[:1], np.array([[np.inf, 0.0, 1.0]]), 0.0, np.arange(1))
