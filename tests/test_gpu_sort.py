"""The radix sort at its tile edges and at the line between its two histogram
layouts: the sorted order equals the stable sort of the Morton keys, for spread
and for clustered keys (equal digits and equal keys)."""
import numpy as np
import pytest

from nemo_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n", [2, 63, 64, 65, 511, 4095, 4096, 4097, 8193, 12287, 12288, 12289, 32768, 131071, 131072, 131073,
                               200001])
@pytest.mark.parametrize("kind", ["spread", "clustered", "massless"])
def test_sorted_order_is_the_stable_sort(eng, n, kind):
    r = np.random.default_rng(n)
    x = r.normal(size=(n, 3))
    m = np.full(n, 1.0 / n)
    if kind == "clustered":
        x = np.round(x * 3) / 3 + 1e-9 * r.integers(0, 3, (n, 3))      # few distinct leading digits, many equal keys
    if kind == "massless":
        m[r.uniform(size=n) < 0.3] = 0.0
        m[0] = 1.0
    eng.upload(m, x)
    eng.eval(E.default_params(tol=1.5, eps=0.05, mode="strict" if n < 3 else "fast"))
    keys = eng.debug_keys()
    if kind == "massless":
        keys = keys & ~np.uint64(1 << 63)      # the test set sorts by position alone
    assert np.array_equal(eng.debug_perm(), np.argsort(keys, kind="stable"))
