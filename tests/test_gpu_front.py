"""The tree build at the lines between its forms (one block for everything, a
sorted tile per block and merging, radix passes; the box by one block, by the
last compacting block, by rounds over many): keys, sorted order and cells equal
the oracle's exactly, for spread keys, runs of equal upper halves of every
handled length, chains of cells, massless bodies and bodies that grow the box
late."""
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


def bodies(n, kind):
    r = np.random.default_rng(n)
    x = r.normal(size=(n, 3))
    m = r.uniform(0.5, 1.5, n) / n
    if kind == "runs":          # knots of 2 .. 1000 bodies, each within 2^-12 of the box
        at = 0
        for k in (2, 3, 8, 9, 10, 63, 64, 65, 511, 512):
            if at + k <= n:
                x[at:at + k] = r.uniform(-1.5, 1.5, 3) + r.uniform(-1e-4, 1e-4, (k, 3))
            at += k
        x = x[r.permutation(n)]
    if kind == "knot":          # most bodies in one knot: no run list holds it
        x[: 3 * n // 4] = 0.3 + 1e-4 * x[: 3 * n // 4]
        x = x[r.permutation(n)]
    if kind == "pairs":         # a chain of cells per pair, many more cells than bodies
        x[1::2] = x[: n // 2 * 2 : 2] + 3e-6
        x = x[r.permutation(n)]
    if kind == "massless":
        m[r.uniform(size=n) < 0.3] = 0.0
        m[:2] = 1.0 / n
    if kind == "late":          # the box grows for bodies far behind the first ones
        for k, i in enumerate(np.unique(np.linspace(n // 2, n - 1, 5).astype(int))):
            x[i] = 10.0 ** (k + 1) * np.array([1.0, -0.5, 0.25])
    return m, x


def expanded(m, x, rmin, size):
    """expandbox (load.c:68-95) in input order, in float64."""
    rmin = np.array(rmin, np.float64)
    i = 0
    while True:
        r = (x[i:] - rmin) / size
        out = np.flatnonzero((m[i:] != 0) & ~((r >= 0.0) & (r < 1.0)).all(1))
        if not len(out):
            return rmin, size
        i += int(out[0])
        while not (((x[i] - rmin) / size >= 0) & ((x[i] - rmin) / size < 1)).all():
            rmin = np.where(x[i] < rmin + 0.5 * size, rmin - size, rmin)
            size = 2.0 * size


def check(e, m, x, rsize):
    st = e.eval(E.default_params(tol=1.5, eps=0.05, rsize=rsize))
    rmin, size = expanded(m, x, np.full(3, -0.5 * rsize), rsize)
    assert st.rsize == size and np.array_equal(np.array(st.rmin), rmin)
    perm = e.debug_perm()
    keys = e.debug_keys() & ~np.uint64(1 << 63)          # the test set sorts by position alone
    assert np.array_equal(perm, np.argsort(keys, kind="stable"))
    k = (np.clip((x - rmin) / size, 0, 1 - 2.0 ** -53) * 2.0 ** 30).astype(np.uint64) >> np.uint64(9)
    want = np.zeros(len(x), np.uint64)
    for b in range(21):
        for c in range(3):
            want |= ((k[:, c] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + 2 - c)
    assert np.array_equal(keys, want)
    c = e.debug_cells()
    t = oracle.tree_cells(m, x, np.full(3, -0.5 * rsize), rsize, maxcell=22 * len(x) + 64, depth_cap=21)
    assert np.array_equal(c["level"], t["level"]) and np.array_equal(c["nbody"], t["nbody"])
    # prefix sums in the place of the oracle's: n additions of terms of one sign
    assert np.abs(c["mass"] - t["mass"]).max() <= len(x) * 2.3e-16 * m.sum()


@pytest.mark.parametrize("n", [2, 3, 64, 1025, 2048, 2049, 6143, 6144, 6145, 12287, 12288, 12289, 16384, 16385, 40961])
@pytest.mark.parametrize("kind", ["spread", "runs", "knot", "pairs", "massless", "late"])
def test_build_at_the_lines(eng, n, kind):
    m, x = bodies(n, kind)
    eng.upload(m, x)
    check(eng, m, x, 4.0)


@pytest.mark.parametrize("n", [4097, 8191, 8192, 16385, 65535, 65536, 65537, 262145, 1 << 19, (1 << 19) + 1, (1 << 20) - 1, 1 << 20,
                               (1 << 20) + 1])
def test_merge_and_radix_sort_at_their_line(eng, n):
    m, x = bodies(n, "massless")
    eng.upload(m, x)
    eng.eval(E.default_params(tol=1.5, eps=0.05))
    keys = eng.debug_keys() & ~np.uint64(1 << 63)
    assert np.array_equal(eng.debug_perm(), np.argsort(keys, kind="stable"))


# (rsize 2^-6 leaves nearly every body outside; 3 is no power of two)
@pytest.mark.parametrize("n", [2000, 9000, (1 << 15) + 8192, (1 << 15) + 8193, 150000, 600000])
@pytest.mark.parametrize("rsize", [2.0 ** -6, 3.0, 64.0])
def test_box_from_any_start(eng, n, rsize):
    m, x = bodies(n, "late")
    eng.upload(m, x)
    st = eng.eval(E.default_params(tol=1.5, eps=0.05, rsize=rsize))
    rmin, size = expanded(m, x, np.full(3, -0.5 * rsize), rsize)
    assert st.rsize == size and np.array_equal(np.array(st.rmin), rmin)


@pytest.mark.parametrize("nt", [1, 2, 2048, 2049, 6145, 12288, 12289])
def test_separate_test_points(eng, nt):
    m, x = bodies(20000, "spread")
    t = bodies(nt + 4000, "knot")[1][:nt]
    eng.upload(m, x, tpos=t)
    eng.eval(E.default_params(tol=0.7, eps=0.05))
    first, count = eng.debug_groups()
    o = np.argsort(first)
    first, count = first[o], count[o]
    assert np.array_equal(np.sort(eng.debug_perm()), np.arange(nt))
    assert first[0] == 0 and np.array_equal(first[1:], np.cumsum(count)[:-1]) and count.sum() == nt
    phi, acc = eng.download()
    eng.eval(E.default_params(tol=0.7, eps=0.05, mode="strict"))
    phi0, acc0 = eng.download()
    # the fast walk opens at least what the strict one opens per group: their
    # difference is within the tree's own error at this tolerance
    assert np.abs(phi / phi0 - 1).max() < 2e-2


# (a mean of 4096 bodies is the line between the two widths of a system's block)
@pytest.mark.parametrize("sizes", [(1, 2, 255, 2047, 2048, 2049, 300), (8191, 8192, 8193, 20000, 1, 64, 5000)])
def test_systems_of_a_batch_get_the_box_of_their_own(eng, sizes):
    off = np.concatenate([[0], np.cumsum(sizes)])
    parts = [bodies(k, "spread") for k in sizes]
    for _, q in parts:          # grows the box late, to 2^7 (a batch has a level less: far from its depth)
        for j, i in enumerate(range(len(q) - 1, len(q) // 2, -max(1, len(q) // 8))):
            q[i] *= 2.0 ** (5 - j)
    m, x = np.concatenate([q[0] for q in parts]), np.concatenate([q[1] for q in parts])
    eng.batch_upload(off, m, x, np.full(len(sizes), 0.05), np.full(len(sizes), 0.8))
    eng.eval(E.default_params())
    phi, acc = eng.download()
    for k, (ms, xs) in enumerate(parts):
        if len(ms) < 3:
            continue
        eng.upload(ms, xs)
        eng.eval(E.default_params(eps=0.05, tol=0.8))
        p1, a1 = eng.download()
        a, b = off[k], off[k + 1]
        assert np.array_equal(phi[a:b], p1) and np.array_equal(acc[a:b], a1)
