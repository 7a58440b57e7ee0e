"""The walk by a team of waves per group (few groups) gives the one-wave walk's
results bit for bit.  A system evaluated alone has few groups and is walked by
teams (a row of a group, or a whole group, per 8 waves; a group per 4 waves);
in a batch with enough other bodies the same groups are walked one wave each,
and a batch's systems have the trees and groups of single runs."""
import numpy as np
import pytest

from nemo_amd import engine as E
from oracle import oracle

pytestmark = pytest.mark.gpu

# sizes: one group, group edges, a row per team, 8 waves and 4 waves per group
SIZES = [2, 63, 65, 129, 500, 3001, 20011, 60013, 150001]


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def systems():
    parts = [E.mkplummer(n, 5 + n, with_vel=False) for n in SIZES + [1 << 20]]
    off = np.concatenate([[0], np.cumsum([len(p[0]) for p in parts])]).astype(np.int64)
    return parts, off, np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])


@pytest.mark.parametrize("group", [64, 128, 192, 256])
@pytest.mark.parametrize("quad,eps,alpha", [(0, 0.03, 0.0), (1, 0.03, 0.0), (0, 0.0, 0.0), (1, 0.0, 0.0), (0, 0.03, 0.2),
                                            (0, 0.0, 0.35)])
def test_team_equals_one_wave(eng, systems, group, quad, eps, alpha):
    parts, off, m, x = systems
    tol = np.linspace(0.6, 0.9, len(parts))
    kw = dict(usequad=quad, group_size=group, nleaf=1, local_alpha=alpha)
    eng.batch_upload(off, m, x, np.full(len(parts), eps), tol)
    eng.eval(E.default_params(**kw))
    phi, acc = eng.download()
    for s, n in enumerate(SIZES):
        p, a, st = eng.force(parts[s][0], parts[s][1], E.default_params(tol=tol[s], eps=eps, **kw))
        assert np.array_equal(phi[off[s]:off[s + 1]], p), n
        assert np.array_equal(acc[off[s]:off[s + 1]], a), n


@pytest.mark.parametrize("criterion", ["hack", "rcrit", "sw94"])
@pytest.mark.parametrize("n,nt", [(9000, 3001), (30011, 200003), (9000, 0)])
def test_team_points_massless_and_criteria(eng, criterion, n, nt):
    """Separate points, massless bodies and treecode1's criteria in each
    regime: at least the strict walk's interactions, its accuracy, and with
    tol = 0 all pairs."""
    r = np.random.default_rng(n + nt)
    m, x, _ = E.mkplummer(n, 11, with_vel=False)
    m[::7] = 0.0
    tp = r.normal(size=(nt, 3)) if nt else None
    kw = dict(tol=0.8, eps=0.02, criterion=criterion, usequad=1)
    phi, acc, st = eng.force(m, x, E.default_params(**kw), tpos=tp)
    sphi, sacc, ss = eng.force(m, x, E.default_params(mode="strict", **kw), tpos=tp)
    assert st.n2btot + st.nbctot > 0 and st.n2btot >= ss.n2btot
    e = np.linalg.norm(acc - sacc, axis=1) / np.linalg.norm(sacc, axis=1)
    assert np.median(e) < 5e-3
    if criterion == "hack" and nt < 10000:
        p0, a0, s0 = eng.force(m, x, E.default_params(tol=0.0, eps=0.02), tpos=tp)
        k = int((m != 0).sum())
        assert s0.nbctot == 0 and s0.n2btot == ((nt * k) if nt else n * k - k)
        if nt == 0:
            idx = np.arange(0, n, 97)
            _, da = oracle.direct(m, x, 0.02, idx)
            assert np.abs(a0[idx] - da).max() < 1e-5 * np.abs(da).max()
