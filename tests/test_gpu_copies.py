"""Host arrays on both sides of the lines between staged and direct copies (512
KB an array, 2 MB together), pageable and page-locked: one force call gives the
same bits as upload, evaluation and download of the other kind, and a state
read back is the one that was given."""
import numpy as np
import pytest
import torch

from nemo_amd import engine as E

pytestmark = pytest.mark.gpu


def locked(a):
    return torch.from_numpy(np.ascontiguousarray(a)).pin_memory()


# 512 KB: 65536 doubles, 21845 positions
@pytest.mark.parametrize("n,nt", [(1, 0), (31, 7), (21845, 0), (21846, 0), (21846, 21845), (65536, 65536), (65537, 20000), (70000, 1)])
def test_force_call_equals_its_parts(n, nt):
    r = np.random.default_rng(n + nt)
    m, x = r.uniform(0.5, 1.5, n) / n, r.normal(size=(n, 3))
    t = r.normal(size=(nt, 3)) if nt else None
    p = E.default_params(tol=0.9, eps=0.05, mode="strict" if n < 3 else "fast")
    a, b = E.Engine(0), E.Engine(0)
    try:
        phi, acc, _ = a.force(m, x, p, tpos=t)
        phi2, acc2, _ = a.force(m, x, p, tpos=t)          # the staging memory again
        lm, lx, lt = locked(m), locked(x), None if t is None else locked(t)
        b.upload(lm.numpy(), lx.numpy(), tpos=None if lt is None else lt.numpy())
        b.eval(p)
        phi3, acc3 = b.download()
        for u, w in ((phi, acc), (phi2, acc2)):
            assert np.array_equal(u, phi3) and np.array_equal(w, acc3)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("n", [5, 21845, 21846, 70000])
def test_leapfrog_state_goes_there_and_back(n):
    r = np.random.default_rng(n)
    m, x, v = r.uniform(0.5, 1.5, n) / n, r.normal(size=(n, 3)), r.normal(size=(n, 3))
    e = E.Engine(0)
    try:
        lf = E.Leapfrog(e, m, x, v, 1.0 / 64.0, tol=1.0, eps=0.05)
        pos, vel, _, _, _ = lf.state()
        assert np.array_equal(pos, x) and np.array_equal(vel, v)
    finally:
        e.close()
