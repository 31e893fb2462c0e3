"""The adjoint's and the 1/N expansion's self-energy passes at the edges of
their forms: compiled whole rows, planes and lines, whole rows and three passes
on both sides of their change in number of rows (which is N_mem - 1, whatever
the steps taken), run-time plans of every class, batches past 64.  The adjoint
against the numpy reverse-mode twin, the 1/N run against the oracle, both in
short windows of their own: nothing is dropped in so few steps, so the results
do not depend on N_mem (tolerance 1e-10, norm-wise relative)."""
import numpy as np
import pytest

from oracle.kb_numpy import kL2_table
from oracle.oracle import Oracle
from tests.adjoint_twin import gradient

pytestmark = pytest.mark.gpu

TOL = 1e-10
T = 6

# (Nx, sdim, N_mem of the device's run)
FORMS = [(n, 3, 8) for n in (9, 10, 13, 15, 16, 17, 19, 20, 21, 22, 23)]   # whole rows
FORMS += [(24, 3, 8), (24, 3, 97), (25, 3, 8), (25, 3, 41), (26, 3, 8), (26, 3, 41)]  # three passes, whole rows
FORMS += [(n, 3, 8) for n in (27, 28, 29, 34, 35, 39)]   # three run-time passes: small, any, wide
FORMS += [(n, 2, 8) for n in (24, 31, 34, 45, 56, 61, 69, 87)]   # planes; batches past 64
FORMS += [(n, 1, 8) for n in (32, 33, 46, 128, 300)]


def rel(a, b):
    d, s = np.max(np.abs(np.asarray(a) - np.asarray(b))), np.max(np.abs(np.asarray(b)))
    return d / s if s > 0 else d


def thermal(k2):
    return 1.0 / (np.exp(np.sqrt(k2 + 1.0) / 2.0) - 1.0)


@pytest.mark.parametrize("Nx,sdim,N", FORMS)
def test_adjoint_forms(Nx, sdim, N):
    from qftkb import KBContext
    print(f"\n[case] adjoint {Nx}^{sdim} N_mem={N}", flush=True)
    k2 = kL2_table(Nx, sdim)
    n0, wgt = thermal(k2), np.exp(-k2)
    g = KBContext(Nx, sdim, N, 0.1, 1.3, 1, 1.0, 1.0)
    g.init_particles(n0, 1.0)
    g.adj_record(0, max_steps=T)
    for t in range(3, T + 1):
        g.step(t)
    got = g.adj_gradient(wgt, n0=True, F0=True)
    g.close()
    _, lam, dn0, dF0 = gradient((Nx, sdim, 8, 0.1, 1.3, 1, 1.0, 1.0), n0, 1.0, T, wgt)
    assert rel(got["lambda"], lam) <= TOL
    assert rel(got["n0"], dn0) <= TOL
    for k in range(3):
        assert rel(got["F0"][k], dF0[k]) <= TOL, k


@pytest.mark.parametrize("Nx,sdim,N", FORMS)
def test_ninverse_forms(Nx, sdim, N):
    from qftkb import KBContext
    print(f"\n[case] 1/N {Nx}^{sdim} N_mem={N}", flush=True)
    g = KBContext(Nx, sdim, N, 0.05, 10.0, 8, 1.0, 1.0, pexp=3)
    o = Oracle(Nx, sdim, 8, 0.05, 10.0, 8, 1.0, 1.0, pexp=3)
    n = thermal(o.kL2())
    for c in (o, g):
        c.init_particles(n, 1.0)
    for t in range(3, T + 1):
        o.evolve(t)
        g.step(t)
    scale = max(np.max(np.abs(o.sigma(w, tp))) for w in "Fr" for tp in range(1, T))
    for tp in range(1, T):
        for w in "Fr":
            assert np.max(np.abs(g.sigma(w, tp) - o.sigma(w, tp))) <= TOL * scale, (w, tp)
            assert rel(g.get(w, T, tp), o.get(w, T, tp)) <= TOL, (w, tp)
    assert rel(g.get("F", T, T), o.get("F", T, T)) <= TOL
    g.close()
    o.close()
