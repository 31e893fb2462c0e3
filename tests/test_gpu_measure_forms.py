"""kb_measure's forms (workers per site block by window length, lattices
written straight to host memory, expanded from orbits, or copied out in
pieces by several threads) against the oracle, 1e-10 norm-wise relative."""
import numpy as np
import pytest

from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

RTOL = 1e-10
CASES = [(6, 3, 3, False), (6, 3, 5, False), (5, 2, 17, False), (9, 1, 130, False), (24, 3, 4, False),
         (57, 3, 3, False), (12, 3, 9, True), (57, 3, 3, True)]  # 6 lattices of 57^3: past the pinned buffer


def rel(a, b):
    d = np.max(np.abs(np.asarray(a) - np.asarray(b)))
    s = np.max(np.abs(np.asarray(b)))
    return d / s if s > 0 else d


@pytest.mark.parametrize("Nx,sdim,N,sym", CASES)
def test_measurement_matches_oracle(Nx, sdim, N, sym):
    from qftkb import KBContext
    print(f"\n[case] measure {Nx}^{sdim} N_mem={N} orbits={sym}", flush=True)
    args = (Nx, sdim, N, 0.1, 1.3, 1, 1.0, 1.0)
    o, g = Oracle(*args), KBContext(*args, symmetric=sym)
    n = 1.0 / (np.exp(np.sqrt(o.kL2() + 1.0) / 2.0) - 1.0)
    for c in (o, g):
        c.fill_free_window(N + 2, n, 1.0)
    t = N + 3
    o.evolve(t)
    g.step(t)
    a, b = g.measure(t), o.measure(t)
    for k in ("E", "E_kin", "E_pot", "E_mem", "M2", "time", "F", "ddF", "r", "n", "omega", "c"):
        assert rel(a[k], b[k]) <= RTOL, k
    assert a["n_unstable"] == b["nstab"]
    assert g.measure(t, modes=False)["E"] == a["E"]
    assert rel(g.get("F", t, t - 1), o.get("F", t, t - 1)) <= RTOL
    h = g.measure_history(t)
    for q, tp in enumerate(range(t - 1, g.window()[0] - 1, -1)):
        assert abs(h["SigF"][q] - o.sigma("F", tp)[0]) <= RTOL * np.max(np.abs(o.sigma("F", tp)))
    g.close()
    o.close()
