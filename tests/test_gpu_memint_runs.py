"""The default shape's equal-run memory integral at the edges of its forms
(one, two, four and eight waves per site block, split over workgroups, the
window limits of each) against the oracle, through wrapped rings and filling
windows (tolerance 1e-10, norm-wise relative)."""
import numpy as np
import pytest

from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

RTOL = 1e-10


def rel(a, b):
    d = np.max(np.abs(np.asarray(a) - np.asarray(b)))
    s = np.max(np.abs(np.asarray(b)))
    return d / s if s > 0 else d


def same_rows(g, o, t, tps):
    for w in "Fr":
        for tp in tps:
            assert rel(g.get(w, t, tp), o.get(w, t, tp)) <= RTOL, (w, t, tp)


# (Nx, sdim, N_mem, orbit storage, window end the run starts from; 0: from the initial rows)
CASES = [
    (6, 3, 3, False, 7), (6, 3, 4, False, 9), (6, 3, 5, False, 5), (6, 3, 23, False, 0),  # four waves per block
    (26, 3, 5, False, 8), (26, 3, 32, False, 45), (26, 3, 32, False, 0),  # one wave
    (26, 3, 33, False, 66), (26, 3, 33, False, 0),  # two waves
    (15, 3, 130, False, 131),  # eight waves
    (8, 2, 47, False, 60), (8, 2, 48, False, 61), (5, 2, 100, False, 0),  # split from 48
    (16, 1, 208, False, 250), (16, 1, 400, False, 777), (9, 1, 600, False, 700), (9, 1, 601, False, 700),
    (12, 3, 60, True, 63), (12, 3, 20, True, 0), (33, 3, 100, True, 120),  # orbit storage: split, whole
    (300, 1, 209, False, 230),  # past the whole-block form
]


@pytest.mark.parametrize("Nx,sdim,N,sym,tmax", CASES)
def test_equal_runs_match_oracle(Nx, sdim, N, sym, tmax):
    from qftkb import KBContext
    print(f"\n[case] {Nx}^{sdim} N_mem={N} orbits={sym} from {tmax}", flush=True)
    args = (Nx, sdim, N, 0.1, 1.3, 1, 1.0, 1.0)
    o, g = Oracle(*args), KBContext(*args, tiles=None, symmetric=sym)
    n = 1.0 / (np.exp(np.sqrt(o.kL2() + 1.0) / 2.0) - 1.0)
    if tmax:
        o.fill_free_window(tmax, n, 1.0)
        g.fill_free_window(tmax, n, 1.0)
        last = tmax + 3
    else:
        o.init_particles(n, 1.0)
        g.init_particles(n, 1.0)
        tmax, last = 2, min(N + 5, 40)
    for t in range(tmax + 1, last + 1):
        o.evolve(t)
        g.step(t)
        tmin = g.window()[0]
        tps = sorted({tmin, tmin + 1, (tmin + t) // 2, t - 3, t - 2, t - 1, t} & set(range(tmin, t + 1)))
        same_rows(g, o, t, tps if Nx ** sdim > 2000 or N > 64 else range(tmin, t + 1))
    g.close()
    o.close()
