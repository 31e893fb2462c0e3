"""A row of kb_sunset has the bits of a step's self-energy stage, whatever form
the two take: lines, planes, whole rows, three passes, compiled lengths and
run-time plans, few rows and many (24^3 changes form with the number of rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (Nx, sdim, N_mem, numbers of rows)
CASES = [(n, 1, 4, (1, 3)) for n in (1, 2, 8, 9, 31, 47, 61, 64)]
CASES += [(n, 2, 4, (1, 3)) for n in (2, 5, 8, 17, 24, 31, 45, 64)]
CASES += [(n, 3, 4, (1, 3)) for n in (2, 8, 9, 13, 16, 17, 23, 24, 25, 26, 27, 29, 32, 34, 45, 48, 61)]
CASES += [(24, 3, 98, (1, 95, 96, 97)), (25, 3, 61, (1, 39, 40, 60)), (26, 3, 61, (1, 39, 40, 60)),
          (24, 3, 20, (1, 19)), (25, 3, 20, (1, 19)), (26, 3, 20, (1, 19))]


@pytest.mark.parametrize("classical", [False, True])
@pytest.mark.parametrize("Nx,sdim,N,counts", CASES)
def test_same_bits_as_the_step(Nx, sdim, N, counts, classical):
    from hipmem import DeviceArray
    from qftkb import KBContext
    from qftkb._abi import sunset, sunset_workspace_bytes
    print(f"\n[case] bits {Nx}^{sdim} N_mem={N} classical={classical}", flush=True)
    V = Nx ** sdim
    g = KBContext(Nx, sdim, N, 0.1, 1.3, 2, 1.0, 1.0, pexp=4 if classical else 1, tiles=None)
    g.fill_free_window(N + 1, np.random.default_rng(Nx + sdim).uniform(0.1, 2.0, V), 1.0)
    t = N + 2
    g.step(t)
    tps = range(g.window()[0], t)
    F, r = (np.array([g.get(w, t - 1, tp) for tp in tps]) for w in "Fr")
    want = [np.array([g.sigma(w, tp) for tp in tps]) for w in "Fr"]
    g.close()
    # (the step took N - 1 rows)
    for rows in counts:
        rows = min(rows, len(tps))
        dF, dr = DeviceArray.from_host(F[:rows]), DeviceArray.from_host(r[:rows])
        out = [DeviceArray(rows * V) for _ in range(2)]
        nb = sunset_workspace_bytes(Nx, sdim, rows)
        ws = DeviceArray(nb, np.uint8)
        sunset(Nx, sdim, 1.3, 2, rows, dF.ptr, dr.ptr, out[0].ptr, out[1].ptr, ws.ptr, nb, classical=classical)
        for a, b in zip(out, want):
            assert np.array_equal(a.host().reshape(rows, V), b[:rows]), rows
