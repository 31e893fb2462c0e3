"""Lines with a prime stage, one per workgroup: a step's stage, the adjoint and
the 1/N passes through lengths with one prime factor above 23, alone and with
others (the stage against numpy's FFT, 1e-12 of the largest value: sums of up to
2039 terms and three transforms, some 1e-14; the adjoint against its twin and the
1/N run against the oracle, 1e-10), and the time of 300 lines of 61 points."""
import time

import numpy as np
import pytest

from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    d, s = np.max(np.abs(np.asarray(a) - np.asarray(b))), np.max(np.abs(np.asarray(b)))
    return d / s if s > 0 else d


@pytest.mark.parametrize("Nx", [29, 31, 58, 61, 62, 127, 131, 899, 1021, 2038, 2039])
def test_stage_of_prime_lines(Nx):
    from qftkb import KBContext
    print(f"\n[case] stage {Nx}^1", flush=True)
    N, t = 4, 6
    g = KBContext(Nx, 1, N, 0.1, 1.3, 2, 1.0, 1.0, tiles=None)
    g.fill_free_window(t, np.random.default_rng(Nx).uniform(0.1, 2.0, Nx), 1.0)
    g.step(t + 1)
    pre = -1.3 ** 2 * 4.0 / 4.0 / Nx ** 3
    for tp in range(g.window()[0], t + 1):
        Fx, rx = (np.fft.fft(g.get(w, t, tp)).real for w in "Fr")
        assert rel(g.sigma("F", tp), pre / 18.0 * np.fft.fft(Fx * (Fx ** 2 - 0.75 * rx ** 2)).real) <= 1e-12, tp
        assert rel(g.sigma("r", tp), pre / 6.0 * np.fft.fft(rx * (Fx ** 2 - rx ** 2 / 12.0)).real) <= 1e-12, tp
    g.close()


@pytest.mark.parametrize("Nx", [29, 58, 61])
def test_adjoint_of_prime_lines(Nx):
    from qftkb import KBContext
    from tests.adjoint_twin import gradient
    print(f"\n[case] adjoint {Nx}^1", flush=True)
    args, T = (Nx, 1, 5, 0.1, 1.0, 1, 1.0, 1.0), 9
    g = KBContext(*args)
    k2 = g.kL2()
    n0, wgt = 1.0 / (np.exp(np.sqrt(k2 + 1.0) / 2.0) - 1.0), np.exp(-k2)
    g.init_particles(n0, 1.0)
    g.adj_record(0, max_steps=T)
    for t in range(3, T + 1):
        g.step(t)
    got = g.adj_gradient(wgt, n0=True, F0=True)
    g.close()
    _, dlam, dn0, dF = gradient(args, n0, 1.0, T, wgt)
    assert rel(got["lambda"], dlam) <= 1e-10
    assert rel(got["n0"], dn0) <= 1e-10
    for x, y in zip(got["F0"], dF):
        assert rel(x, y) <= 1e-10


@pytest.mark.parametrize("Nx", [31, 58, 61])
def test_ninverse_of_prime_lines(Nx):
    from qftkb import KBContext
    print(f"\n[case] 1/N {Nx}^1", flush=True)
    args = (Nx, 1, 5, 0.1, 1.2, 4, 1.0, 1.0)
    o, g = Oracle(*args, pexp=3), KBContext(*args, pexp=3)
    n = 1.0 / (np.exp(np.sqrt(o.kL2() + 1.0) / 2.0) - 1.0)
    for c in (o, g):
        c.init_particles(n, 1.0)
    for t in range(3, 10):
        o.evolve(t)
        g.step(t)
        for tp in range(g.window()[0], t + 1):
            for w in "Fr":
                assert rel(g.get(w, t, tp), o.get(w, t, tp)) <= 1e-10, (w, t, tp)
    g.close()
    o.close()


def test_prime_lines_take_less_than_three_times_a_line_of_64():
    from hipmem import DeviceArray, synchronize
    from qftkb._abi import sunset, sunset_workspace_bytes
    best = []
    for Nx in (61, 64):
        F, r = (DeviceArray.from_host(x) for x in np.random.default_rng(1).standard_normal((2, 300 * Nx)))
        a, b = (DeviceArray(300 * Nx) for _ in range(2))
        nb = sunset_workspace_bytes(Nx, 1, 300)
        ws = DeviceArray(nb, np.uint8)
        times = []
        for _ in range(12):
            synchronize()
            t = time.perf_counter()
            for _ in range(200):
                sunset(Nx, 1, 1.0, 1, 300, F.ptr, r.ptr, a.ptr, b.ptr, ws.ptr, nb)
            synchronize()
            times.append(time.perf_counter() - t)
        best.append(min(times))
    print(f"\n[case] 300 lines of 61 over 300 of 64: {best[0] / best[1]:.2f}", flush=True)
    assert best[0] <= 3.0 * best[1]  # (four pairs to an item: 5.6)
