"""The self-energy transforms at the edges of their forms, on random rows that
are not even under reflection, against numpy's FFT: lines, planes and whole
rows in LDS, three passes, batches past Nx = 64, compiled lengths and run-time
plans with every radix and with prime stages; the 1/N passes and the adjoint's
use the same passes (tolerance 1e-12 of the largest value: some 10 log2(V)
roundings of 1.1e-16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def rel(a, b):  # (absolute where the reference is exactly zero: rho(t, t))
    d, s = np.max(np.abs(a - b)), np.max(np.abs(b))
    return d / s if s > 0 else d


def sunset(F, r, lam, ON):
    ax = tuple(range(1, F.ndim))
    ivol = 1.0 / np.prod(F.shape[1:])
    Fx, rx = np.fft.fftn(F, axes=ax).real, np.fft.fftn(r, axes=ax).real
    pre = -lam ** 2 * (ON + 2) / ON ** 2 * ivol ** 3
    SF = pre / 18.0 * np.fft.fftn(Fx * (Fx ** 2 - 0.75 * rx ** 2), axes=ax).real
    SR = pre / 6.0 * np.fft.fftn(rx * (Fx ** 2 - rx ** 2 / 12.0), axes=ax).real
    return SF, SR


# (Nx, sdim, rows)
FORMS = [(n, 1, 3) for n in (1, 2, 3, 8, 9, 11, 13, 17, 32, 47, 60, 64)]
FORMS += [(n, 2, 3) for n in (1, 2, 5, 8, 13, 17, 26, 32, 45, 56, 61, 63, 64)]
FORMS += [(n, 3, 3) for n in (1, 2, 3, 8, 9, 10, 11, 13, 15, 16, 17, 19, 22, 23, 24, 25, 26, 27, 29, 32, 34, 39, 40,
                                46, 47, 57)]
FORMS += [(24, 3, 95), (24, 3, 96), (16, 3, 600), (49, 3, 2), (56, 3, 2), (63, 3, 1), (64, 3, 1)]


@pytest.mark.parametrize("Nx,sdim,rows", FORMS)
def test_sunset_forms(Nx, sdim, rows):
    from hipmem import DeviceArray
    from qftkb._abi import sunset as device_sunset, sunset_workspace_bytes
    print(f"\n[case] sunset {Nx}^{sdim} x {rows}", flush=True)
    V, lam, ON = Nx ** sdim, 1.7, 3
    rng = np.random.default_rng(Nx + 100 * sdim + rows)
    F, r = rng.standard_normal((2, rows) + (Nx,) * sdim)
    SF, SR = DeviceArray(rows * V), DeviceArray(rows * V)
    nb = sunset_workspace_bytes(Nx, sdim, rows)
    ws = DeviceArray(nb, np.uint8)
    dF, dr = DeviceArray.from_host(F.reshape(rows, V)), DeviceArray.from_host(r.reshape(rows, V))
    device_sunset(Nx, sdim, lam, ON, rows, dF.ptr, dr.ptr, SF.ptr, SR.ptr, ws.ptr, nb)
    for got, want in zip((SF.host(), SR.host()), sunset(F, r, lam, ON)):
        got = got.reshape(want.shape)
        for q in range(rows):
            assert rel(got[q], want[q]) <= RTOL, q


# past Nx = 64 (no kb_sunset there): the stage of a step, against the transforms
# of the rows it read
@pytest.mark.parametrize("Nx,sdim", [(100, 1), (128, 1), (251, 1), (500, 1), (1024, 1), (2000, 1),
                                     (65, 2), (66, 2), (69, 2), (87, 2), (97, 2), (131, 2), (256, 2),
                                     (65, 3), (67, 3), (72, 3), (76, 3), (99, 3)])
def test_batched_passes(Nx, sdim):
    from qftkb import KBContext
    print(f"\n[case] stage {Nx}^{sdim}", flush=True)
    N, t = 3, 5
    g = KBContext(Nx, sdim, N, 0.1, 1.3, 2, 1.0, 1.0, tiles=None)
    rng = np.random.default_rng(Nx + sdim)
    g.fill_free_window(t, rng.uniform(0.1, 2.0, Nx ** sdim), 1.0)
    g.step(t + 1)
    tps = range(g.window()[0], t + 1)
    shape = (len(tps),) + (Nx,) * sdim
    F = np.array([g.get("F", t, tp) for tp in tps]).reshape(shape)
    r = np.array([g.get("r", t, tp) for tp in tps]).reshape(shape)
    got = [np.array([g.sigma(w, tp) for tp in tps]).reshape(shape) for w in "Fr"]
    for a, b in zip(got, sunset(F, r, 1.3, 2)):
        for q in range(len(tps)):
            assert rel(a[q], b[q]) <= RTOL, tps[q]
    g.close()
