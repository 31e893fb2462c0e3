"""What a context or an ensemble takes on the device comes back when it is
destroyed: free device memory after each of several rounds of creating,
using and destroying every kind of one equals that after the first."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BASE = dict(dt=0.1, Lambda=1.0, Mass=1.0, Mass2=1.0)


def free_bytes():
    from hipmem import hip, synchronize
    synchronize()
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


def one(kind):
    from qftkb import KBContext, KBEnsemble
    if kind == "ensemble":
        e = KBEnsemble([dict(Nx=n, sdim=3, NstepsinMemory=4, ONgroup=1, symmetric=s, **BASE)
                        for n, s in ((40, False), (33, False), (48, True))])
        for m in e.members:
            m.fill_free_window(4, np.ones(m.V), 1.0)
        e.step(5)
        e.close()
        return
    pexp, sym = {"full": (1, False), "lo": (0, False), "orbits": (1, True), "ninverse": (3, False),
                 "past the pinned buffer": (1, False), "adjoint": (1, False)}[kind]
    Nx = 64 if kind == "past the pinned buffer" else 40
    c = KBContext(Nx, 3, 4, ONgroup=1, pexp=pexp, symmetric=sym, **BASE)
    if kind == "adjoint":
        c.init_particles(np.ones(c.V), 1.0)
        c.adj_record(0, max_steps=6)
        for t in range(3, 7):
            c.step(t)
        c.adj_gradient(np.ones(c.V))
    else:
        c.fill_free_window(4, np.ones(c.V), 1.0)
        c.use_graph(True)
        for t in range(5, 8):
            c.step(t)
        c.measure(7)
    c.close()


@pytest.mark.parametrize("kind", ["full", "lo", "orbits", "ninverse", "past the pinned buffer", "adjoint",
                                  "ensemble"])
def test_destroy_returns_device_memory(kind):
    print(f"\n[case] create and destroy: {kind}", flush=True)
    one(kind)
    one(kind)  # (what the runtime and the code objects take on first use)
    before = free_bytes()
    for _ in range(6):
        one(kind)
    assert free_bytes() == before
