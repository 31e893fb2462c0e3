"""The equal-run memory integral of whole site blocks at the limits of its
forms (site blocks enough that none is split: eight waves per block and four
from 512 blocks on, two from 2048 on up to N_mem = 152 where their rounds fill
the chip, the longest window of 208, the item form where the
last round would be nearly empty), for one run and for an ensemble's table, against the item form
of the same integrals (shape 1, tested against the oracle), through a wrapped
ring; tolerance 1e-10, norm-wise relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-10
ITEMS = 1


def rel(a, b):
    d, s = np.max(np.abs(a - b)), np.max(np.abs(b))
    return d / s if s > 0 else d


def same_row(a, b, t):
    tmin = b.window()[0]
    for tp in sorted({tmin, tmin + 1, (tmin + t) // 2, t - 3, t - 2, t - 1, t}):
        for w in "Fr":
            assert rel(a.get(w, t, tp), b.get(w, t, tp)) <= RTOL, (w, t, tp)


# 422 site blocks: eight waves from N_mem = 128 to 208; 512: four; 1000: four, items
# from 153 on; 2197: four at 64 (two at 112); 2744: two at 128 and 152
@pytest.mark.parametrize("Nx,N", [(15, 127), (15, 128), (15, 208), (15, 209), (16, 202), (16, 208), (20, 152),
                                  (20, 153), (26, 64), (26, 112), (26, 192), (26, 193), (28, 128), (28, 152), (28, 153)])
def test_whole_blocks_match_items(Nx, N):
    from qftkb import KBContext
    print(f"\n[case] whole blocks {Nx}^3 N_mem={N}", flush=True)
    pair = [KBContext(Nx, 3, N, 0.1, 1.3, 1, 1.0, 1.0, tiles=s) for s in (None, ITEMS)]
    n = 1.0 / (np.exp(np.sqrt(pair[0].kL2() + 1.0) / 2.0) - 1.0)
    t = N + N // 3
    for c in pair:
        c.fill_free_window(t, n, 1.0)
    for t in range(t + 1, t + 4):
        for c in pair:
            c.step(t)
        same_row(*pair, t)
    for c in pair:
        c.close()


# 3000 site blocks: one wave up to N_mem = 32, two at 33, 64 and 112; 2729: four past
# 152; 895: four, items from 153 on; 281: eight past 127
@pytest.mark.parametrize("sizes,N", [((20, 20, 20), 24), ((20, 20, 20), 33), ((20, 20, 20), 64),
                                     ((20, 20, 20), 112), ((16, 12, 11), 64), ((16, 12, 11), 130), ((16, 12, 11), 160), ((9, 8, 10), 130), ((20, 18, 20), 153),
                                     ((20, 18, 20), 193)])
def test_tables_match_items(sizes, N):
    from qftkb import KBContext, KBEnsemble
    print(f"\n[case] ensemble {sizes} N_mem={N}", flush=True)
    args = [dict(Nx=n, sdim=3, NstepsinMemory=N, dt=0.1, Lambda=1.3, ONgroup=1, Mass=1.0, Mass2=1.0) for n in sizes]
    e = KBEnsemble(args)
    alone = [KBContext(**a, tiles=ITEMS) for a in args]
    t = N + N // 3
    for m, c in zip(e.members, alone):
        n = 1.0 / (np.exp(np.sqrt(c.kL2() + 1.0) / 2.0) - 1.0)
        m.fill_free_window(t, n, 1.0)
        c.fill_free_window(t, n, 1.0)
    for t in range(t + 1, t + 4):
        e.step(t)
        for m, c in zip(e.members, alone):
            c.step(t)
            same_row(m, c, t)
    e.close()
    for c in alone:
        c.close()
