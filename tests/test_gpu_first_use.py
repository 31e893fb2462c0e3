"""The code of the self-energy passes is loaded by the first context that runs
them, mode by mode: a process's first context does not pay for the others'."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import time
from qftkb import KBContext

def create(pexp, Nx=8):
    t = time.perf_counter()
    c = KBContext(Nx, 3, 4, 0.1, 1.0, 1, 1.0, 1.0, pexp=pexp)
    t = time.perf_counter() - t
    c.close()
    return t

create(0)
create(0)
for pexp in (1, 3):
    first = create(pexp)
    print(pexp, first, min(create(pexp) for _ in range(8)))
first = create(1, 31)
print("31^3", first, min(create(1, 31) for _ in range(8)))
"""


def test_passes_are_loaded_when_first_used():
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "qftdynamicsm.jl_amd"))
    out = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    rows = [line.split() for line in out.stdout.splitlines()]
    assert len(rows) == 3
    for what, first, later in rows:
        print(f"\n[case] {what}: first create {1e3 * float(first):.2f} ms, later {1e3 * float(later):.2f}", flush=True)
        # (code that an earlier context had loaded: level)
        assert float(first) > 2 * float(later), what
