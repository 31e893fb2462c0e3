"""The compile-time twiddle table (csrc/kb_twiddles.h), built for the host: its
pairs are read as 16-byte values on the device, so it is aligned to 16 bytes;
every value is exp(-2 pi i k / n), from 60-digit series, correctly rounded, and
the quarter turns are exact."""
import os
import subprocess
from decimal import Decimal, getcontext

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qftdynamicsm.jl_amd", "csrc")

PROGRAM = """
#include <cstdio>
#include "kb_twiddles.h"
using namespace qftkb;
static constexpr TwiddleTable t = make_twiddles();
int main() {
  std::printf("%zu %d\\n", alignof(TwiddleTable), TWIDDLE_MAX);
  for (int n = 1; n <= TWIDDLE_MAX; ++n)
    for (int k = 0; k < n; ++k)
      std::printf("%a %a\\n", t.v[2 * (twiddle_start(n) + k)], t.v[2 * (twiddle_start(n) + k) + 1]);
}
"""


def cos_sin(k, n):
    """cos and sin of 2 pi k / n to some 55 digits (Machin's formula, Taylor series)."""
    getcontext().prec = 60

    def arctan_inverse(x):
        total, term, j = Decimal(0), Decimal(1) / x, 0
        while abs(term) > Decimal(10) ** -58:
            total += term / (2 * j + 1) if j % 2 == 0 else -term / (2 * j + 1)
            term /= x * x
            j += 1
        return total

    a = 2 * (16 * arctan_inverse(5) - 4 * arctan_inverse(239)) * k / n
    out = []
    for j in (0, 1):
        total, term = Decimal(0), a ** j if j else Decimal(1)
        while abs(term) > Decimal(10) ** -58 or j < a:
            total += term
            term *= -a * a / ((j + 1) * (j + 2))
            j += 2
        out.append(total)
    return out


def test_table_is_aligned_and_rounded(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fconstexpr-ops-limit=200000000", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    align, top = map(int, lines[0].split())
    assert align % 16 == 0
    v = np.array([[float.fromhex(x) for x in line.split()] for line in lines[1:] if line])
    assert len(v) == top * (top + 1) // 2
    at = 0
    for n in range(1, top + 1):
        for k in range(n):
            c, s = cos_sin(k, n)
            want = (float(c), -float(s)) if 4 * k % n else [(1, 0), (0, -1), (-1, 0), (0, 1)][4 * k // n]
            assert tuple(v[at + k]) == want, (n, k)
        at += n
