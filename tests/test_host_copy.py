"""The threaded way of large results to the caller (csrc/kb_hostcopy.h), built
for the host: every value arrives for lengths around the pieces' edges, an
error of the fetch ends the copy, and nothing is thrown where memory or threads
run out (it runs below C entry points)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qftdynamicsm.jl_amd", "csrc")

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>
#include "kb_hostcopy.h"

static std::atomic<long> allowed{-1};  // allocations until they fail; < 0: never
void* operator new(std::size_t n) {
  if (allowed.load() >= 0 && allowed.fetch_sub(1) <= 0) {
    allowed.store(0);
    throw std::bad_alloc();
  }
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

// one copy; fail_at: the fetch that fails (< 0: none); news: allocations allowed
int run(int narr, size_t n, size_t half, int fail_at, long news) {
  std::vector<std::vector<double>> src(narr), dst(narr);
  std::vector<const double*> s(narr);
  std::vector<double*> d(narr);
  for (int k = 0; k < narr; ++k) {
    src[k].resize(n);
    dst[k].assign(n + 1, -1.0);
    for (size_t i = 0; i < n; ++i) src[k][i] = 1e6 * k + i;
    s[k] = src[k].data();
    d[k] = dst[k].data();
  }
  std::vector<double> stage(2 * half);
  int fetches = 0;
  allowed.store(news);
  const int err = qftkb_host::copy_out(narr, d.data(), s.data(), n, stage.data(), half,
                                       [&](double* to, const double* from, size_t count) -> int {
                                         if (fetches++ == fail_at) return 7;
                                         std::memcpy(to, from, count * sizeof(double));
                                         return 0;
                                       });
  allowed.store(-1);
  if (fail_at >= 0) return err == 7 && fetches == fail_at + 1 ? 0 : 1;
  if (err) return 2;
  for (int k = 0; k < narr; ++k) {
    if (std::memcmp(d[k], s[k], n * sizeof(double))) return 3;
    if (dst[k][n] != -1.0) return 4;
  }
  return 0;
}

int main() {
  for (int narr : {1, 2, 6})
    for (size_t half : {1, 7, 64, 1000})
      for (size_t n : {half - 1, half, half + 1, 2 * half, 3 * half + 1, 5 * half - 1})
        for (long news : {-1L, 0L, 1L, 3L})
          if (int e = run(narr, n, half, -1, news)) {
            std::printf("narr %d half %zu n %zu allocations %ld: %d\\n", narr, half, n, news, e);
            return 1;
          }
  for (int at : {0, 1, 2, 5})
    for (long news : {-1L, 0L, 2L})
      if (int e = run(2, 3 * 64 + 1, 64, at, news)) {
        std::printf("error at fetch %d, allocations %ld: %d\\n", at, news, e);
        return 1;
      }
  return 0;
}
"""


def test_copy_out(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr[-2000:]
