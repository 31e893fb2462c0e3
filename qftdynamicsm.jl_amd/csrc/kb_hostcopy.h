// kb_hostcopy.h -- large results on their way to the caller's memory: pieces
// are fetched into two halves of a staging buffer in turn, and written out by
// HOST_COPY_THREADS threads while the next one is fetched (the caller's fresh
// pages cost a single thread more time than the fetch).
//
// Plain C++ with nothing of the device: the fetch is the caller's.  It is
// called below C entry points, so nothing is thrown and nothing needs memory
// to succeed: where threads cannot be had, those that there are write, or the
// calling thread.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace qftkb_host {

constexpr int HOST_COPY_THREADS = 6;

// narr arrays of n doubles from src to dst through stage (two halves of `half`
// doubles).  fetch(to, from, count) returns when the piece is there, 0 or an
// error, which ends the copy and is returned.
template <class Fetch>
int copy_out(int narr, double* const* dst, const double* const* src, size_t n, double* stage, size_t half,
             Fetch fetch) {
  const size_t per = (n + half - 1) / half, np = per * narr;  // pieces of an array, and in all
  auto begin = [&](size_t p) { return p % per * half; };
  auto length = [&](size_t p) { return std::min(half, n - begin(p)); };
  // pieces handed out (STOP: no more), their threads, and the shares of the
  // last one that are not written yet
  constexpr size_t STOP = ~size_t(0);
  std::atomic<size_t> ready{0};
  std::atomic<int> workers{0}, left{0};
  auto share = [&](size_t p, int i, int of) {
    const size_t b = length(p) * i / of, e = length(p) * (i + 1) / of;
    std::memcpy(dst[p / per] + begin(p) + b, stage + (p & 1) * half + b, (e - b) * sizeof(double));
  };
  auto work = [&](int i) {
    for (size_t p = 0; p < np; ++p) {
      size_t r;
      while ((r = ready.load(std::memory_order_acquire)) <= p) std::this_thread::yield();
      if (r == STOP) return;
      share(p, i, workers.load(std::memory_order_relaxed));
      left.fetch_sub(1, std::memory_order_release);
    }
  };
  std::thread pool[HOST_COPY_THREADS];
  int nw = 0;
  try {
    for (; nw < HOST_COPY_THREADS; ++nw) pool[nw] = std::thread(work, nw);
  } catch (...) {
    // as many as there are
  }
  workers.store(nw, std::memory_order_relaxed);
  auto drain = [&] {
    while (left.load(std::memory_order_acquire) > 0) std::this_thread::yield();
  };
  int err = 0;
  for (size_t p = 0; p < np; ++p) {
    // into the half that piece p - 2 left: it was drained before piece p - 1
    // was handed out
    if ((err = fetch(stage + (p & 1) * half, src[p / per] + begin(p), length(p)))) break;
    drain();
    if (nw) {
      left.store(nw, std::memory_order_relaxed);
      ready.store(p + 1, std::memory_order_release);
    } else {
      share(p, 0, 1);
    }
  }
  drain();
  if (err) ready.store(STOP, std::memory_order_release);
  for (int i = 0; i < nw; ++i) pool[i].join();
  return err;
}

}  // namespace qftkb_host
